"""Performance cases: the work a program has this library do, through its public Python
face, over the range of sizes in which it is used.

A case is a dict of plain values; "path" names the entry point it goes through:

* qwen2_decode: `DecoderSession.decode_greedy` (and a last `decode` that hands out the
  logits) of the 28-layer Qwen2-1.5B shape behind `context` cached positions.
* qwen2_prefill: `DecoderSession.prefill` of `tokens` tokens behind `context` positions.
* nukopel, lirulix: a `FolderSession`; `prefill` of a prompt, then `new` steps through
  `decode`, whose logits the program looks at itself (sampling, scoring).
* mlp: `ops.mlp_block_w8a32`, the feed-forward block of a decoder for 1 to 16 rows.
* w8a8: `buddy_hip_w8a8_matmul`, int8 weights and activations quantised on the way.

All weights are random with the spread of trained ones and are made from the seed.
"""
from __future__ import annotations

import math
import tempfile

import numpy as np
import torch

from buddy_mlir_amd import check, lib, ops, synthetic
from buddy_mlir_amd.session import DecoderSession, FolderSession, Shape

F64 = torch.float64

# (hidden, intermediate) of the feed-forward blocks: the Qwen2-1.5B, the Llama-3-8B shape
MLP_SHAPES = ((1536, 8960), (4096, 14336))
# (K, N) of the matrices of a Qwen2-1.5B layer
LINEAR_SHAPES = ((1536, 1536), (1536, 8960), (8960, 1536))
# the layers of real models, as the benchmark takes them
NUKOPEL = dict(width=1536, layers="alaa", heads=12, window=1024, experts=16, top=4, ff=1792)
LIRULIX = dict(width=1536, layers="fdsf", heads=12, kv_heads=2, window=1024, ff=8960)

# positions a session leaves room for, beyond those a case fills
ROOM = 64


def listed():
    return [
        # an assistant's answer, 32 of its tokens behind a filled context: what a user waits
        # for most of the time
        {"name": "decode at 1024", "path": "qwen2_decode", "context": 1024, "steps": 32,
         "qkv": "int8"},
        # the same about a long document, with the f32 q|k|v of the reference's shipped graph
        {"name": "decode at 12000", "path": "qwen2_decode", "context": 12000, "steps": 12,
         "qkv": "f32"},
        # a short question
        {"name": "prompt of 27", "path": "qwen2_prefill", "tokens": 27, "context": 0, "qkv": "int8",
         "precision": "digits"},
        # the next question in a conversation, activations cast to bfloat16 on request
        {"name": "prompt of 150 behind 1900", "path": "qwen2_prefill", "tokens": 150,
         "context": 1900, "qkv": "int8", "precision": "bf16"},
        # the prompt length the benchmark names
        {"name": "prompt of 512", "path": "qwen2_prefill", "tokens": 512, "context": 0,
         "qkv": "int8", "precision": "digits"},
        # a document, of a length that fills no tile
        {"name": "prompt of 1931", "path": "qwen2_prefill", "tokens": 1931, "context": 0,
         "qkv": "int8", "precision": "digits"},
        # a document through latent and lightning attention and routed experts
        {"name": "nukopel prompt of 2048", "path": "nukopel", "tokens": 2048, "new": 0,
         "dtype": "bfloat16"},
        # a turn of a chat with it
        {"name": "nukopel 45 and 24 new", "path": "nukopel", "tokens": 45, "new": 24,
         "dtype": "bfloat16"},
        # a prompt through attention with a sink, differential attention and the delta rule
        {"name": "lirulix prompt of 777", "path": "lirulix", "tokens": 777, "new": 0,
         "dtype": "bfloat16"},
        # a turn of a chat with it where every activation stays 32-bit
        {"name": "lirulix f32 300 and 16 new", "path": "lirulix", "tokens": 300, "new": 16,
         "dtype": "float32"},
        # one decoder block for a batch of decoding requests
        {"name": "mlp block of 12 rows", "path": "mlp", "rows": 12, "hidden": 1536, "inter": 8960},
        # a matrix of the int8-activation variant on a prompt
        {"name": "w8a8 of 512 rows", "path": "w8a8", "rows": 512, "k": 1536, "n": 8960},
    ]


def _log(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    path = rng.choice(["qwen2_decode", "qwen2_prefill", "qwen2_prefill", "nukopel", "lirulix",
                       "mlp", "w8a8"])
    if path == "qwen2_decode":
        return {"path": path, "context": _log(rng, 1, 16000), "steps": rng.randint(4, 24),
                "qkv": rng.choice(["int8", "int8", "f32"])}
    if path == "qwen2_prefill":
        return {"path": path, "tokens": _log(rng, 2, 2000),
                "context": rng.choice([0, 0, _log(rng, 16, 2000)]), "qkv": "int8",
                "precision": rng.choice(["digits", "digits", "digits", "digits2", "bf16"])}
    if path in ("nukopel", "lirulix"):
        return {"path": path, "tokens": _log(rng, 8, 2000), "new": rng.choice([0, rng.randint(1, 24)]),
                "dtype": rng.choice(["bfloat16", "bfloat16", "float32"])}
    if path == "mlp":
        hidden, inter = rng.choice(MLP_SHAPES)
        return {"path": path, "rows": rng.randint(1, 16), "hidden": hidden, "inter": inter}
    k, n = rng.choice(LINEAR_SHAPES)
    return {"path": path, "rows": _log(rng, 8, 1000), "k": k, "n": n}


# ---- inputs ----------------------------------------------------------------------

def _gen(*key):
    """A generator on the GPU from the seed and what it is for."""
    n = 0
    for k in key:
        n = (n * 1000003 + int(k)) & 0x7FFFFFFF
    return torch.Generator(device="cuda").manual_seed(n)


def _int8(gen, K, N, std=0.02):
    """W[K, N] per output channel in int8 with its scales."""
    w = torch.randn((K, N), generator=gen, device="cuda") * std
    s = (w.abs().amax(0) / 127.0).clamp_min(1e-10)
    return torch.round(w / s).clamp_(-128, 127).to(torch.int8), s


def _tokens(seed, n, vocab):
    return np.random.default_rng(seed).integers(0, vocab, n).astype(np.int32)


def _qwen2_shape(c):
    used = c["context"] + (c["steps"] + 1 if c["path"] == "qwen2_decode" else c["tokens"])
    return Shape(max_len=used + ROOM)


def _qwen2_layer(s, c, seed, i):
    g = _gen(seed, 1, i)
    QN, KVN = s.heads * s.head_dim, s.kv_heads * s.head_dim
    w = {n: 1.0 + 0.1 * torch.randn(s.hidden, generator=g, device="cuda") for n in ("ln1", "ln2")}
    for n, N in (("q", QN), ("k", KVN), ("v", KVN)):
        if c["qkv"] == "f32":
            w["f" + n] = torch.randn((s.hidden, N), generator=g, device="cuda") * 0.02
        else:
            w["w" + n], w["s" + n] = _int8(g, s.hidden, N)
        w["b" + n] = torch.randn(N, generator=g, device="cuda") * 0.1
    for n, K, N in (("o", QN, s.hidden), ("g", s.hidden, s.inter), ("u", s.hidden, s.inter),
                    ("d", s.inter, s.hidden)):
        w["w" + n], w["s" + n] = _int8(g, K, N)
    return w


def _qwen2_globals(s, seed):
    g = _gen(seed, 2)
    i = torch.arange(0, s.head_dim, 2, device="cuda", dtype=F64)
    w, sc = _int8(g, s.hidden, s.vocab)
    return {"embed": torch.randn((s.vocab, s.hidden), generator=g, device="cuda") * 0.02,
            "inv_freq": (1e6 ** (-i / s.head_dim)).float(),
            "ln_f": 1.0 + 0.1 * torch.randn(s.hidden, generator=g, device="cuda"),
            "w_lm": w, "s_lm": sc}


def _qwen2_kv(s, c, seed, index):
    t = torch.zeros((s.kv_heads, s.max_len, s.head_dim), device="cuda")
    t[:, :c["context"]] = torch.randn((s.kv_heads, c["context"], s.head_dim),
                                      generator=_gen(seed, 3, index), device="cuda")
    return t


def _qwen2_session(c, seed):
    s = _qwen2_shape(c)
    sess = DecoderSession(s)
    sess.set_globals(**_qwen2_globals(s, seed))
    for i in range(s.layers):
        sess.set_layer(i, _qwen2_layer(s, c, seed, i))
    if c["context"]:
        for i in range(2 * s.layers):
            sess.set_kv(i, _qwen2_kv(s, c, seed, i))
    n = 1 if c["path"] == "qwen2_decode" else c["tokens"]
    return {"session": sess, "tokens": _tokens(seed, n, s.vocab)}


def _folder_config(c):
    if c["path"] == "nukopel":
        return synthetic.nukopel_config(**NUKOPEL)
    return synthetic.lirulix_config(**LIRULIX)


def _folder_shapes(c, cfg):
    make = synthetic.nukopel_shapes if c["path"] == "nukopel" else synthetic.lirulix_shapes
    return list(make(cfg))


def _folder_session(c, seed):
    cfg = _folder_config(c)
    with tempfile.TemporaryDirectory() as folder:
        synthetic.write_folder(folder, cfg, _folder_shapes(c, cfg), seed)
        sess = FolderSession(folder, c["dtype"], max_len=c["tokens"] + c["new"] + ROOM)
    return {"session": sess, "tokens": _tokens(seed, c["tokens"] + c["new"], cfg["vocab"])}


def _mlp_inputs(c, seed):
    g = _gen(seed, 4)
    H, I = c["hidden"], c["inter"]
    d = {n: _int8(g, K, N) for n, K, N in (("gate", H, I), ("up", H, I), ("down", I, H))}
    d["norm"] = 1.0 + 0.1 * torch.randn(H, generator=g, device="cuda")
    d["x"] = torch.randn((c["rows"], H), generator=g, device="cuda")
    return d


def _w8a8_inputs(c, seed):
    g = _gen(seed, 5)
    q, s = _int8(g, c["k"], c["n"])
    return q, s, torch.randn((c["rows"], c["k"]), generator=g, device="cuda")


def prepare(case, seed):
    c = case
    if c["path"].startswith("qwen2"):
        state = _qwen2_session(c, seed)
    elif c["path"] in ("nukopel", "lirulix"):
        state = _folder_session(c, seed)
    elif c["path"] == "mlp":
        d = _mlp_inputs(c, seed)
        state = {n: (ops.pack_w8(d[n][0]), d[n][1]) for n in ("gate", "up", "down")}
        state.update(x=d["x"], norm=d["norm"], workspace=torch.empty(
            lib().buddy_hip_mlp_block_workspace_bytes(c["rows"], c["inter"]), dtype=torch.uint8,
            device="cuda"))
    else:
        q, s, x = _w8a8_inputs(c, seed)
        state = {"packed": ops.pack_w8(q), "scale": s, "x": x, "workspace": torch.empty(
            lib().buddy_hip_w8a8_workspace_bytes(c["rows"], c["k"]), dtype=torch.uint8,
            device="cuda")}
    state["case"] = dict(c)
    return state


# ---- one pass --------------------------------------------------------------------

def run(state):
    c = state["case"]
    if c["path"] == "qwen2_decode":
        sess = state["session"]
        toks = sess.decode_greedy(int(state["tokens"][0]), c["context"], c["steps"])
        nxt, logits = sess.decode(int(toks[-1]), c["context"] + c["steps"])
        return {"tokens": toks, "next": nxt, "logits": logits}
    if c["path"] == "qwen2_prefill":
        nxt, logits = state["session"].prefill(state["tokens"], c["context"],
                                               precision=c["precision"])
        return {"next": nxt, "logits": logits}
    if c["path"] in ("nukopel", "lirulix"):
        sess, toks, n = state["session"], state["tokens"], c["tokens"]
        rows = [sess.prefill(toks[:n], 0)[1]]
        for i in range(n, n + c["new"]):
            rows.append(sess.decode(int(toks[i]), i)[1])
        return rows
    if c["path"] == "mlp":
        return ops.mlp_block_w8a32(state["x"], *state["gate"], *state["up"], *state["down"],
                                   c["hidden"], c["inter"], norm_w=state["norm"], norm_eps=1e-6,
                                   workspace=state["workspace"])
    x, ws = state["x"], state["workspace"]
    out = torch.empty((c["rows"], c["n"]), device="cuda")
    check(lib().buddy_hip_w8a8_matmul(
        x.data_ptr(), state["packed"].data_ptr(), state["scale"].data_ptr(), out.data_ptr(), None,
        c["rows"], c["k"], c["n"], ws.data_ptr(), ws.numel(),
        torch.cuda.current_stream().cuda_stream), "w8a8_matmul")
    return out


# ---- what a pass cannot do without -------------------------------------------------

def _qwen2_work(c):
    s = Shape()
    H, QN, KVN = s.hidden, s.heads * s.head_dim, s.kv_heads * s.head_dim
    mats = ((H, QN + 2 * KVN), (QN, H), (H, 2 * s.inter), (s.inter, H))
    qkv = 4 if c["qkv"] == "f32" else 1
    layer_bytes = sum(K * N * (qkv if i == 0 else 1) + 4 * N for i, (K, N) in enumerate(mats)) + 8 * H
    layer_flops = 2 * sum(K * N for K, N in mats)
    head = s.vocab * (H + 4 + 4)
    row = 2 * 4 * KVN  # a position's key and value in one layer
    n, ctx = c.get("tokens", 1), c["context"]
    passes = c["steps"] + 1 if c["path"] == "qwen2_decode" else 1
    b = f = 0
    for t in range(passes):
        seen = ctx + t
        b += s.layers * (layer_bytes + row * (seen + n)) + head + 4 * H * n
        f += s.layers * (layer_flops * n + 4 * QN * (n * seen + n * (n + 1) // 2)) + 2 * H * s.vocab
    return b, f


def _seen(n, new, window=None):
    """Keys that the rows of a prompt and of the steps behind it look at, all together."""
    return sum(min(p + 1, window or p + 1) for p in range(n + new))


def _folder_work(c):
    cfg = _folder_config(c)
    n, new, size = c["tokens"], c["new"], 2 if c["dtype"] == "bfloat16" else 4
    shapes = {name: shape for name, shape, _ in _folder_shapes(c, cfg)}
    W, V = cfg["width"], cfg["vocab"]
    fixed = 2 * V * W                      # bytes of the weights that every row needs
    dense = 0                              # multiply-adds of a row
    experts = 0                            # bytes of one expert, over the layers
    state_bytes = attention = 0
    for i, layer in enumerate(cfg["layers"]):
        p, m = f"l{i}.", layer["mixer"]
        for name, shape in shapes.items():
            if name.startswith(p) and len(shape) == 2 and ".e" not in name:
                fixed += 2 * shape[0] * shape[1]
                dense += shape[0] * shape[1]
        H, D, VD = m["heads"], m["dim"], m["vdim"]
        if c["path"] == "nukopel":
            f = layer["mlp"]
            one = 3 * W * f["expert"]["ff"]
            experts += 2 * one
            dense += f["router"]["top"] * one
        if layer["type"] in ("lightning", "channel_delta"):
            state_bytes += 2 * 4 * H * D * VD * (1 + new)
            dense += 2 * H * D * VD
        else:
            maps = 2 if layer["type"] == "attention_2" else 1
            window = m["mask"]["size"] if "mask" in m else None
            row = m["kv_rank"] + m["rot_dim"] if "kv_rank" in m else m["kv_heads"] * (maps * D + VD)
            q = D + m.get("rot_dim", 0)
            attention += 2 * H * maps * (q + VD) * _seen(n, new, window)
            state_bytes += size * row * (n + sum(min(n + t + 1, window or n + t + 1)
                                                 for t in range(new)))
    routed = 0
    if experts:
        r = cfg["layers"][0]["mlp"]["router"]
        routed = experts * (min(r["experts"], n * r["top"]) + new * r["top"])
    b = fixed * (1 + new) + routed + state_bytes + 4 * V * (1 + new) + 2 * W * (n + new)
    return b, 2 * dense * (n + new) + attention + 2 * V * W * (1 + new)


def work(case):
    c = case
    if c["path"].startswith("qwen2"):
        b, f = _qwen2_work(c)
    elif c["path"] in ("nukopel", "lirulix"):
        b, f = _folder_work(c)
    elif c["path"] == "mlp":
        H, I = c["hidden"], c["inter"]
        b, f = 3 * H * I + 4 * (2 * I + 2 * H) + 8 * c["rows"] * H, 6 * c["rows"] * H * I
    else:
        M, K, N = c["rows"], c["k"], c["n"]
        b, f = K * N + 4 * N + 4 * M * (K + N), 2 * M * K * N
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times what was measured against 64 bits."""
    c = case
    if c["path"] == "qwen2_prefill":
        # 32-bit sums, 2^-23 of a row's largest value; 2^-15 of it; 2^-8 of every value
        return {"rel": {"digits": 2e-5, "digits2": 4.5e-3, "bf16": 3e-2}[c["precision"]]}
    if c["path"] in ("nukopel", "lirulix"):
        return {"rel": 2e-2 if c["dtype"] == "bfloat16" else 1e-5}
    if c["path"] == "w8a8":
        return {"rel": 2e-7}  # whole numbers up to the last product
    return {"rel": 8e-6 if c["path"] == "qwen2_decode" else 3e-6}


# ---- the same in 64 bits -----------------------------------------------------------

def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _softmax(s, sink=None):
    m = s.amax(-1, keepdim=True)
    e = torch.exp(s - m)
    total = e.sum(-1, keepdim=True)
    return e / (total if sink is None else total + torch.exp(sink - m))


def _turn(x, angle, factor=1.0):
    """x [heads, tokens, dims]: coordinate i turns with i + dims / 2."""
    half = x.shape[-1] // 2
    c, s = torch.cos(angle) * factor, torch.sin(angle) * factor
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _plain(q, s):
    return q.to(F64) * s.to(F64)


class _Qwen2:
    """The decoder of the qwen2 cases on whole blocks of tokens."""

    def __init__(self, c, seed):
        self.s, self.g, self.layers, self.kv = _qwen2_shape(c), None, [], []
        self.g = _qwen2_globals(self.s, seed)
        self.g["lm"] = _plain(self.g.pop("w_lm"), self.g["s_lm"])
        for i in range(self.s.layers):
            w = _qwen2_layer(self.s, c, seed, i)
            for n in "qkvogud":
                w[n] = w["f" + n].to(F64) if "f" + n in w else _plain(w["w" + n], w["s" + n])
                w.pop("w" + n, None)
            self.layers.append(w)
            self.kv.append([_qwen2_kv(self.s, c, seed, 2 * i + j).to(F64) for j in (0, 1)])

    def block(self, tokens, pos):
        """Logits behind the last of the tokens, the first of which stands at `pos`."""
        s, n = self.s, len(tokens)
        x = self.g["embed"][torch.as_tensor(np.asarray(tokens), device="cuda").long()].to(F64)
        at = torch.arange(pos, pos + n, device="cuda")
        # an angle is the product of a position and a frequency in f32, as the model defines it
        angle = (at.float()[:, None] * self.g["inv_freq"][None, :]).to(F64)
        seen = torch.arange(pos + n, device="cuda")[None, :] <= at[:, None]
        for w, (kc, vc) in zip(self.layers, self.kv):
            h = _rms(x, s.rms_eps) * w["ln1"].to(F64)
            q, k, v = (((h @ w[t]) + w["b" + t].to(F64)).reshape(n, -1, s.head_dim).transpose(0, 1)
                       for t in "qkv")
            kc[:, pos:pos + n], vc[:, pos:pos + n] = _turn(k, angle), v
            q = _turn(q, angle).reshape(s.kv_heads, -1, s.head_dim)
            outs = []
            for g in range(s.kv_heads):
                sc = (q[g] @ kc[g, :pos + n].T) * s.head_dim ** -0.5
                sc = sc.reshape(-1, n, pos + n).masked_fill(~seen[None], -math.inf)
                outs.append((_softmax(sc).reshape(-1, pos + n) @ vc[g, :pos + n])
                            .reshape(-1, n, s.head_dim))
            o = torch.cat(outs).transpose(0, 1).reshape(n, -1)
            x = x + o @ w["o"]
            h = _rms(x, s.rms_eps) * w["ln2"].to(F64)
            x = x + (torch.nn.functional.silu(h @ w["g"]) * (h @ w["u"])) @ w["d"]
        return (_rms(x[-1], s.rms_eps) * self.g["ln_f"].to(F64)) @ self.g["lm"]


def _qwen2_exact(c, seed):
    m = _Qwen2(c, seed)
    if c["path"] == "qwen2_prefill":
        logits = m.block(_tokens(seed, c["tokens"], m.s.vocab), c["context"])
        return {"next": int(logits.argmax()), "logits": logits}
    tok, toks = int(_tokens(seed, 1, m.s.vocab)[0]), []
    for t in range(c["steps"] + 1):
        logits = m.block([tok], c["context"] + t)
        tok = int(logits.argmax())
        toks.append(tok)
    return {"tokens": np.asarray(toks[:-1], np.int32), "next": tok, "logits": logits}


def _folder_tensors(c, cfg, seed):
    """The tensors of the folder, as write_folder draws them, in 64 bits."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return {name: torch.ones(shape, dtype=F64, device="cuda") if std is None else
            (torch.randn(shape, generator=g, device="cuda") * std).bfloat16().to(F64)
            for name, shape, std in _folder_shapes(c, cfg)}


def _conv(x, taps):
    """Causal depth-wise convolution; taps [channels, taps], the last of them is now."""
    out, n, T = torch.zeros_like(x), x.shape[0], taps.shape[1]
    for back in range(min(T, n)):
        out[back:] += taps[:, T - 1 - back] * x[:n - back]
    return out


def _heads(x, H):
    return x.reshape(x.shape[0], H, -1).transpose(0, 1)


def _visible(n, window=None):
    gap = torch.arange(n, device="cuda")[:, None] - torch.arange(n, device="cuda")[None, :]
    return (gap >= 0) & (gap < (window or n))


def _angle(n, freq):
    return torch.arange(n, device="cuda", dtype=F64)[:, None] * freq[None, :]


def _plain_freq(dims, base):
    return base ** (-torch.arange(0, dims, 2, device="cuda", dtype=F64) / dims)


def _nukopel_expert(h, w, p, limit):
    g = (h @ w[p + "gate"].T).clamp_max(limit)
    u = (h @ w[p + "up"].T).clamp(-limit, limit)
    return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w[p + "down"].T


def _nukopel_mixer(h, w, layer, eps):
    n, m = h.shape[0], layer["mixer"]
    H, D, VD = m["heads"], m["dim"], m["vdim"]
    if layer["type"] == "lightning":
        q, k, v = (_heads(torch.nn.functional.silu(h @ w[t].T), H) for t in "qkv")
        gap = _angle(n, torch.ones(1, device="cuda", dtype=F64))
        gap = (gap - gap.T).clamp_min(0.0)
        o = torch.empty((H, n, VD), device="cuda", dtype=F64)
        for i, d in enumerate(m["decay"]):
            o[i] = (torch.where(_visible(n), d ** gap, 0.0) * (q[i] @ k[i].T)) @ v[i]
        o = _rms(o.transpose(0, 1).reshape(n, -1), eps) * w["norm"]
        return (o * torch.sigmoid(h @ w["g"].T)) @ w["o"].T
    R, L = m["rot_dim"], m["kv_rank"]
    angle = _angle(n, _plain_freq(R, m["rot"]["base"]))
    q, down = _heads(h @ w["q"].T, H), h @ w["dkv"].T
    lat = _rms(down[:, :L], eps) * w["dkv.norm"]
    k, v = _heads(lat @ w["uk"].T, H), _heads(lat @ w["uv"].T, H)
    k_rot, q_rot = _turn(down[None, :, L:], angle)[0], _turn(q[..., D:], angle)
    seen = _visible(n, m["mask"]["size"])
    o = torch.empty((n, H, VD), device="cuda", dtype=F64)
    for i in range(H):
        sc = (q[i, :, :D] @ k[i].T + q_rot[i] @ k_rot.T) * m["scale"]
        o[:, i] = _softmax(sc.masked_fill(~seen, -math.inf)) @ v[i]
    o = o * torch.sigmoid(h @ w["g"].T)[:, :, None]
    return o.reshape(n, -1) @ w["o"].T


def _nukopel_exact(cfg, t, tokens):
    eps = cfg["norm"]["eps"]
    x = t["embed"][tokens] * cfg["embedding"]["scale"]
    for i, layer in enumerate(cfg["layers"]):
        w = {k[len(f"l{i}."):]: v for k, v in t.items() if k.startswith(f"l{i}.")}
        h = _rms(x, eps) * w["norm1"]
        h = h + _conv(h, w["canon1"])
        mix = {k[4:]: v for k, v in w.items() if k.startswith("mix.")}
        x = x + _rms(_nukopel_mixer(h, mix, layer, eps), eps) * w["norm1b"]
        h, f = _rms(x, eps) * w["norm2"], layer["mlp"]
        z, chosen = torch.topk(h @ w["mlp.router"].T, f["router"]["top"], dim=-1)
        weight = _softmax(z)
        y = _nukopel_expert(h, w, "mlp.shared.", f["shared"]["limit"])
        for e in range(f["router"]["experts"]):
            row, slot = torch.nonzero(chosen == e, as_tuple=True)
            if row.numel():
                y[row] += weight[row, slot][:, None] * _nukopel_expert(
                    h[row], w, f"mlp.e{e}.", f["expert"]["limit"])
        x = x + _rms(y, eps) * w["norm2b"]
    return _rms(x, eps) * t["final.norm"]


def _yarn(dims, base, s):
    def turn_dim(t):
        return dims * math.log(s["original"] / (2 * math.pi * t)) / (2 * math.log(base))
    lo = max(math.floor(turn_dim(s["fast"])), 0)
    hi = min(math.ceil(turn_dim(s["slow"])), dims - 1)
    i = torch.arange(dims // 2, device="cuda", dtype=F64)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    f = _plain_freq(dims, base)
    return f / s["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(s["factor"]) + 1.0


def _banded(dims, base, s):
    f = _plain_freq(dims, base)
    t = ((s["original"] * f / (2 * math.pi) - s["low"]) / (s["high"] - s["low"])).clamp(0.0, 1.0)
    return (1 - t) * f / s["factor"] + t * f


def _delta(h, w, m, eps):
    n, H, G, D, VD = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (torch.nn.functional.silu(_conv(h @ w[t].T, w[t + ".conv"])) for t in "qkv")
    q, k = (y.reshape(n, G, D).repeat_interleave(H // G, 1) for y in (q, k))
    q, k = (y * torch.rsqrt((y * y).sum(-1, keepdim=True) + 1e-6) for y in (q, k))
    v, beta = v.reshape(n, H, VD), torch.sigmoid(h @ w["b"].T)
    dt = torch.nn.functional.softplus((h @ w["a1"].T) @ w["a2"].T + w["dt_bias"]).reshape(n, H, D)
    decay = torch.exp(-torch.exp(w["A_log"])[:, None] * dt)
    S, o = torch.zeros((H, D, VD), device="cuda", dtype=F64), torch.empty_like(v)
    q = q * D ** -0.5
    for t in range(n):
        S = S * decay[t][:, :, None]
        u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
        S = S + k[t][:, :, None] * u[:, None, :]
        o[t] = (S * q[t][:, :, None]).sum(1)
    o = (_rms(o, eps) * w["norm"]).reshape(n, -1)
    return (o * torch.sigmoid((h @ w["g1"].T) @ w["g2"].T)) @ w["o"].T


def _lirulix_mixer(h, w, layer, eps):
    n, m = h.shape[0], layer["mixer"]
    if layer["type"] == "channel_delta":
        return _delta(h, w, m, eps)
    H, G, VD = m["heads"], m["kv_heads"], m["vdim"]
    maps = 2 if layer["type"] == "attention_2" else 1
    rot, factor = m["rot"], 1.0
    if maps == 1:
        freq, factor = _yarn(rot["dims"], rot["base"], rot["scaling"])
    else:
        freq = _banded(rot["dims"], rot["base"], rot["scaling"])
        lam = (torch.exp(w["lq1"] @ w["lk1"]) - torch.exp(w["lq2"] @ w["lk2"])) + m["diff"]
    angle = _angle(n, freq)
    q, k = (_turn(_heads(h @ w[t].T, x * maps), angle, factor) for t, x in (("q", H), ("k", G)))
    v, seen = _heads(h @ w["v"].T, G), _visible(n, m["mask"]["size"] if maps == 2 else None)
    o = torch.empty((n, H, VD), device="cuda", dtype=F64)
    for i in range(H):
        g = i // (H // G)
        a = [_softmax(((q[i * maps + j] @ k[g * maps + j].T) * m["scale"])
                      .masked_fill(~seen, -math.inf), w["sink"][i] if maps == 1 else None) @ v[g]
             for j in range(maps)]
        o[:, i] = a[0] if maps == 1 else _rms(a[0] - lam * a[1], eps) * (1.0 - m["diff"])
    o = o.reshape(n, -1)
    return (o if maps == 1 else o * torch.sigmoid(h @ w["g"].T)) @ w["o"].T


def _lirulix_exact(cfg, t, tokens):
    eps, loop = cfg["norm"]["eps"], cfg["loop"]

    def norm(x, w):
        return _rms(x, eps) * (1.0 + w)

    x = norm(t["embed"][tokens], t["embed.norm"])
    start, stop = loop["start"], loop["stop"]
    order = [(i, None) for i in range(start)]
    for p in range(loop["times"]):
        order += [(i, p if i == start else None) for i in range(start, stop)]
    for i, p in order + [(i, None) for i in range(stop, len(cfg["layers"]))]:
        if p is not None:
            x = x + t["loop.step"][p]
        w = {k[len(f"l{i}."):]: v for k, v in t.items() if k.startswith(f"l{i}.")}
        mix = {k[4:]: v for k, v in w.items() if k.startswith("mix.")}
        x = x + _lirulix_mixer(norm(x, w["norm1"]), mix, cfg["layers"][i], eps)
        h = norm(x, w["norm2"])
        gate = torch.nn.functional.gelu(h @ w["mlp.gate"].T, approximate="tanh")
        x = x + (gate * (h @ w["mlp.up"].T)) @ w["mlp.down"].T
    return norm(x, t["final.norm"])


def _folder_exact(c, seed):
    cfg = _folder_config(c)
    t = _folder_tensors(c, cfg, seed)
    toks = torch.as_tensor(_tokens(seed, c["tokens"] + c["new"], cfg["vocab"])).long().cuda()
    x = (_nukopel_exact if c["path"] == "nukopel" else _lirulix_exact)(cfg, t, toks)
    return list(x[c["tokens"] - 1:] @ t["head"].T)


def exact(case, seed):
    c = case
    if c["path"].startswith("qwen2"):
        return _qwen2_exact(c, seed)
    if c["path"] in ("nukopel", "lirulix"):
        return _folder_exact(c, seed)
    if c["path"] == "mlp":
        d = _mlp_inputs(c, seed)
        h = _rms(d["x"].to(F64), 1e-6) * d["norm"].to(F64)
        gate, up, down = (_plain(*d[n]) for n in ("gate", "up", "down"))
        return (torch.nn.functional.silu(h @ gate) * (h @ up)) @ down
    q, s, x = _w8a8_inputs(c, seed)
    # the activations' scale and rounding are part of the operation, in f32
    step = (x.abs().amax() * (1.0 / 127.0)).clamp_min(1e-10)
    a = torch.round(x * (1.0 / step)).clamp_(-128, 127)
    return ((a.to(F64) @ q.to(F64)) * (step * s).to(F64))
