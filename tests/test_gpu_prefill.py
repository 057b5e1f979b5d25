"""GPU parity of the prefill path: the MFMA int8 dequant matmul against the
oracle's BLIS restatement, the causal GQA attention against the oracle's
flash-attention restatement, and block prefill of the resident session against
token-by-token decode steps of the oracle."""
import numpy as np
import pytest
import torch

import buddy_mlir_amd as bma
from buddy_mlir_amd import ops, synthetic
from buddy_mlir_amd.session import Shape
from buddy_mlir_amd.session import DecoderSession
from parity import check_close
from test_gpu_decode import SMALL, oracle_model
from tile_report import tiles_run

pytestmark = pytest.mark.gpu

SCALE = np.float32(0.0883883461)


def bf16_round(a: np.ndarray) -> np.ndarray:
    return torch.from_numpy(a).to(torch.bfloat16).to(torch.float32).numpy()


GEMM_SHAPES = [(512, 1536, 1536), (512, 1536, 256), (512, 1536, 8960), (512, 8960, 1536),
               (9, 4, 17), (65, 129, 257), (1, 64, 16), (130, 200, 130),
               # ragged in every dimension and wide enough for the kernel that does
               # not split K (64 x 256 workgroup tiles)
               (500, 200, 6500), (1000, 72, 3300)]


def fixed_point_round(a: np.ndarray, digits: int = 3):
    """What the int8 matmul multiplies: per row the smallest power-of-two step s
    with max|a| / s < 2^(8 digits - 2), and rint(a / s) * s."""
    mx = np.abs(a).max(axis=1, keepdims=True).astype(np.float64)
    e = np.floor(np.log2(np.where(mx > 0, mx, 1.0))) + 1 - (8 * digits - 2)
    step = np.exp2(np.maximum(e, -126))
    return (np.rint(a.astype(np.float64) / step) * step).astype(np.float32), step


@pytest.mark.parametrize("M,K,N", GEMM_SHAPES)
@pytest.mark.parametrize("mode", ["bf16", "exact", "digits", "digits2"])
def test_prefill_gemm_matches_blis_oracle(oracle, M, K, N, mode):
    q, s = synthetic.quantized_linear(K, N, M + K + N)
    packed = ops.pack_w8(q)
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn((M, K), generator=g, device="cuda")
    if mode.startswith("digits") and M > 2:
        x[1] *= 1e-30   # rows of very different magnitude: the step is per row
        x[2, 0] = 300.0  # one large element in a row of small ones
    y = ops.gemm_w8a32(x, packed, s, K, N, exact=mode == "exact",
                       digits={"digits": 3, "digits2": 2}.get(mode, False))
    torch.cuda.synchronize()
    xh = x.cpu().numpy()
    if mode == "digits2":
        # two digit planes: 15 bits below each row's maximum, the fixed-point
        # counterpart of the bf16 cast.  Like that mode it is held to the oracle
        # fed the same rounded activations (only summation order is left) ...
        got = y.cpu().numpy()
        a_in, _ = fixed_point_round(xh, digits=2)
        want = oracle.blis_gemm_w8a32(a_in, q.cpu().numpy(), s.cpu().numpy())
        for m in range(M):
            check_close(got[m], want[m], normwise=4e-6)
        # ... and stays within the rounding it states of the plain f32 input:
        # norm-wise 2^-15 max|row| sqrt(K) / |row| at most, far inside the bf16
        # cast's 2^-9
        want = oracle.blis_gemm_w8a32(xh, q.cpu().numpy(), s.cpu().numpy())
        for m in range(M):
            if m != 2 or M <= 2:  # (the row with the 300 sigma outlier: its step is 2^-6)
                assert np.linalg.norm(got[m] - want[m]) <= 2e-4 * np.linalg.norm(want[m]) + 1e-30
        return
    if mode == "digits":
        # against the plain f32 input at the stated bar, per row (rows differ by
        # 30 orders of magnitude) ...
        want = oracle.blis_gemm_w8a32(xh, q.cpu().numpy(), s.cpu().numpy())
        got = y.cpu().numpy()
        for m in range(M):
            check_close(got[m], want[m])
        # ... and against the oracle fed the same fixed-point activations, where
        # what is left is summation order only
        a_in, _ = fixed_point_round(xh)
        want = oracle.blis_gemm_w8a32(a_in, q.cpu().numpy(), s.cpu().numpy())
        for m in range(M):
            check_close(got[m], want[m], normwise=4e-6)
        return
    # "activations cast to bf16": the oracle gets the same rounded activations
    a_in = xh if mode == "exact" else bf16_round(xh)
    want = oracle.blis_gemm_w8a32(a_in, q.cpu().numpy(), s.cpu().numpy())
    check_close(y.cpu().numpy(), want)


@pytest.mark.parametrize("M,K,N", [(512, 1536, 8960), (512, 8960, 1536), (70, 200, 48)])
def test_non_finite_activation_rows_come_out_nan_in_the_digit_mode(M, K, N):
    """The reference's prefill kernel is an f32 multiply-add chain
    (MatMulBlisVectorization.cpp:644-740): a NaN in a row of A makes that row of
    C NaN, an infinity makes it +-inf or NaN.  The digit-plane matmul gives such a
    row a NaN step: every element of the row is NaN, every other row is what it
    is without the poison, bit for bit."""
    q, s = synthetic.quantized_linear(K, N, 5)
    packed = ops.pack_w8(q)
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x = torch.randn((M, K), generator=g, device="cuda")
    clean = ops.gemm_w8a32(x, packed, s, K, N, digits=True).cpu().numpy()
    x[3, K // 2] = float("nan")
    x[M - 2, 0] = float("-inf")
    x[5, K - 1] = float("inf")
    got = ops.gemm_w8a32(x, packed, s, K, N, digits=True).cpu().numpy()
    bad = [3, 5, M - 2]
    assert np.isnan(got[bad]).all()
    rest = np.delete(np.arange(M), bad)
    assert np.isfinite(got[rest]).all()
    np.testing.assert_array_equal(got[rest], clean[rest])
    # the paired gate|up form with SiLU*mul in its epilogue
    if N % 64 == 0:
        both = torch.cat([packed, packed])
        got = ops.gemm_w8a32(x, both, torch.cat([s, s]), K, N, digits=True,
                             silu_pair=True).cpu().numpy()
        assert np.isnan(got[bad]).all() and np.isfinite(got[rest]).all()


def test_non_finite_token_through_session_prefill():
    """A prompt whose last token's embedding row holds a NaN (then an infinity):
    that row's logits are NaN; the logits of every earlier row are those of the
    clean prompt bit for bit (causality), through every digit-plane producer of
    the block (RMSNorm rows, SiLU*mul rows, the slice-adding kernel that writes
    the next layer's rows).  The poisoned token is the first of a 16-row block of
    the attention kernel: a masked key still meets the queries of its own block
    in the P.V matrix product as 0 x NaN (in the reference the additive -inf
    mask lets a NaN key reach every query of the prompt)."""
    sess, _ = synthetic.build_session(SMALL, context=0, ln_jitter=0.1)
    lib = bma.lib()
    V = SMALL.vocab
    toks = synthetic.first_tokens(SMALL, 33, seed=5).astype(np.int32)
    poisoned = int(toks[-1])
    toks[:-1][toks[:-1] == poisoned] = (poisoned + 1) % V

    def all_logits():
        out = np.empty((toks.size, V), np.float32)
        bma.check(lib.buddy_hip_session_prefill_all_logits(
            sess._h, toks.ctypes.data, toks.size, 0, out.ctypes.data), "prefill_all_logits")
        return out

    clean = all_logits()
    assert np.isfinite(clean).all()
    embed = sess._globals["embed"]
    for poison in (float("nan"), float("-inf")):
        keep = embed[poisoned].clone()
        embed[poisoned, 7] = poison
        torch.cuda.synchronize()
        got = all_logits()
        embed[poisoned] = keep
        torch.cuda.synchronize()
        assert np.isnan(got[-1]).all()
        np.testing.assert_array_equal(got[:-1], clean[:-1])
    np.testing.assert_array_equal(all_logits(), clean)
    sess.close()


@pytest.mark.parametrize("M,K", [(1, 64), (5, 100), (70, 1536), (48, 8960)])
def test_digit_planes_are_the_rounded_fixed_point(M, K):
    """W = 127 I with scale 1/127 copies the activations: what comes out is
    rint(a / s) * s exactly, row by row."""
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn((M, K), generator=g, device="cuda") * 3.0
    x[0, 0] = 0.0
    if M > 1:
        x[1] = 0.0  # an all-zero row
        x[M - 1] *= 2.0 ** -100
    q = (torch.eye(K, device="cuda") * 127).to(torch.int8)
    s = torch.full((K,), 1.0 / 127.0, device="cuda")
    y = ops.gemm_w8a32(x, ops.pack_w8(q), s, K, K, digits=True)
    torch.cuda.synchronize()
    want, step = fixed_point_round(x.cpu().numpy())
    got = y.cpu().numpy().astype(np.float64)
    # 127 * (1/127 rounded to f32) is 1 to within 1 ulp of f32
    np.testing.assert_allclose(got, want, rtol=2e-7, atol=0)
    xh = x.cpu().numpy().astype(np.float64)
    assert (np.abs(got - xh) <= 0.5 * step + 2e-7 * np.abs(xh)).all()


# rows that stay in registers, in each number of runs of four a thread, ending within one and at its end,
# against rows one float into a buffer, which go through LDS: the same digits, so the same bits of the product
@pytest.mark.parametrize("M,K", [(1, 4), (17, 1020), (33, 2048), (31, 2052), (40, 4100), (65, 6148), (18, 10240),
                                 (16, 10244), (34, 14336)])
@pytest.mark.parametrize("digits", [2, 3])
def test_rows_become_digits_in_registers_as_in_lds(M, K, digits):
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x = torch.randn((M, K), generator=g, device="cuda")
    x[M // 2] *= 2.0 ** 90
    x[M - 1, K - 1] = float("inf") if M > 1 else 2.0 ** -130
    shifted = torch.empty(M * K + 1, device="cuda")[1:].reshape(M, K)
    shifted.copy_(x)
    q, s = synthetic.quantized_linear(K, 48, M)
    packed = ops.pack_w8(q)
    a, b = (ops.gemm_w8a32(t, packed, s, K, 48, digits=digits) for t in (x, shifted))
    torch.cuda.synchronize()
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))


# gate and up in one launch with SiLU(gate) * up in its epilogue: the model's
# shape, one shape for each of the four workgroup tiles, single-tile and ragged rows
SILU_PAIR_SHAPES = [(512, 1536, 8960), (144, 256, 8192), (300, 256, 5120), (200, 192, 8192),
                    (512, 192, 4480), (17, 64, 16), (100, 100, 160)]


def silu_pair_case(oracle, M, K, N, digits=3):
    q0, s0 = synthetic.quantized_linear(K, N, M + K + N)
    q1, s1 = synthetic.quantized_linear(K, N, M + K + N + 1)
    packed = torch.cat([ops.pack_w8(q0), ops.pack_w8(q1)])
    scale = torch.cat([s0, s1])
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn((M, K), generator=g, device="cuda")
    y = ops.gemm_w8a32(x, packed, scale, K, N, digits=digits, silu_pair=True)
    torch.cuda.synchronize()
    xh = x.cpu().numpy()
    if digits == 2:  # the oracle gets the same 15-bit fixed-point activations
        xh, _ = fixed_point_round(xh, digits=2)
    gate = oracle.blis_gemm_w8a32(xh, q0.cpu().numpy(), s0.cpu().numpy())
    up = oracle.blis_gemm_w8a32(xh, q1.cpu().numpy(), s1.cpu().numpy())
    got = y.cpu().numpy()
    assert got.shape == (M, N)
    for m in range(M):
        check_close(got[m], oracle.silu_mul(gate[m], up[m]))


@pytest.mark.parametrize("M,K,N", SILU_PAIR_SHAPES)
def test_prefill_gemm_silu_pair(oracle, M, K, N):
    silu_pair_case(oracle, M, K, N)


@pytest.mark.parametrize("digits", [3, 2])
def test_prefill_gemm_silu_pair_of_4_gib_matrices(digits):
    """The second matrix lies 2^32 bytes behind the first: gate's weights are all 1, up's all 2."""
    M, K, N = 64, 65536, 65536
    packed = torch.empty(2 * K * N, dtype=torch.int8, device="cuda")
    packed[:K * N].fill_(1)
    packed[K * N:].fill_(2)
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn((M, K), generator=g, device="cuda")
    scale = (0.5 + torch.rand(2 * N, generator=g, device="cuda")) / 256
    got = ops.gemm_w8a32(x, packed, scale, K, N, digits=digits, silu_pair=True).double()
    del packed
    rounded, step = fixed_point_round(x.cpu().numpy(), digits=digits)
    # both sums: 24 roundings of at most the sum of the digits' magnitudes, as at tile edges
    size = torch.from_numpy((np.abs(rounded).astype(np.float64) + step * 2.0**16).sum(1)).cuda()[:, None]
    total = torch.from_numpy(rounded.astype(np.float64).sum(1)).cuda()[:, None]
    s = scale.double()
    gate, up, err = total * s[:N], 2 * total * s[N:], 24 * 2.0**-24 * size
    silu = gate * torch.sigmoid(gate)
    # SiLU's slope stays below 1.1; ten roundings in it and the product
    bound = 1.1 * err * s[:N] * up.abs() + silu.abs() * 2 * err * s[N:] + 10 * 2.0**-24 * (gate * up).abs()
    assert ((got - silu * up).abs() <= bound).all()


def test_prefill_gemm_silu_pair_refusals(bh):
    x = torch.zeros((32, 64), device="cuda")
    w = torch.zeros((2 * 64 * 64,), dtype=torch.int8, device="cuda")
    s = torch.ones((128,), device="cuda")
    c = torch.zeros((32, 64), device="cuda")
    # not without the digit planes, not with accumulation, not with a ragged N
    assert bh.buddy_hip_gemm_w8a32(x.data_ptr(), w.data_ptr(), s.data_ptr(), c.data_ptr(),
                                   32, 64, 64, ops.GEMM_SILU_PAIR, None) != 0
    assert bh.buddy_hip_gemm_w8a32(x.data_ptr(), w.data_ptr(), s.data_ptr(), c.data_ptr(),
                                   32, 64, 64, ops.GEMM_SILU_PAIR | ops.GEMM_A_I8_DIGITS |
                                   ops.GEMV_ACCUMULATE, None) != 0
    assert bh.buddy_hip_gemm_w8a32(x.data_ptr(), w.data_ptr(), s.data_ptr(), c.data_ptr(),
                                   32, 64, 40, ops.GEMM_SILU_PAIR | ops.GEMM_A_I8_DIGITS,
                                   None) != 0
    torch.cuda.synchronize()


@pytest.mark.parametrize("mode", ["bf16", "exact", "digits", "digits2"])
def test_captured_matmul_keeps_its_workspace(mode):
    """A stream that ran its largest product can record a smaller one, whose K slices may
    want more workspace (then K stays whole); eager products that want more afterwards leave
    the recorded one its buffer."""
    K, N = 8960, 1536
    kw = dict(exact=mode == "exact", digits={"digits": 3, "digits2": 2}.get(mode, False))
    q, s = synthetic.quantized_linear(K, N, 5)
    packed = ops.pack_w8(q)
    x = torch.randn((1931, K), generator=torch.Generator(device="cuda").manual_seed(2), device="cuda")
    w64 = q.double() * s.double()
    more = [(n, ops.pack_w8(torch.cat([q] * (n // N), 1).contiguous()), torch.cat([s] * (n // N)))
            for n in (3072, 4608, 6144)]
    stream = torch.cuda.Stream()
    outs = {M: torch.empty((M, N), device="cuda") for M in (400, 300, 100)}
    with torch.cuda.stream(stream):
        ops.gemm_w8a32(x, packed, s, K, N, **kw)
    torch.cuda.synchronize()
    graphs = []
    for M, out in outs.items():
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            ops.gemm_w8a32(x[:M], packed, s, K, N, out=out, **kw)
        graphs.append(g)
        with torch.cuda.stream(stream):  # eager: the next capture finds its workspace
            ops.gemm_w8a32(x[:M], packed, s, K, N, **kw)
        torch.cuda.synchronize()
    xh = x[:400].double()
    if mode == "bf16":
        xh = x[:400].bfloat16().double()
    elif mode == "digits2":
        xh = torch.from_numpy(fixed_point_round(x[:400].cpu().numpy(), 2)[0]).cuda().double()
    want = xh @ w64
    first = {}
    for turn in range(4):
        for (M, out), g in zip(outs.items(), graphs):
            out.fill_(7.0)
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            first.setdefault(M, out.clone())
            assert torch.equal(out, first[M])
            err = float((out - want[:M]).abs().max())
            assert err < 2e-5 * float(want.abs().max()), (M, err)
        n, p, sc = more[turn % 3]
        with torch.cuda.stream(stream):
            ops.gemm_w8a32(x[:300 + 100 * turn], p, sc, K, n, **kw)
        torch.cuda.synchronize()


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("M,K,N", [(100, 256, 96), (490, 136, 6600)])
def test_prefill_gemm_accumulates(oracle, M, K, N, exact):
    q, s = synthetic.quantized_linear(K, N, 77)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn((M, K), generator=g, device="cuda")
    c0 = torch.randn((M, N), generator=g, device="cuda")
    c = c0.clone()
    ops.gemm_w8a32(x, ops.pack_w8(q), s, K, N, out=c, accumulate=True, exact=exact,
                   digits=not exact)
    torch.cuda.synchronize()
    want = oracle.blis_gemm_w8a32(x.cpu().numpy(), q.cpu().numpy(), s.cpu().numpy(),
                                  c0.cpu().numpy())
    check_close(c.cpu().numpy(), want)


def run_attn(bh, q, k, v, mask, heads, kv_heads, Lq, Lk):
    out = torch.empty_like(q)
    torch.cuda.synchronize()
    bma.check(bh.buddy_hip_prefill_attention(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), None if mask is None else mask.data_ptr(),
        out.data_ptr(), heads, kv_heads, 128, Lq, Lk, float(SCALE), None))
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("L", [16, 40, 512])
def test_prefill_attention_reference_shape(bh, oracle, L):
    """q, k, v all [12, L, 128] with an additive causal mask, the call shape of
    flash_attention_for_cpu_prefill_op; also the implicit causal mask."""
    H = 12
    g = torch.Generator(device="cuda").manual_seed(L)
    q, k, v = (torch.randn((H, L, 128), generator=g, device="cuda") for _ in range(3))
    mh = np.where(np.tril(np.ones((L, L), bool)), 0.0, -np.inf).astype(np.float32)
    want = oracle.prefill_flash_attention(q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(),
                                          mh, SCALE)
    got_mask = run_attn(bh, q, k, v, torch.from_numpy(mh).cuda(), H, H, L, L)
    got_causal = run_attn(bh, q, k, v, None, H, H, L, L)
    check_close(got_mask, want)
    check_close(got_causal, want)


def test_prefill_attention_gqa_and_longer_keys(bh, oracle):
    """2 KV heads read in place = 12 repeated heads; 37 queries over 100 keys
    (a prompt continuing after 63 cached positions)."""
    H, HKV, Lq, Lk = 12, 2, 37, 100
    g = torch.Generator(device="cuda").manual_seed(5)
    q = torch.randn((H, Lq, 128), generator=g, device="cuda")
    k = torch.randn((HKV, Lk, 128), generator=g, device="cuda")
    v = torch.randn((HKV, Lk, 128), generator=g, device="cuda")
    kk = k.repeat_interleave(H // HKV, dim=0).cpu().numpy()
    vv = v.repeat_interleave(H // HKV, dim=0).cpu().numpy()
    qi = np.arange(Lq)[:, None] + (Lk - Lq)
    mh = np.where(np.arange(Lk)[None, :] <= qi, 0.0, -np.inf).astype(np.float32)
    want = oracle.prefill_flash_attention(q.cpu().numpy(), kk, vv, mh, SCALE)
    check_close(run_attn(bh, q, k, v, None, H, HKV, Lq, Lk), want)


@pytest.mark.parametrize("Lq,Lk", [(1, 1), (5, 5), (17, 17), (33, 33), (95, 95), (129, 129),
                                   (1, 300), (16, 130), (50, 51), (200, 333)])
def test_prefill_attention_ragged_lengths(bh, oracle, Lq, Lk):
    """A workgroup takes a query block and its mirror image, and its wavefronts
    split the key blocks of the two: one query block alone, an odd number of
    them (the middle one on its own), a last block of 1 row, fewer key blocks than
    wavefronts, and prompts that continue behind cached positions -- with the
    implicit causal mask and with the same mask passed as a tensor."""
    H, HKV = 4, 2
    g = torch.Generator(device="cuda").manual_seed(1000 * Lq + Lk)
    q = torch.randn((H, Lq, 128), generator=g, device="cuda")
    k = torch.randn((HKV, Lk, 128), generator=g, device="cuda")
    v = torch.randn((HKV, Lk, 128), generator=g, device="cuda")
    kk = k.repeat_interleave(H // HKV, dim=0).cpu().numpy()
    vv = v.repeat_interleave(H // HKV, dim=0).cpu().numpy()
    qi = np.arange(Lq)[:, None] + (Lk - Lq)
    mh = np.where(np.arange(Lk)[None, :] <= qi, 0.0, -np.inf).astype(np.float32)
    want = oracle.prefill_flash_attention(q.cpu().numpy(), kk, vv, mh, SCALE)
    check_close(run_attn(bh, q, k, v, None, H, HKV, Lq, Lk), want)
    check_close(run_attn(bh, q, k, v, torch.from_numpy(mh).cuda(), H, HKV, Lq, Lk), want)


@pytest.mark.parametrize("H,HKV,Lq,Lk", [(32, 8, 272, 272), (12, 2, 600, 700)])
def test_prefill_attention_launches_of_several_rounds(bh, oracle, H, HKV, Lq, Lk):
    """More workgroups than compute units: the launch takes the form with four
    wavefronts per workgroup (two workgroups per compute unit)."""
    g = torch.Generator(device="cuda").manual_seed(H + Lq)
    q = torch.randn((H, Lq, 128), generator=g, device="cuda")
    k = torch.randn((HKV, Lk, 128), generator=g, device="cuda")
    v = torch.randn((HKV, Lk, 128), generator=g, device="cuda")
    kk = k.repeat_interleave(H // HKV, dim=0).cpu().numpy()
    vv = v.repeat_interleave(H // HKV, dim=0).cpu().numpy()
    qi = np.arange(Lq)[:, None] + (Lk - Lq)
    mh = np.where(np.arange(Lk)[None, :] <= qi, 0.0, -np.inf).astype(np.float32)
    want = oracle.prefill_flash_attention(q.cpu().numpy(), kk, vv, mh, SCALE)
    check_close(run_attn(bh, q, k, v, None, H, HKV, Lq, Lk), want)
    check_close(run_attn(bh, q, k, v, torch.from_numpy(mh).cuda(), H, HKV, Lq, Lk), want)


def test_prefill_attention_refuses_unaligned_operands(bh):
    t = torch.zeros(4 * 16 * 128 + 4, device="cuda")
    p = t.data_ptr()
    rc = bh.buddy_hip_prefill_attention(p + 4, p, p, None, p, 4, 4, 128, 16, 16, float(SCALE), None)
    assert rc == 1 and b"16-byte aligned" in bh.buddy_hip_last_error()


@pytest.mark.parametrize("precision", ["digits", "exact", "bf16", "digits2"])
def test_small_model_block_prefill_equals_token_by_token(oracle, precision):
    """Prefill of 40 prompt tokens as one block against 40 oracle decode steps:
    last-token logits, greedy token and every cache row written; then decode
    continues from the prefilled cache."""
    sess, host = synthetic.build_session(SMALL, context=0, keep_host=True, ln_jitter=0.1)
    om = oracle_model(oracle, SMALL, host)
    kv = [a.copy() for a in host["kv"]]
    toks = synthetic.first_tokens(SMALL, 40, seed=3).tolist()
    for pos, t in enumerate(toks):
        otok, ologits = om.decode_step(t, pos, kv)
    nxt, logits = sess.prefill(toks, 0, precision=precision)
    if precision not in ("bf16", "digits2"):
        check_close(logits, ologits)
        assert nxt == otok
        for j in range(2 * SMALL.layers):
            check_close(sess.get_kv(j)[:, :40, :], kv[j][:, :40, :])
        # decoding on from the prefilled cache
        tok = otok
        for step in range(6):
            n2, lg = sess.decode(tok, 40 + step)
            tok, olg = om.decode_step(tok, 40 + step, kv)
            check_close(lg, olg)
            assert n2 == tok
    elif precision == "digits2":
        # activations rounded to 2^-15 of their row's maximum in every matmul
        check_close(logits, ologits, rtol=5e-3, atol_frac=1e-3, normwise=1e-3)
        assert nxt == otok
    else:
        # activations cast to bf16 in every matmul of every layer: compared at
        # the looser bound that rounding allows
        check_close(logits, ologits, rtol=5e-2, atol_frac=2e-2, normwise=2e-2)
    sess.close()


def test_prefill_in_two_blocks_and_after_decode_steps(oracle):
    """A prompt fed as two blocks (the second starts at position 24 and attends
    to the cache rows of the first), then decode steps, then a third block: the
    same logits and cache rows as 53 oracle decode steps."""
    sess, host = synthetic.build_session(SMALL, context=0, keep_host=True, ln_jitter=0.1)
    om = oracle_model(oracle, SMALL, host)
    kv = [a.copy() for a in host["kv"]]
    toks = synthetic.first_tokens(SMALL, 53, seed=11).tolist()
    want = []
    for pos, t in enumerate(toks):
        otok, ologits = om.decode_step(t, pos, kv)
        want.append((otok, ologits))
    nxt, logits = sess.prefill(toks[:24], 0)
    check_close(logits, want[23][1])
    assert nxt == want[23][0]
    nxt, logits = sess.prefill(toks[24:40], 24)
    check_close(logits, want[39][1])
    assert nxt == want[39][0]
    for pos in range(40, 43):  # three tokens one by one
        n2, lg = sess.decode(toks[pos], pos)
        check_close(lg, want[pos][1])
        assert n2 == want[pos][0]
    nxt, logits = sess.prefill(toks[43:53], 43)  # a ragged block of 10
    check_close(logits, want[52][1])
    assert nxt == want[52][0]
    for j in range(2 * SMALL.layers):
        check_close(sess.get_kv(j)[:, :53, :], kv[j][:, :53, :])
    sess.close()


# the attention that shares out key tiles: row blocks of 256 rows (42.67 tokens of six heads)
# and tiles of 32 keys at, below and beyond their edges, one and several KV heads, groups of
# one to eight heads, one row behind a long context, more blocks than workgroups take whole
@pytest.mark.parametrize("heads,kv_heads,before,n", [
    (6, 1, 128, 1), (6, 1, 159, 1), (6, 1, 160, 43), (6, 1, 0, 641), (6, 1, 0, 683), (6, 1, 700, 130),
    (2, 2, 130, 255), (2, 2, 0, 769), (8, 1, 129, 32), (8, 1, 0, 673), (3, 1, 1000, 86),
    (4, 2, 300, 127), (12, 2, 0, 650)])
def test_prompt_attention_equals_token_by_token(heads, kv_heads, before, n):
    """A prompt as one block against the same tokens through the decode step, whose
    attention is another kernel: logits of the last row and the second layer's cache rows,
    which hold what the first layer's attention gave."""
    shape = Shape(layers=2, hidden=256, heads=heads, kv_heads=kv_heads, head_dim=128, inter=256,
                  vocab=320, max_len=before + n + 8)
    toks = synthetic.first_tokens(shape, n, seed=before + n).astype(np.int32)
    for precision in ("digits", "exact"):
        sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
        _, got = sess.prefill(toks, before, precision=precision)
        rows = [sess.get_kv(j)[:, before:before + n] for j in (2, 3)]
        sess.close()
        sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
        for i, t in enumerate(toks):
            _, want = sess.decode(int(t), before + i, want_logits=i + 1 == n)
        check_close(got, want)
        for j in (2, 3):
            check_close(rows[j - 2], sess.get_kv(j)[:, before:before + n])
        sess.close()


# on both sides of the line between the two attentions: one token, behind whole key tiles and
# behind a last one of a single key; tokens that fill blocks of 256 rows and some that do not;
# few heads and many
@pytest.mark.parametrize("heads,kv_heads,before,n,precision,split", [
    (6, 1, 128, 1, "digits", 0), (6, 1, 600, 1, "digits", 1), (6, 1, 607, 1, "exact", 1),
    (8, 1, 129, 32, "exact", 0), (8, 1, 600, 32, "exact", 1), (12, 2, 128, 300, "digits", 0),
    (12, 2, 400, 300, "digits", 1), (12, 2, 0, 801, "digits", 0), (12, 2, 0, 901, "digits", 1),
    (64, 8, 128, 27, "digits", 0), (64, 8, 1200, 33, "digits", 1), (1, 1, 128, 96, "exact", 1)])
def test_which_prompt_attention(bh, heads, kv_heads, before, n, precision, split, hidden=256):
    shape = Shape(layers=2, hidden=hidden, heads=heads, kv_heads=kv_heads, head_dim=128, inter=256,
                  vocab=320, max_len=before + n + 8)
    toks = synthetic.first_tokens(shape, n, seed=before + n).astype(np.int32)
    sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
    bh.buddy_hip_variant_reset()
    _, got = sess.prefill(toks, before, precision=precision)
    assert tiles_run(bh)["attn_prompt_kernel<256>"] == split * shape.layers
    rows = [sess.get_kv(j)[:, before:before + n] for j in (2, 3)]
    sess.close()
    sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
    for i, t in enumerate(toks):
        _, want = sess.decode(int(t), before + i, want_logits=i + 1 == n)
    check_close(got, want)
    for j in (2, 3):
        check_close(rows[j - 2], sess.get_kv(j)[:, before:before + n])
    sess.close()


# the same prompt: digits that the output product makes itself, rows that take a launch of their own
@pytest.mark.parametrize("heads,kv_heads,before,n,precision,split", [
    (12, 2, 310, 27, "digits", 0), (12, 2, 310, 27, "exact", 1), (12, 2, 256, 16, "digits", 0),
    (12, 2, 700, 16, "digits", 1), (64, 8, 390, 128, "digits", 0), (64, 8, 390, 256, "digits", 1)])
def test_which_prompt_attention_by_conversion(bh, heads, kv_heads, before, n, precision, split):
    test_which_prompt_attention(bh, heads, kv_heads, before, n, precision, split)


# output products of more channels than the chip has compute units for rows of them as they come
@pytest.mark.parametrize("hidden,made", [(4096, 2), (4224, 0)])
def test_which_prompt_attention_by_product(bh, hidden, made):
    test_which_prompt_attention(bh, 8, 1, 390, 100, "digits", 0 if made else 1, hidden=hidden)
    assert sum(v for k, v in tiles_run(bh).items() if k.startswith("gemm_w8_i8_rows_kernel<3, 9>")) == made


# q | k | v with the rotation and the cache rows behind it: K in more slices than are asked for at
# once (2 trips), in two to eight (1) and whole (0), of digit planes and of terms; one head and many;
# tokens behind a context
@pytest.mark.parametrize("precision", ["digits", "digits2", "exact", "bf16"])
@pytest.mark.parametrize("hidden,heads,kv_heads,before,n,trips", [
    (2048, 1, 1, 0, 3, (2, 2)), (1536, 2, 1, 7, 40, (2, 2)), (1536, 12, 2, 0, 27, (1, 2)),
    (1536, 12, 2, 5, 100, (1, 1)), (320, 6, 3, 130, 17, (0, 0)), (64, 12, 2, 0, 33, (0, 0)),
    (256, 12, 2, 3, 900, (0, 0))])
def test_rotation_behind_qkv(bh, hidden, heads, kv_heads, before, n, trips, precision):
    shape = Shape(layers=2, hidden=hidden, heads=heads, kv_heads=kv_heads, head_dim=128, inter=64, vocab=320,
                  max_len=before + n + 8)
    toks = synthetic.first_tokens(shape, n, seed=n).astype(np.int32)
    sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
    bh.buddy_hip_variant_reset()
    sess.prefill(toks, before, precision=precision)
    ran, trips = tiles_run(bh), trips[not precision.startswith("digits")]
    assert [ran[f"reduce_slices_rope_kernel<{k}>"] for k in (1, 2)] == \
        [shape.layers * (trips == k) for k in (1, 2)]
    rows = [sess.get_kv(j)[:, :before + n] for j in range(4)]
    sess.close()
    sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
    for i, t in enumerate(toks):
        sess.decode(int(t), before + i, want_logits=False)
    for j in range(4):
        want = sess.get_kv(j)[:, :before + n]
        np.testing.assert_array_equal(rows[j][:, :before], want[:, :before])
        rows[j], want = rows[j][:, before:], want[:, before:]
        if precision in ("digits", "exact"):
            check_close(rows[j], want)
        else:  # some ten roundings on the way: of 2^-15 of a row's largest value, of 2^-9 of each
            bound = 2.0**-10 if precision == "digits2" else 10 * 2.0**-9
            assert np.linalg.norm(rows[j] - want) < bound * np.linalg.norm(want)
    sess.close()


# the rotation within q | k | v's product: tiles of one head and of two, of which one may be queries and one
# keys, or keys and values, or the last alone; part of a tile of 32 rows, whole ones, one row more; alone,
# where keys and values leave as terms too, and behind a context
@pytest.mark.parametrize("precision", ["digits", "digits2"])
@pytest.mark.parametrize("heads,kv_heads,before,n,gp", [
    (12, 2, 0, 33, (1, 1)), (3, 3, 0, 17, (1, 1)), (8, 1, 9, 64, (1, 1)), (12, 2, 0, 901, (2, 1)),
    (12, 2, 0, 1376, (2, 2)), (15, 5, 0, 800, (2, 0)), (15, 3, 3, 864, (2, 0))])
def test_rotation_within_qkv(bh, heads, kv_heads, before, n, gp, precision):
    shape = Shape(layers=2, hidden=256, heads=heads, kv_heads=kv_heads, head_dim=128, inter=64, vocab=320,
                  max_len=before + n + 8)
    toks = synthetic.first_tokens(shape, n, seed=n).astype(np.int32)
    rows = []
    for by_token in (False, True):
        sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
        bh.buddy_hip_variant_reset()
        if by_token:
            for i, t in enumerate(toks):
                sess.decode(int(t), before + i, want_logits=False)
        else:
            sess.prefill(toks, before, precision=precision)
            D = 3 if precision == "digits" else 2  # (0: tiles that leave it to a launch behind them)
            assert [tiles_run(bh)[f"gemm_w8_i8 rotates<{D}, {g}>"] for g in (1, 2)] == \
                [shape.layers * (gp[precision == "digits2"] == g) for g in (1, 2)]
        rows.append([sess.get_kv(j)[:, :before + n] for j in range(4)])
        sess.close()
    for got, want in zip(*rows):
        np.testing.assert_array_equal(got[:, :before], want[:, :before])
        got, want = got[:, before:], want[:, before:]
        if precision == "digits":
            check_close(got, want)
        else:  # roundings of 2^-15 of a row's largest value, as in the test above
            assert np.linalg.norm(got - want) < 2.0**-10 * np.linalg.norm(want)


# bfloat16 modes: gate and up as one product whose result leaves as terms, on tiles of one and of
# two channel tiles per wavefront, a result that ends inside 64 channels; the norm behind o and down
# in the kernel that adds slices of K and as a launch of its own; the attention's fold as terms
@pytest.mark.parametrize("precision", ["bf16", "exact"])
@pytest.mark.parametrize("hidden,inter,before,n,gp", [
    (256, 272, 0, 5, 1), (256, 1040, 0, 33, 1), (256, 8976, 0, 65, 0), (256, 8976, 0, 150, 2),
    (1536, 8960, 0, 300, 2), (1536, 48, 600, 40, 1), (320, 4112, 600, 70, 0)])
def test_prompt_layers_in_bf16_terms(bh, hidden, inter, before, n, gp, precision):
    shape = Shape(layers=2, hidden=hidden, heads=6, kv_heads=1, head_dim=128, inter=inter, vocab=320,
                  max_len=before + n + 8)
    toks = synthetic.first_tokens(shape, n, seed=n + inter).astype(np.int32)
    sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
    bh.buddy_hip_variant_reset()
    _, got = sess.prefill(toks, before, precision=precision)
    ran = {k for k, v in tiles_run(bh).items() if v and k.startswith("gemm_w8_bf16_kernel pair")}
    terms = 1 if precision == "bf16" else 3
    assert len(ran) == 1 and (gp == 0 or ran == {f"gemm_w8_bf16_kernel pair<{terms}, {gp}>"}), ran
    rows = [sess.get_kv(j)[:, before:before + n] for j in (2, 3)]
    sess.close()
    sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
    for i, t in enumerate(toks):
        _, want = sess.decode(int(t), before + i, want_logits=i + 1 == n)
    pairs = [(got, want)] + [(rows[j - 2], sess.get_kv(j)[:, before:before + n]) for j in (2, 3)]
    sess.close()
    for g, w in pairs:
        if precision == "exact":
            check_close(g, w)
        else:  # 2^-9 per activation, some ten roundings on the way
            g, w = np.asarray(g, np.float64), np.asarray(w, np.float64)
            assert np.linalg.norm(g - w) < 10 * 2.0**-9 * np.linalg.norm(w)


def test_workspace_of_the_prompt_attention_follows_the_session(bh):
    """One KV head behind 640 positions has 20 tiles of keys for 20 workgroups: 5 MB of partial
    results, not the 67 MB of a full chip."""
    shape = Shape(layers=1, hidden=256, heads=6, kv_heads=1, head_dim=128, inter=256, vocab=320,
                  max_len=640)
    sess, _ = synthetic.build_session(shape, context=600, ln_jitter=0.1)
    sess.prefill(np.arange(30, dtype=np.int32), 0)  # the other buffers
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    bh.buddy_hip_variant_reset()
    sess.prefill(np.arange(30, dtype=np.int32), 600)
    assert tiles_run(bh)["attn_prompt_kernel<256>"] == 1
    assert free - torch.cuda.mem_get_info()[0] < 16 << 20
    sess.close()


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_prompt_attention_keeps_non_finite_tokens_from_earlier_rows(bad):
    """A token in the middle of a long prompt whose embedding is not finite: rows that do not
    see it are what they are without, bit for bit; rows that do are NaN."""
    shape = Shape(layers=2, hidden=256, heads=6, kv_heads=1, head_dim=128, inter=256, vocab=320,
                  max_len=720)
    toks = (synthetic.first_tokens(shape, 700, seed=1) % 300).astype(np.int32)
    at = 450
    toks[at] = 310
    sess, _ = synthetic.build_session(shape, context=0, ln_jitter=0.1)
    embed = sess._globals["embed"]

    def rows():
        sess.prefill(toks, 0)
        return [sess.get_kv(j)[0, :700].copy() for j in (2, 3)]

    clean = rows()
    embed[310, 7] = bad
    torch.cuda.synchronize()
    for got, want in zip(rows(), clean):
        np.testing.assert_array_equal(got[:at], want[:at])
        assert np.isnan(got[at:]).any(axis=1).all()
    sess.close()


@pytest.mark.parametrize("precision", ["digits", "exact"])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), 3.4e38])
def test_prompt_attention_of_a_key_beyond_bfloat16(bad, precision):
    """A cached key with one channel infinite, or larger than any bfloat16 value: a row of
    whose query that channel is negative gives it a score of -inf and no weight.  Finite and
    non-finite rows are those of the decode step, whose attention is another kernel."""
    before, n = 200, 150
    shape = Shape(layers=2, hidden=256, heads=1, kv_heads=1, head_dim=128, inter=256, vocab=320,
                  max_len=before + n + 8)
    toks = synthetic.first_tokens(shape, n, seed=3).astype(np.int32)
    rows = []
    for by_token in (False, True):
        sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
        k = sess.get_kv(0)
        k[0, 77, 9] = bad
        sess.set_kv(0, k)
        if by_token:
            for i, t in enumerate(toks):
                sess.decode(int(t), before + i, want_logits=False)
        else:
            sess.prefill(toks, before, precision=precision)
        rows.append([sess.get_kv(j)[0, before:before + n] for j in (2, 3)])
        sess.close()
    for got, want in zip(*rows):
        finite = np.isfinite(want).all(axis=1)
        assert finite.sum() > n // 4
        if np.isinf(bad):
            assert (~finite).sum() > n // 4
        assert not np.isfinite(got[~finite]).all(axis=1).any()
        check_close(got[finite], want[finite])


@pytest.mark.parametrize("heads,kv_heads", [(20, 4), (100, 20)])
def test_prompt_attention_of_a_key_beyond_bfloat16_in_long_rows(heads, kv_heads):
    """More heads than a workgroup of the fold has half wavefronts; a row of 12800 values,
    which the kernel that writes its digits computes twice."""
    before, n = 600, 17
    shape = Shape(layers=2, hidden=256, heads=heads, kv_heads=kv_heads, head_dim=128, inter=256,
                  vocab=320, max_len=before + n + 8)
    toks = synthetic.first_tokens(shape, n, seed=4).astype(np.int32)
    rows = []
    for by_token in (False, True):
        sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
        k = sess.get_kv(0)
        k[kv_heads - 1, 77, 9] = 3.4e38
        sess.set_kv(0, k)
        if by_token:
            for i, t in enumerate(toks):
                sess.decode(int(t), before + i, want_logits=False)
        else:
            sess.prefill(toks, before)
        rows.append([sess.get_kv(j)[:, before:before + n] for j in (2, 3)])
        sess.close()
    for got, want in zip(*rows):
        assert np.isfinite(want).all()
        check_close(got, want)


# a prompt alone on the terms that the rotation leaves: part of a block of 32 rows, a tile of 32 keys and one more, a
# tile to each wavefront and one more, groups that divide a block and that do not; the rotation in the
# kernel that adds slices and as a launch of its own, q | k | v in f32
@pytest.mark.parametrize("heads,kv_heads,n", [(6, 1, 17), (12, 2, 18), (12, 2, 27), (4, 4, 32), (6, 2, 33), (5, 1, 100),
                                              (8, 1, 257), (12, 2, 300), (3, 3, 545)])
@pytest.mark.parametrize("qkv_f32", [False, True])
def test_prompt_attention_on_terms_of_the_rotation(bh, heads, kv_heads, n, qkv_f32):
    """Behind a longer prompt with a token that is not finite, whose terms are left in the buffer."""
    shape = Shape(layers=2, hidden=256, heads=heads, kv_heads=kv_heads, head_dim=128, inter=256, vocab=320,
                  max_len=n + 48)
    toks = (synthetic.first_tokens(shape, n, seed=n) % 300).astype(np.int32)
    sess, g = DecoderSession(shape), synthetic.make_globals(shape)
    g["embed"][310, 7] = float("nan")
    sess.set_globals(g["embed"], g["inv_freq"], g["ln_f"], g["w_lm"], g["s_lm"])
    for i in range(shape.layers):
        w = synthetic.make_layer(shape, i, 0.1)
        for t in "qkv" if qkv_f32 else "":
            w["f" + t] = w.pop("w" + t).float() * w.pop("s" + t)
            w["b" + t] = torch.zeros(w["f" + t].shape[1], device="cuda")
        sess.set_layer(i, w)
    torch.cuda.synchronize()
    sess.prefill(np.concatenate([toks[:1], [310], np.tile(toks, 40)[:n + 20]]).astype(np.int32), 0)
    bh.buddy_hip_variant_reset()
    _, got = sess.prefill(toks, 0)
    assert tiles_run(bh)["attn_terms_kernel<32>"] == shape.layers
    rows = [sess.get_kv(j)[:, :n] for j in (2, 3)]
    for i, t in enumerate(toks):
        _, want = sess.decode(int(t), i, want_logits=i + 1 == n)
    check_close(got, want)
    for j in (2, 3):
        check_close(rows[j - 2], sess.get_kv(j)[:, :n])
    sess.close()


@pytest.mark.parametrize("heads,n,kernel", [(12, 1, None), (12, 27, None), (12, 300, None), (64, 600, "attn_prompt_kernel<256>")])
def test_every_bit_of_a_prompt_alone(bh, heads, n, kernel):
    """Where every f32 bit is asked for, a prompt's attention is on f32 instructions, that of long ones on terms."""
    shape = Shape(layers=2, hidden=256, heads=heads, kv_heads=heads // 4, head_dim=128, inter=256, vocab=320,
                  max_len=n + 8)
    toks = synthetic.first_tokens(shape, n, seed=n).astype(np.int32)
    sess, _ = synthetic.build_session(shape, context=0, ln_jitter=0.1)
    bh.buddy_hip_variant_reset()
    sess.prefill(toks, 0, precision="exact")
    ran = tiles_run(bh)
    for name in ("attn_terms_kernel<32>", "attn_prompt_kernel<256>"):
        assert ran[name] == (shape.layers if name == kernel else 0)
    rows = [sess.get_kv(j)[:, :n] for j in (2, 3)]
    for i, t in enumerate(toks):
        sess.decode(int(t), i, want_logits=False)
    for j in (2, 3):
        check_close(rows[j - 2], sess.get_kv(j)[:, :n])
    sess.close()


@pytest.mark.parametrize("which,powers", [
    ("v", [0, -20, 9, 3]), ("v", [30, 31, 28, 30]), ("v", [-100, -90, -95, -100]), ("k", [-30, 0, -3, 2]),
    ("k", [-120, -120, -119, -118]), ("channel", [10, 10, 10, 10]), ("zero", [0, 0, 0, 0])])
def test_prompt_attention_over_magnitudes(which, powers):
    """Rows of cached keys or values that differ by powers of two, are all large or all tiny; one channel of the
    values 2^10 above the others; rows of zeros: as the decode step has them, whose attention is f32."""
    before, n = 600, 70
    shape = Shape(layers=2, hidden=256, heads=6, kv_heads=1, head_dim=128, inter=256, vocab=320,
                  max_len=before + n + 8)
    toks = synthetic.first_tokens(shape, n, seed=6).astype(np.int32)
    rows = []
    for by_token in (False, True):
        sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
        t = sess.get_kv(0 if which == "k" else 1)
        if which == "zero":
            t[0, 5:before:7] = 0
        elif which == "channel":
            t[0, :before, 77] *= 2.0**10
        else:
            t[0, :before] *= 2.0**np.array(powers, np.float32)[np.arange(before) % 4][:, None]
        sess.set_kv(0 if which == "k" else 1, t)
        if by_token:
            for i, tok in enumerate(toks):
                sess.decode(int(tok), before + i, want_logits=False)
        else:
            sess.prefill(toks, before, precision="exact")
        rows.append([sess.get_kv(j)[0, before:before + n] for j in (2, 3)])
        sess.close()
    for got, want in zip(*rows):
        assert np.isfinite(want).all()
        check_close(got, want)


# Values that are zero, or so small beside others that their scales are far apart: their keys have weight all the
# same.  The first tile of 32 keys a wavefront or a workgroup takes, tiles further on, all there are.
@pytest.mark.parametrize("precision", ["digits", "exact"])
@pytest.mark.parametrize("rows,power", [((0, 32), None), ((0, 64), None), ((96, 128), None), ((0, 600), None),
                                        ((0, 32), -120), ((0, 600), -105), ((0, 600), -40), ((31, 600), None),
                                        ((1, 600, 3), None), ((0, 600, 2), -60), ((0, 600, 2), -38),
                                        ((1, 600, 3), 38)])
@pytest.mark.parametrize("beside", [0, 9, 30])
def test_prompt_attention_of_values_without_magnitude(bh, rows, power, beside, precision):
    """Behind a context, in one of two KV heads (in both a common factor of the sums of weights would be lost in the
    norm that follows); the others' cached values times 2^beside: as the decode step has them."""
    before, n = 600, 70
    shape = Shape(layers=2, hidden=256, heads=6, kv_heads=2, head_dim=128, inter=256, vocab=320,
                  max_len=before + n + 8)
    toks = synthetic.first_tokens(shape, n, seed=6).astype(np.int32)
    got = []
    for by_token in (False, True):
        sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
        t = sess.get_kv(1)
        few = t[0, slice(*rows)] * np.float32(0.0 if power is None else 2.0**power)
        t[:, :before] *= np.float32(2.0**beside)
        t[0, slice(*rows)] = few
        sess.set_kv(1, t)
        if by_token:
            for i, tok in enumerate(toks):
                sess.decode(int(tok), before + i, want_logits=False)
        else:
            bh.buddy_hip_variant_reset()
            sess.prefill(toks, before, precision=precision)
            assert tiles_run(bh)["attn_prompt_kernel<256>"] == shape.layers
        got.append([sess.get_kv(j)[:, before:before + n] for j in (2, 3)])
        sess.close()
    for a, b in zip(*got):
        check_close(a, b)


# ... of a prompt alone, whose tokens' embedding is zero, or so small that their values are, on all three kernels
@pytest.mark.parametrize("heads,kv_heads,n,precision,kernel", [
    (12, 2, 300, "digits", "attn_terms_kernel<32>"), (64, 8, 320, "digits", "attn_prompt_kernel<256>"),
    (12, 2, 300, "exact", None)])
@pytest.mark.parametrize("at", [(0, 32), (32, 33), (64, 65), (96, 160), (0, 257)])
@pytest.mark.parametrize("size", [0.0, 2.0**-110])
def test_prompt_alone_of_values_without_magnitude(bh, heads, kv_heads, n, precision, kernel, at, size):
    shape = Shape(layers=2, hidden=256, heads=heads, kv_heads=kv_heads, head_dim=128, inter=256, vocab=320,
                  max_len=n + 8)
    toks = (synthetic.first_tokens(shape, n, seed=n) % 300).astype(np.int32)
    toks[at[0]:at[1]] = 310
    sess, g = DecoderSession(shape), synthetic.make_globals(shape)
    g["embed"][310] *= size
    sess.set_globals(g["embed"], g["inv_freq"], g["ln_f"], g["w_lm"], g["s_lm"])
    for i in range(shape.layers):
        sess.set_layer(i, synthetic.make_layer(shape, i, 0.1))
    torch.cuda.synchronize()
    bh.buddy_hip_variant_reset()
    sess.prefill(toks, 0, precision=precision)
    if kernel:
        assert tiles_run(bh)[kernel] == shape.layers
    got = [sess.get_kv(j)[:, :n] for j in range(4)]
    for i, t in enumerate(toks):
        sess.decode(int(t), i, want_logits=False)
    for j in range(4):
        check_close(got[j], sess.get_kv(j)[:, :n])
    sess.close()


@pytest.mark.parametrize("at", [0, 3, 4, 15, 16, 31, 63, 70])
@pytest.mark.parametrize("size", [3.4e38, 8e38])  # above the largest bfloat16 value; infinite
def test_prompt_attention_of_a_value_beyond_bfloat16(at, size):
    """One channel of one token's value is huge or infinite, its key is not: rows ahead of
    the token are what they are without, bit for bit, also in its tile of 32 keys.  Behind it
    a huge value changes its own channel alone (o_proj takes nothing from that channel, and
    the other channels give what they give without it); an infinite one makes NaN of 0 * inf."""
    before, n, c, big = 192, 96, 5, 310
    shape = Shape(layers=2, hidden=256, heads=2, kv_heads=1, head_dim=128, inter=256, vocab=320,
                  max_len=before + n + 8)

    def session(factor):
        sess = DecoderSession(shape)
        g = synthetic.make_globals(shape)
        g["embed"][:, 0] = 0.0
        g["embed"][big, 0] = 0.05
        sess.set_globals(g["embed"], g["inv_freq"], g["ln_f"], g["w_lm"], g["s_lm"])
        for i in range(shape.layers):
            w = synthetic.make_layer(shape, i, 0.1)
            if i == 0:  # channel c of the values is that of the big token's embedding, or 0
                w["wv"][:, c] = 0
                w["wv"][0, c] = 100
                w["sv"][c] = factor
                w["wo"][c::128] = 0
            sess.set_layer(i, w)
        for j in range(2 * shape.layers):
            sess.set_kv(j, synthetic.make_kv(shape, j, before))
        torch.cuda.synchronize()
        return sess

    toks = (synthetic.first_tokens(shape, n, seed=5) % 300).astype(np.int32)
    toks[at] = big
    rows, factor = [], 1.0
    for want_size in (None, size):
        sess = session(factor)
        sess.prefill(toks, before, precision="exact")
        rows.append([sess.get_kv(j)[0, before:before + n] for j in (2, 3)])
        value = abs(float(sess.get_kv(1)[0, before + at, c]))
        if want_size is None:
            factor = size / value
        else:
            assert np.isinf(value) if size > 3.5e38 else 3.3962e38 < value < np.inf
        sess.close()
    for want, got in zip(*rows):
        np.testing.assert_array_equal(got[:at], want[:at])
        if size > 3.5e38:
            assert not np.isfinite(got[at:]).all(axis=1).any()
        else:
            check_close(got[at:], want[at:])


@pytest.mark.parametrize("precision", ["digits", "exact"])
def test_wide_hidden_size_through_the_slice_adding_norm_kernel(bh, oracle, precision):
    """hidden = 9216: the kernel that adds the K slices of o_proj / down and
    writes the next RMSNorm's digit planes or terms keeps two copies of a row in LDS,
    72 KiB here -- more than the 64 KiB a kernel gets without asking.  A
    prompt of 64 tokens (one row tile: the matmuls then split K over
    workgroups) against 64 oracle decode steps."""
    shape = Shape(layers=2, hidden=9216, heads=8, kv_heads=2, head_dim=128, inter=2048,
                  vocab=512, max_len=128, rms_eps=1e-6)
    sess, host = synthetic.build_session(shape, context=0, keep_host=True, ln_jitter=0.1)
    om = oracle_model(oracle, shape, host)
    kv = [a.copy() for a in host["kv"]]
    toks = synthetic.first_tokens(shape, 64, seed=23).tolist()
    for pos, t in enumerate(toks):
        otok, ologits = om.decode_step(t, pos, kv)
    bh.buddy_hip_variant_reset()
    nxt, logits = sess.prefill(toks, 0, precision=precision)
    if precision == "exact":
        assert tiles_run(bh)["add_slices_norm_kernel<1>"]
    check_close(logits, ologits)
    assert nxt == otok
    for j in range(2 * shape.layers):
        check_close(sess.get_kv(j)[:, :64, :], kv[j][:, :64, :])
    sess.close()


@pytest.mark.parametrize("precision", ["digits", "exact"])
@pytest.mark.parametrize("n", [20, 70])
def test_hidden_size_beyond_the_slice_adding_norm_kernel(bh, n, precision):
    """hidden = 12352: a row is longer than that kernel holds; the norm is a launch of its own
    behind products with whole sums and with K in slices."""
    shape = Shape(layers=2, hidden=12352, heads=8, kv_heads=2, head_dim=128, inter=2048,
                  vocab=320, max_len=128)
    toks = synthetic.first_tokens(shape, n, seed=n).astype(np.int32)
    sess, _ = synthetic.build_session(shape, context=0, ln_jitter=0.1)
    bh.buddy_hip_variant_reset()
    _, got = sess.prefill(toks, 0, precision=precision)
    if precision == "exact":
        assert bool(tiles_run(bh)["add_slices_kernel and a norm behind it<1>"]) == (n == 20)
    rows = [sess.get_kv(j)[:, :n].copy() for j in range(4)]
    for i, t in enumerate(toks):
        _, want = sess.decode(int(t), i, want_logits=i + 1 == n)
    check_close(got, want)
    for j in range(4):
        check_close(rows[j], sess.get_kv(j)[:, :n])
    sess.close()


@pytest.mark.timeout(900)
def test_qwen2_1p5b_shape_512_token_prefill(oracle):
    """The full 28-layer shape, a prompt of 512 tokens as one block (digit-plane
    matmuls, the default) against 512 oracle decode steps: last-row logits, the
    greedy token, and the cache rows of the first and the last layer; then the
    last-row logits of the three other activation modes."""
    shape = Shape()
    sess, host = synthetic.build_session(shape, context=0, keep_host=True)
    om = oracle_model(oracle, shape, host)
    kv = host["kv"]
    toks = synthetic.first_tokens(shape, 512, seed=21).tolist()
    for pos, t in enumerate(toks):
        otok, ologits = om.decode_step(t, pos, kv)
    nxt, logits = sess.prefill(toks, 0)
    check_close(logits, ologits)
    top2 = np.partition(ologits, -2)[-2:]
    assert nxt == otok, f"top-2 logit margin {float(top2[1] - top2[0]):.3e}"
    for j in (0, 1, 2 * shape.layers - 2, 2 * shape.layers - 1):
        check_close(sess.get_kv(j)[:, :512, :], kv[j][:, :512, :])
    # one decode step on from the prefilled cache
    n2, lg = sess.decode(otok, 512)
    t2, olg = om.decode_step(otok, 512, kv)
    check_close(lg, olg)
    assert n2 == t2
    # the same prompt in the other activation modes, at the bound each one's
    # rounding allows over 28 layers: every f32 bit (three bf16 terms) at the f32
    # bar, two digit planes (2^-15 of a row's maximum per matmul), activations cast
    # to bf16 (2^-9 per element: the precision BASELINE's prefill case names)
    _, exact = sess.prefill(toks, 0, precision="exact")
    check_close(exact, ologits)
    _, two = sess.prefill(toks, 0, precision="digits2")
    nw2 = check_close(two, ologits, rtol=2e-2, atol_frac=3e-3, normwise=3e-3)
    _, cast = sess.prefill(toks, 0, precision="bf16")
    nwc = check_close(cast, ologits, rtol=5e-2, atol_frac=2e-2, normwise=2e-2)
    print(f"norm-wise error of the last-row logits: two planes {nw2:.2e}, bf16 cast {nwc:.2e}")
    assert nw2 < nwc
    for lg_mode in (exact, two, cast):
        assert int(np.argmax(lg_mode)) == otok or float(top2[1] - top2[0]) < 0.05 * float(
            np.abs(ologits).max())
    sess.close()


def test_session_prefill_refuses_overflow(bh):
    sess, _ = synthetic.build_session(SMALL, context=0)
    with pytest.raises(bma.BuddyHipError):
        sess.prefill(list(range(10)), SMALL.max_len - 5)
    sess.close()


# Output and down products of few rows that are turned into digits within the product: every number
# of chunks to a slice, a last slice of fewer, K that ends inside a chunk, one and two tiles of rows;
# and one row too many
@pytest.mark.parametrize("precision", ["digits", "digits2"])
@pytest.mark.parametrize("hidden,heads,inter,n,chunks", [
    (384, 3, 336, 18, {2}), (1536, 12, 8960, 27, {2, 9}), (1536, 12, 8960, 64, {3, 14}), (256, 4, 4112, 33, {2, 5}),
    (100, 1, 16, 17, {2}), (1536, 12, 336, 128, {2, 5}), (384, 3, 336, 129, set())])
def test_few_rows_become_digits_within_the_product(bh, hidden, heads, inter, n, chunks, precision):
    shape = Shape(layers=2, hidden=hidden, heads=heads, kv_heads=1, head_dim=128, inter=inter, vocab=320, max_len=n + 8) \
        if heads <= 8 else Shape(layers=2, hidden=hidden, heads=heads, kv_heads=2, head_dim=128, inter=inter, vocab=320,
                                 max_len=n + 8)
    toks = synthetic.first_tokens(shape, n, seed=n + inter).astype(np.int32)
    sess, _ = synthetic.build_session(shape, context=0, ln_jitter=0.1)
    bh.buddy_hip_variant_reset()
    _, got = sess.prefill(toks, 0, precision=precision)
    planes = 3 if precision == "digits" else 2
    ran = {k for k, v in tiles_run(bh).items() if v and k.startswith("gemm_w8_i8_rows_kernel")}
    assert ran == {f"gemm_w8_i8_rows_kernel<{planes}, {c}>" for c in chunks}
    rows = [sess.get_kv(j)[:, :n] for j in (2, 3)]
    sess.close()
    sess, _ = synthetic.build_session(shape, context=0, ln_jitter=0.1)
    for i, t in enumerate(toks):
        _, want = sess.decode(int(t), i, want_logits=i + 1 == n)
    pairs = [(got, want)] + [(rows[j - 2], sess.get_kv(j)[:, :n]) for j in (2, 3)]
    sess.close()
    for g, w in pairs:
        if planes == 3:
            check_close(g, w)
        else:  # some ten roundings on the way, of 2^-15 of a row's largest value
            g, w = np.asarray(g, np.float64), np.asarray(w, np.float64)
            assert np.linalg.norm(g - w) < 2.0**-10 * np.linalg.norm(w)


# Up to 16 tokens through the products of a decode step: every row count at which their kernels change,
# q | k | v of enough channels and of fewer, behind a context whose attention leaves parts to fold, gate and up
# apart (a width that sixteen does not divide), and one token too many
@pytest.mark.parametrize("precision", ["digits", "digits2", "bf16"])
@pytest.mark.parametrize("hidden,heads,kv_heads,inter,before,n", [
    (384, 12, 2, 336, 0, 1), (384, 12, 2, 336, 0, 2), (1088, 12, 2, 4112, 7, 5), (384, 12, 2, 336, 3, 9),
    (1536, 12, 2, 8960, 0, 16), (384, 12, 2, 336, 400, 8), (384, 3, 1, 336, 0, 6), (384, 12, 2, 330, 0, 4),
    (384, 12, 2, 336, 0, 17)])
def test_prompts_of_few_tokens(bh, hidden, heads, kv_heads, inter, before, n, precision):
    shape = Shape(layers=2, hidden=hidden, heads=heads, kv_heads=kv_heads, head_dim=128, inter=inter, vocab=320,
                  max_len=before + n + 8)
    toks = synthetic.first_tokens(shape, n, seed=n + inter).astype(np.int32)
    sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
    bh.buddy_hip_variant_reset()
    _, got = sess.prefill(toks, before, precision=precision)
    wide = (heads + 2 * kv_heads) * 128 >= 2048
    few = n <= 16 and inter % 16 == 0 and (wide or precision != "bf16")
    ran = {k for k, v in tiles_run(bh).items() if v and ("pair" in k and "batch" not in k or "rope" in k or "rows_kernel" in k)}
    if few and wide or n > 16:
        assert bool(ran) == (n > 16), ran
    rows = [sess.get_kv(j)[:, before:before + n] for j in (2, 3)]
    sess.close()
    sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
    for i, t in enumerate(toks):
        _, want = sess.decode(int(t), before + i, want_logits=i + 1 == n)
    pairs = [(got, want)] + [(rows[j - 2], sess.get_kv(j)[:, before:before + n]) for j in (2, 3)]
    sess.close()
    for g, w in pairs:
        if precision == "digits" or few and wide and before < 200:
            check_close(g, w)
        else:
            bound = 2.0**-10 if precision == "digits2" else 10 * 2.0**-9
            g, w = np.asarray(g, np.float64), np.asarray(w, np.float64)
            assert np.linalg.norm(g - w) < bound * np.linalg.norm(w)


# ... behind contexts whose attention leaves parts, fewer and more than are asked for at once: folded to f32 rows
@pytest.mark.parametrize("precision", ["digits", "digits2", "bf16"])
@pytest.mark.parametrize("heads,kv_heads,before,n", [(12, 2, 400, 8), (16, 2, 1500, 16), (12, 2, 3000, 2), (8, 4, 900, 5)])
def test_few_tokens_behind_long_contexts(heads, kv_heads, before, n, precision):
    shape = Shape(layers=2, hidden=384, heads=heads, kv_heads=kv_heads, head_dim=128, inter=336, vocab=320,
                  max_len=before + n + 8)
    toks = synthetic.first_tokens(shape, n, seed=n).astype(np.int32)
    sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
    _, got = sess.prefill(toks, before, precision=precision)
    sess.close()
    sess, _ = synthetic.build_session(shape, context=before, ln_jitter=0.1)
    for i, t in enumerate(toks):
        _, want = sess.decode(int(t), before + i, want_logits=i + 1 == n)
    sess.close()
    check_close(got, want)


# Where that ends: rows cast to bfloat16 in layers of 80, 128 and 250 million weights, and rows that are not
# read 16 bytes at a time
@pytest.mark.parametrize("precision,hidden,heads,kv_heads,inter,n,few", [
    ("bf16", 2048, 16, 2, 11008, 16, True), ("bf16", 2560, 20, 4, 9728, 12, True), ("bf16", 2560, 20, 4, 9728, 13, False),
    ("bf16", 4096, 32, 8, 11008, 8, True), ("bf16", 4096, 32, 8, 11008, 9, False), ("bf16", 4096, 32, 8, 11008, 4, True),
    ("bf16", 5120, 40, 8, 13824, 2, True), ("bf16", 5120, 40, 8, 13824, 3, False), ("bf16", 5120, 40, 8, 13824, 4, False),
    ("bf16", 5120, 40, 8, 13824, 5, True), ("digits", 5120, 40, 8, 13824, 16, True), ("bf16", 1534, 12, 2, 336, 4, True),
    ("digits2", 4096, 32, 8, 11008, 12, True), ("digits2", 4096, 32, 8, 11008, 13, False),
    ("bf16", 1534, 12, 2, 336, 5, False), ("digits2", 1534, 12, 2, 336, 8, True), ("digits", 1534, 12, 2, 336, 9, False)])
def test_which_prompts_have_few_tokens(bh, precision, hidden, heads, kv_heads, inter, n, few):
    shape = Shape(layers=1, hidden=hidden, heads=heads, kv_heads=kv_heads, head_dim=128, inter=inter, vocab=320,
                  max_len=n + 8)
    toks = synthetic.first_tokens(shape, n, seed=n).astype(np.int32)
    sess, _ = synthetic.build_session(shape, context=0, ln_jitter=0.1)
    bh.buddy_hip_variant_reset()
    _, got = sess.prefill(toks, 0, precision=precision)
    ran = {k for k, v in tiles_run(bh).items() if v and ("pair" in k and "batch" not in k or "rope" in k or "rows_kernel" in k)}
    assert bool(ran) != few, ran
    for i, t in enumerate(toks):
        _, want = sess.decode(int(t), i, want_logits=i + 1 == n)
    sess.close()
    if few or precision == "digits":
        check_close(got, want)
    else:
        bound = 2.0**-10 if precision == "digits2" else 10 * 2.0**-9
        got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
        assert np.linalg.norm(got - want) < bound * np.linalg.norm(want)


# The last launch of one query block to a workgroup of eight wavefronts, and the first of two
@pytest.mark.parametrize("H,HKV,Lq,Lk", [(16, 4, 256, 256), (16, 4, 257, 300), (128, 16, 32, 40), (128, 16, 33, 33)])
def test_prefill_attention_pairs_where_the_chip_is_full(bh, oracle, H, HKV, Lq, Lk):
    test_prefill_attention_launches_of_several_rounds(bh, oracle, H, HKV, Lq, Lk)
