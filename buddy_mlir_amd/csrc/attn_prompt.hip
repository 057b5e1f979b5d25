// attn_prompt.hip -- causal GQA attention of a session's prompt tokens over its KV cache.
//
// The same operation as attn_prefill.hip (flash_attention_for_cpu_prefill_op,
// frontend/Python/ops/tosa.py:4326-4810) with a workspace and on the bfloat16 matrix
// cores: an f32 value is the sum of three bfloat16 values of 8 bits each, rounded to
// nearest, which is every bit of it; of the nine products of two such sums the six of
// more than 2^-24 of the largest are taken, each exact, all summed in f32.  Six
// instructions at sixteen times the rate of the f32 matrix instructions.  The error
// against 64 bits is that of the f32 kernel (a 28-layer prompt of 1931 tokens: 3.6e-6
// with either).
//
// What bounds it: per tile of 256 rows x 32 keys a SIMD has 6144 cycles of matrix
// instructions and 3600 of vector instructions (softmax, conversions), which run one
// after the other as if they were one kind, and the chip draws so much power meanwhile
// that it clocks at 1.6 GHz: 6 us a tile.  (The two wavefronts of a SIMD in opposite
// phases, with the values a tile behind the scores: the same 6 us.)  What a launch costs
// beside its tiles is some 9 us: the share, queries and their terms, the first tile's way.
// 12 query heads, 2 KV heads, us per layer, this kernel and the fold behind it against
// attn_prefill.hip and the conversion behind that (attn_prompt_pays says which is taken):
//   2000 tokens 104 vs 156, 4096 tokens 332 vs 655, 150 behind 1900 36 vs 64,
//   27 behind 1900 27 vs 58, 512 tokens 28 vs 25, 256 tokens 21 vs 17
#include "attn.h"
#include "attn_fold.h"
#include "bf16_dev.h"

#include <algorithm>
#include <cmath>

namespace bh {
namespace {

constexpr int kThreads = 2 * kPromptRows; // a wavefront has 32 rows
constexpr int kKeys = 32;                 // of a tile
constexpr int kTerm = kKeys * kPromptD * 2; // bytes of one term of a tile's keys or values
constexpr int kHalf = 3 * kTerm;          // keys, then values
constexpr int kBuf = 2 * kHalf;
constexpr int kLds = 2 * kBuf + kThreads / 64 * 4096;
constexpr float kSeedM = -1.0e30f;        // tosa.py:4383
constexpr float kSlack = 8.0f;

struct PromptArgs {
  const float *q, *k, *v;
  float *out;
  int64_t q_stride, q_hstride, o_stride, o_hstride, kv_stride;
  int kv_heads, group, q_len, k_len, q_offset, nblk;
  int per_head;     // tiles of a KV head
  int share, extra; // tiles of a workgroup; the first `extra` ones take one more
  float scale;      // of the scores, times log2 e
  float *acc, *ml;
  PromptBlock *blocks;
};

// tiles of keys that block b of 256 rows sees
__device__ __forceinline__ int tiles_of(const PromptArgs &a, int b) {
  const int row = min((b + 1) * kPromptRows, a.q_len * a.group) - 1;
  return (min(a.k_len, a.q_offset + row / a.group + 1) + kKeys - 1) / kKeys;
}
__device__ __forceinline__ int wave_scan(int v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(v, o, 64);
    if (lane >= o)
      v += u;
  }
  return v;
}
// the block that tile t of a KV head belongs to (t becomes the tile within it), or
// nblk with t the number of tiles beyond the last block
__device__ __forceinline__ int find_block(const PromptArgs &a, int lane, int &t) {
  for (int base = 0; base < a.nblk; base += 64) {
    const int n = base + lane < a.nblk ? tiles_of(a, base + lane) : 0;
    const int incl = wave_scan(n, lane);
    const unsigned long long past = __ballot(incl > t);
    if (past) {
      const int l = __builtin_ctzll(past);
      t -= __builtin_amdgcn_readlane(incl - n, l);
      return base + l;
    }
    t -= __builtin_amdgcn_readlane(incl, 63);
  }
  return a.nblk;
}

__device__ __forceinline__ f32x16 mma(uint4 a, uint4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned round2(float x, float y) { // one instruction
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{x, y}), bf16x2));
}
// two values as three words of two bfloat16 terms; returns NaN where one is not finite
__device__ __forceinline__ float split2(float x, float y, unsigned &t0, unsigned &t1, unsigned &t2) {
  t0 = round2(x, y);
  x -= bf_lo(t0);
  y -= bf_hi(t0);
  t1 = round2(x, y);
  x -= bf_lo(t1);
  y -= bf_hi(t1);
  t2 = round2(x, y);
  return x + y;
}
__device__ __forceinline__ float split8(const float (&x)[8], uint4 (&t)[3]) {
  unsigned w[3][4];
  float bad = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    bad += split2(x[2 * i], x[2 * i + 1], w[0][i], w[1][i], w[2][i]);
#pragma unroll
  for (int p = 0; p < 3; ++p)
    t[p] = uint4{w[p][0], w[p][1], w[p][2], w[p][3]};
  return bad;
}
// the six products of more than 2^-24: (term of a, term of b), small ones first
constexpr int kProdA[6] = {0, 2, 1, 0, 1, 0};
constexpr int kProdB[6] = {2, 0, 1, 1, 0, 0};

// Workgroup i takes an equal share of all (KV head, row block, key tile) triples in that
// order, wherever it begins and ends: blocks it holds whole leave as finished rows, the
// others as partial results.  Its eight wavefronts have 32 rows each and share the tiles,
// of which each turns an eighth into terms a tile ahead.
//   S^T[key, row] = K . Q^T;  O^T[d, row] += V^T . P^T
// and the registers of S^T are the operand P^T as they lie: a lane has keys
// 8 j + 4 (lane / 32) + 0..3 of row lane % 32, and V^T is stored with its keys in that
// order.  LDS: [buffer][keys | values][term][step][lane][16 bytes], operands as they are
// read; the keys' slots are permuted within a step so that writing them by rows meets
// every bank once.
__global__ void __launch_bounds__(kThreads)
attn_prompt_kernel(const float *p_k, const float *p_v, int64_t p_kv_stride, int p_share, int p_extra,
                   int p_per_head, int p_nblk, int p_group, int p_q_len, int p_k_len, int p_q_offset,
                   PromptArgs rest) {
  // what comes before the first load arrives in SGPRs (-amdgpu-kernarg-preload-count)
  PromptArgs a = rest;
  a.k = p_k;
  a.v = p_v;
  a.kv_stride = p_kv_stride;
  a.share = p_share;
  a.extra = p_extra;
  a.per_head = p_per_head;
  a.nblk = p_nblk;
  a.group = p_group;
  a.q_len = p_q_len;
  a.k_len = p_k_len;
  a.q_offset = p_q_offset;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[]; // [2][kBuf], then 4 KiB per wavefront
  __shared__ unsigned bad_s[3];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, up = lane >> 5;

  // this workgroup's tiles [t, t1) of all
  const int self = blockIdx.x;
  auto begins = [&](int i) { return i * a.share + min(i, a.extra); };
  int t = begins(self);
  const int t0 = t, t1 = begins(self + 1);

  struct Place {
    int h, b, j, n; // KV head, row block, tile within it, tiles of the block
  };
  Place at;
  {
    at.h = t / a.per_head;
    int r = t - at.h * a.per_head;
    at.b = find_block(a, lane, r);
    at.j = r;
    at.n = tiles_of(a, at.b);
  }
  auto next_of = [&](Place p) {
    if (++p.j == p.n) {
      p.j = 0;
      if (++p.b == a.nblk) {
        p.b = 0;
        if (p.h + 1 < a.kv_heads)
          ++p.h;
      }
      p.n = tiles_of(a, p.b);
    }
    return p;
  };

  // ---- a tile on its way ------------------------------------------------------------
  // Each wavefront brings what it converts itself into 4 KiB of LDS of its own, a tile
  // ahead and past the registers (there are none left), by the four instructions below:
  // rows 4 wave .. + 3 of the keys, and of the values the eight keys and 64 channels whose
  // columns its lanes turn.  The compiler does not see these loads; bring_wait() waits for
  // them, and nothing else reads that memory.
  const int g8 = tid & 15, ch = tid & 127, vks = wave >> 2, vhalf = (wave >> 1) & 1;
  unsigned char *raw = lds + 2 * kBuf + wave * 4096;
  auto bring = [&](const Place &p) {
    const float *k = a.k + (int64_t)p.h * a.kv_stride * kPromptD, *v = a.v + (int64_t)p.h * a.kv_stride * kPromptD;
    const int k0 = p.j * kKeys;
    const unsigned to = (unsigned)__builtin_amdgcn_readfirstlane(
        (int)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)raw);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float *src;
      if (i < 2) {
        const int key = min(k0 + 4 * wave + 2 * i + up, a.k_len - 1);
        src = k + (int64_t)key * kPromptD + col * 4;
      } else { // row e of the eight: 16 vks + 8 (e / 4) + 4 vhalf + e % 4
        const int key = min(k0 + 16 * vks + 8 * (i - 2) + 4 * vhalf + (lane >> 4), a.k_len - 1);
        src = v + (int64_t)key * kPromptD + (wave & 1) * 64 + (lane & 15) * 4;
      }
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(to + i * 1024)
                   : "memory", "m0");
    }
  };
  auto bring_wait = []() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  auto put_keys = [&](unsigned char *buf) {
    const float4 x0 = *reinterpret_cast<const float4 *>(raw + (lane >> 4) * 512 + g8 * 32);
    const float4 x1 = *reinterpret_cast<const float4 *>(raw + (lane >> 4) * 512 + g8 * 32 + 16);
    const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    uint4 term[3];
    split8(x, term);
    const int key = tid >> 4;
#pragma unroll
    for (int p = 0; p < 3; ++p)
      *reinterpret_cast<uint4 *>(buf + ((p * 8 + (g8 >> 1)) * 64 + (g8 & 1) * 32 + (key ^ g8)) * 16) = term[p];
  };
  auto put_values = [&](const float (&x)[8], unsigned char *buf) {
    uint4 term[3];
    const float rest = split8(x, term);
#pragma unroll
    for (int p = 0; p < 3; ++p)
      *reinterpret_cast<uint4 *>(buf + (((p * 4 + (ch >> 5)) * 2 + vks) * 64 + vhalf * 32 + (ch & 31)) * 16) =
          term[p];
    return rest;
  };
  auto put_values_checked = [&](unsigned char *buf, unsigned *bad) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      x[e] = *reinterpret_cast<const float *>(raw + 2048 + e * 256 + lane * 4);
    const float rest = put_values(x, buf);
    if (rest != rest) {
      // A value that has no terms must not reach rows that do not see its key, whose
      // weight there is zero: it goes in as zero, and its key makes NaN of the rows that
      // do see it (see add_values), which the fold then computes again.
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (!(fabsf(x[e]) < 3.3895e38f)) {
          x[e] = 0.f;
          atomicOr(bad, 1u << (16 * vks + 8 * (e >> 2) + 4 * vhalf + (e & 3)));
        }
      put_values(x, buf);
    }
  };

  uint4 qf[8][3];
  f32x16 o[4];
  float m = kSeedM, l = 0.f; // l: this lane's share
  int qpos = 0, pos_first = 0, pos_last = 0; // of this lane's row; of the wavefront's rows
  auto begin_block = [&](const Place &p) {
    const int row = min(p.b * kPromptRows + wave * 32 + col, a.q_len * a.group - 1);
    const int tok = row / a.group, hh = row - tok * a.group;
    qpos = a.q_offset + tok;
    pos_first = __builtin_amdgcn_readfirstlane(qpos);
    pos_last = __builtin_amdgcn_readlane(qpos, 31);
    const float *src = a.q + (int64_t)tok * a.q_stride + (int64_t)(p.h * a.group + hh) * a.q_hstride + up * 8;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const float4 x0 = *reinterpret_cast<const float4 *>(src + s * 16);
      const float4 x1 = *reinterpret_cast<const float4 *>(src + s * 16 + 4);
      const float y[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
      split8(y, qf[s]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = f32x16{};
    m = kSeedM;
    l = 0.f;
  };

  float w[16];    // scores of this lane's row, then their weights
  uint4 pf[2][3]; // the weights as terms
  auto scores = [&](const unsigned char *buf) {
    f32x16 s0{}, s1{};
    // the slot of this lane's key in step s is (col ^ up) ^ 2 s: worked out at each tile,
    // not kept in registers that there are not
    int at_key = up * 512 + (col ^ up) * 16;
    asm volatile("" : "+v"(at_key));
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      uint4 kf[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
        kf[p] = *reinterpret_cast<const uint4 *>(buf + (at_key ^ (32 * s)) + (p * 8 + s) * 1024);
#pragma unroll
      for (int c = 0; c < 6; c += 2) { // two chains: an instruction waits for the sum it adds to
        s0 = mma(kf[kProdA[c]], qf[s][kProdB[c]], s0);
        s1 = mma(kf[kProdA[c + 1]], qf[s][kProdB[c + 1]], s1);
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
      w[i] = s0[i] + s1[i];
  };
  auto weights = [&](int k0) {
    if (k0 + kKeys - 1 > pos_first) { // some of the tile's keys are behind some row
#pragma unroll
      for (int i = 0; i < 16; ++i)
        w[i] = k0 + 8 * (i >> 2) + 4 * up + (i & 3) <= qpos ? w[i] : -INFINITY;
    }
    float mt = w[0];
#pragma unroll
    for (int i = 1; i < 16; ++i)
      mt = fmaxf(mt, w[i]);
    float x, y;
    lane_pair<32>(mt, x, y);
    mt = fmaxf(x, y) * a.scale;
    // the maximum moves, and the sums are rescaled, only when a score exceeds it by more
    // than kSlack: the weights stay below 2^kSlack
    if (__any(mt > m + kSlack)) {
      mt = fmaxf(mt, m);
      const float alpha = __builtin_amdgcn_exp2f(m - mt);
      m = mt;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        o[i] *= alpha;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      w[i] = __builtin_amdgcn_exp2f(fmaf(w[i], a.scale, -m)); // one rounding before the exponential
      l += w[i];
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const float p8[8] = {w[8 * ks], w[8 * ks + 1], w[8 * ks + 2], w[8 * ks + 3],
                           w[8 * ks + 4], w[8 * ks + 5], w[8 * ks + 6], w[8 * ks + 7]};
      split8(p8, pf[ks]);
    }
  };
  auto add_values = [&](const unsigned char *buf, int k0, unsigned bad) {
    if (bad) { // keys up to this row's own position
      const int last = qpos - k0;
      if (last >= 0 && (bad & (last >= 31 ? ~0u : (2u << last) - 1u)))
        l = __uint_as_float(0x7fc00000u);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) { // 16 keys, two of the four blocks of 32 channels
      uint4 vf[3][2];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          vf[p][e] = *reinterpret_cast<const uint4 *>(
              buf + (((p * 4 + 2 * (i & 1) + e) * 2 + (i >> 1)) * 64 + lane) * 16);
#pragma unroll
      for (int c = 0; c < 6; ++c)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          o[2 * (i & 1) + e] = mma(vf[kProdA[c]][e], pf[i >> 1][kProdB[c]], o[2 * (i & 1) + e]);
    }
  };

  auto end_block = [&](const Place &p, int first_tile, bool from_start, bool whole) {
    float x, y;
    lane_pair<32>(l, x, y);
    const float sum = x + y;
    const int r = wave * 32 + col, row = p.b * kPromptRows + r;
    float *dst;
    float f = 1.0f;
    if (whole) {
      const int tok = row / a.group, hh = row - tok * a.group;
      dst = a.out + (int64_t)tok * a.o_stride + (int64_t)(p.h * a.group + hh) * a.o_hstride;
      f = 1.0f / sum;
    } else {
      // the first part of this workgroup's share in slot 2 i, one behind it in 2 i + 1
      const size_t slot = 2 * (size_t)self + (first_tile > t0 ? 1 : 0);
      dst = a.acc + (slot * kPromptRows + r) * kPromptD;
      if (up == 0) {
        a.ml[(slot * kPromptRows + r) * 2] = m;
        a.ml[(slot * kPromptRows + r) * 2 + 1] = sum;
      }
    }
    if (row < a.q_len * a.group) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          *reinterpret_cast<float4 *>(dst + dt * 32 + 8 * j + 4 * up) =
              float4{o[dt][4 * j] * f, o[dt][4 * j + 1] * f, o[dt][4 * j + 2] * f, o[dt][4 * j + 3] * f};
    }
    if (tid == 0 && from_start) {
      // whoever has the block's first tile says where its parts are
      PromptBlock d{0, 0, 0, 0};
      if (!whole) {
        const int last = first_tile + p.n - 1, longer = a.extra * (a.share + 1);
        const int i = last < longer ? last / (a.share + 1) : a.extra + (last - longer) / a.share;
        d.first = 2 * self + (first_tile > t0 ? 1 : 0);
        d.owner = self;
        d.parts = i - self + 1;
      }
      a.blocks[p.h * a.nblk + p.b] = d;
    }
  };

  if (tid < 3)
    bad_s[tid] = 0;
  bring(at);
  __syncthreads();
  Place nx = next_of(at);
  begin_block(at);
  bring_wait();
  put_keys(lds);
  put_values_checked(lds + kHalf, &bad_s[0]);
  if (t + 1 < t1)
    bring(nx);
  int seg0 = t; // first tile of the block's part held here
  bool from_start = at.j == 0;
  int cur = 0, bad_at = 0; // (t - t0) & 1 and (t - t0) % 3
  for (;;) {
    __syncthreads();
    const int bad_next = bad_at == 2 ? 0 : bad_at + 1, bad_after = bad_next == 2 ? 0 : bad_next + 1;
    const unsigned bad = __builtin_amdgcn_readfirstlane(bad_s[bad_at]);
    if (tid == 0)
      bad_s[bad_after] = 0;
    const bool more = t + 1 < t1;
    const Place nn = next_of(nx);
    unsigned char *buf = lds + cur * kBuf, *other = lds + (cur ^ 1) * kBuf;
    auto stage = [&]() {
      if (!more)
        return;
      bring_wait();
      put_keys(other);
      put_values_checked(other + kHalf, &bad_s[bad_next]);
      if (t + 2 < t1)
        bring(nn);
    };
    // the two wavefronts of a SIMD in opposite order: one's conversion beside the other's
    // products
    if (wave < 4)
      stage();
    if (at.j * kKeys <= pos_last) {
      scores(buf);
      weights(at.j * kKeys);
      add_values(buf + kHalf, at.j * kKeys, bad);
    }
    if (wave >= 4)
      stage();
    const bool ends = at.j + 1 == at.n;
    if (ends || !more)
      end_block(at, seg0, from_start, ends && from_start);
    if (!more)
      break;
    ++t;
    if (ends) {
      begin_block(nx);
      seg0 = t;
      from_start = true;
    }
    at = nx;
    nx = nn;
    cur ^= 1;
    bad_at = bad_next;
  }
}

} // namespace

// The (KV head, row block, key tile) triples of a launch and who takes them.
namespace {
BH_TILE_FAMILY(PromptFamily, "attn_prompt_kernel");
struct PromptShare {
  int64_t rows, tiles; // rows of a KV head; tiles of all
  int nblk, workgroups;
};
PromptShare share_out(int q_len, int q_offset, int heads, int kv_heads) {
  PromptShare s;
  const int group = heads / kv_heads;
  s.rows = (int64_t)q_len * group;
  s.nblk = (int)ceil_div(s.rows, kPromptRows);
  s.tiles = 0;
  for (int b = 0; b < s.nblk; ++b) {
    const int64_t last = std::min((int64_t)(b + 1) * kPromptRows, s.rows) - 1;
    s.tiles += ceil_div(q_offset + last / group + 1, kKeys);
  }
  s.tiles *= kv_heads;
  s.workgroups = (int)std::min<int64_t>(kPromptWorkgroups, s.tiles); // each at least a tile
  return s;
}
} // namespace

// An estimate of both ways in microseconds, fitted to 1748 prompts of 12 layers: eight shapes of 1 to
// 64 heads, 4 to 1000 tokens behind 0 to 1200, in three modes.  `converts`: behind the other way the
// rows take a launch of their own to become the output product's input, which the fold is here
// (not up to 16 tokens as f32, nor up to 128 as digits, which that product makes itself).
// The choice is up to 13 % of a layer slower than the better way and 0.25 % on average.  us a
// layer with its products, the other way and this one, where the line lies:
//   12 heads, 2 KV heads, digits: 4 behind 400 40.9, 42.3, behind 700 47.0, 43.9, 32 behind 256
//     53.3, 54.9, behind 700 60.7, 58.0, 256 behind 400 70.1, 70.1, 500 alone 74.9, 75.6, behind
//     128 79.5, 86.7, behind 400 93.0, 90.3, 730 alone 99.8, 102.0, 920 115.9, 113.7
//   64 and 8, digits: 32 behind 256 63.6, 77.2, 128 behind 700 107.7, 107.0, 256 behind 128 111,
//     115, behind 256 123, 118, 500 alone 165, 160
//   one head, every bit: 64 behind 64 54.7, 56.5, behind 128 57.4, 56.8, 256 behind 64 65.6, 64.6
// More than 32 tokens behind 400 and more go this way in doubt, up to 6 us, and more than 640 up to
// 2.5: it asks for each key once for all heads of a KV head, and what is not finite stays with the
// rows that see it.
bool attn_prompt_pays(int q_len, int q_offset, int heads, int kv_heads, bool converts) {
  const double kilo_rows = 1e-4 * q_len * heads; // tens of thousands of (token, head)
  // attn_prefill.hip: blocks of 16 queries, one to a workgroup of eight wavefronts, then two, while
  // those fit the chip; steps of 16 keys per wavefront
  const int64_t nqb = ceil_div(q_len, 16);
  double steps;
  if (nqb == 1 || heads * nqb <= 256)
    steps = 2.7 * (double)ceil_div(q_offset + q_len, 16) / 8;
  else if (heads * ceil_div(nqb, 2) <= 256)
    steps = 1.5 + 2.4 * (2.0 * q_offset + q_len + 16) / 128;
  else
    steps = 0.3 + 2.7 * (1.0 * heads * q_len * q_len / (16 * 32 * 256) +
                         (double)ceil_div(heads * nqb, 256) * q_offset / 16) / 8;
  const double other = 4.7 + (converts ? 3.9 : 0.0) + steps + 2.5 * kilo_rows;
  // here: tiles of the longest share, wavefronts that have rows, blocks that begin and end, and
  // the fold's trips to memory and its bytes
  const PromptShare s = share_out(q_len, q_offset, heads, kv_heads);
  const double share = (double)s.tiles / s.workgroups;
  const double parts = (double)ceil_div(q_offset + q_len, kKeys) / share;
  const int64_t waves = std::min<int64_t>(8, ceil_div(s.rows, 32));
  const double trips = parts <= 4 ? 1 : parts <= 8 ? 2 : 2 * std::ceil(parts / 16);
  const double here = 10.6 + 5.1 * (double)(ceil_div(s.tiles, s.workgroups) - 1) +
                      0.8 * (double)std::max<int64_t>(0, waves - 4) + 4.3 * s.workgroups / 256 +
                      0.85 * s.nblk * kv_heads / s.workgroups +
                      0.9 * (double)ceil_div(heads, 16) * trips +
                      0.46 * kilo_rows * std::min(parts, 20.0);
  return here < other + (q_len > 32 && q_offset >= 400 ? 6.0 : q_len > 640 ? 2.5 : 0.0);
}

// Two slots for every workgroup there can be: 67 MB where all compute units have tiles.
size_t attn_prompt_workspace_bytes(int q_len, int k_len, int heads, int kv_heads) {
  const int64_t blocks = (int64_t)kv_heads * ceil_div((int64_t)q_len * (heads / kv_heads), kPromptRows);
  const size_t slots = 2 * (size_t)std::min<int64_t>(kPromptWorkgroups, blocks * ceil_div(k_len, kKeys));
  return slots * kPromptRows * (kPromptD + 2) * sizeof(float) + (size_t)blocks * sizeof(PromptBlock);
}

int launch_attn_prompt(const AttnPrefillArgs &in, void *workspace, PromptFold &fold, hipStream_t stream) {
  BH_REQUIRE(in.q && in.k && in.v && in.out && workspace && !in.mask, "attn_prompt: null pointer or mask");
  BH_REQUIRE(in.head_dim == kPromptD && in.kv_heads > 0 && in.heads % in.kv_heads == 0 && in.q_len > 0 &&
                 in.k_len >= in.q_len && in.kv_stride >= in.k_len,
             "attn_prompt: heads=%d kv_heads=%d q_len=%d k_len=%d", in.heads, in.kv_heads, in.q_len,
             in.k_len);
  BH_REQUIRE(in.q_stride % 4 == 0 && in.q_hstride % 4 == 0 && in.o_stride % 4 == 0 &&
                 in.o_hstride == kPromptD &&
                 ((reinterpret_cast<uintptr_t>(in.q) | reinterpret_cast<uintptr_t>(in.k) |
                   reinterpret_cast<uintptr_t>(in.v) | reinterpret_cast<uintptr_t>(in.out) |
                   reinterpret_cast<uintptr_t>(workspace)) & 15) == 0,
             "attn_prompt: strides and pointers must keep 16-byte alignment");
  PromptArgs a;
  a.q = in.q;
  a.k = in.k;
  a.v = in.v;
  a.out = in.out;
  a.q_stride = in.q_stride;
  a.q_hstride = in.q_hstride;
  a.o_stride = in.o_stride;
  a.o_hstride = in.o_hstride;
  a.kv_stride = in.kv_stride;
  a.kv_heads = in.kv_heads;
  a.group = in.heads / in.kv_heads;
  a.q_len = in.q_len;
  a.k_len = in.k_len;
  a.q_offset = in.k_len - in.q_len;
  a.scale = (float)(in.scale * 1.4426950408889634);
  BH_REQUIRE((int64_t)in.q_len * a.group < (1 << 30), "attn_prompt: q_len %d too long", in.q_len);
  const PromptShare share = share_out(in.q_len, a.q_offset, in.heads, in.kv_heads);
  BH_REQUIRE(share.tiles < (1u << 30), "attn_prompt: %lld tiles of keys", (long long)share.tiles);
  a.nblk = share.nblk;
  a.acc = static_cast<float *>(workspace);
  const size_t slots = 2 * (size_t)share.workgroups;
  a.ml = a.acc + slots * kPromptRows * kPromptD;
  a.blocks = reinterpret_cast<PromptBlock *>(a.ml + slots * kPromptRows * 2);
  a.per_head = (int)(share.tiles / in.kv_heads);
  a.share = (int)(share.tiles / share.workgroups);
  a.extra = (int)(share.tiles % share.workgroups);
  BH_NOTE_VARIANT(PromptFamily, kPromptRows);
  static DynLdsOnce dyn_lds;
  BH_CHECK_HIP(ensure_dyn_lds(dyn_lds, reinterpret_cast<const void *>(attn_prompt_kernel), kLds));
  hipLaunchKernelGGL(attn_prompt_kernel, dim3((unsigned)share.workgroups), dim3(kThreads), kLds, stream, a.k, a.v,
                     a.kv_stride, a.share, a.extra, a.per_head, a.nblk, a.group, a.q_len, a.k_len, a.q_offset, a);
  BH_CHECK_HIP(hipGetLastError());
  fold.out = in.out;
  fold.acc = a.acc;
  fold.ml = a.ml;
  fold.blocks = a.blocks;
  fold.group = a.group;
  fold.nblk = a.nblk;
  fold.q = a.q;
  fold.k = a.k;
  fold.v = a.v;
  fold.q_stride = a.q_stride;
  fold.q_hstride = a.q_hstride;
  fold.kv_stride = a.kv_stride;
  fold.q_offset = a.q_offset;
  fold.scale = a.scale;
  return BUDDY_HIP_OK;
}

} // namespace bh
