// attn_terms.hip -- causal GQA attention of a session's prompt ahead of which there is nothing, over keys and
// values that lie as float16 terms (attn_terms.h), which the kernels that rotate q | k | v left beside the cache.
//
// The same operation as attn_prompt.hip (flash_attention_for_cpu_prefill_op,
// frontend/Python/ops/tosa.py:4326-4810) for prompts too short to share their tiles out: a workgroup takes 32
// rows of a KV head (row r is query r / group, head r % group of the group) and every key that they see, its eight
// wavefronts every eighth tile of 32 keys each, straight from memory as operands; they meet in LDS and leave
// finished rows.
//
// What bounds it: a launch, a trip to memory for the queries and first keys, one or two tiles to a wavefront (some
// 1500 cycles of matrix and 900 of vector instructions each, two wavefronts to a SIMD), and the meeting.  12 query
// heads, 2 KV heads, us against attn_prefill.hip's f32 instructions on rows as they lie: 27 tokens 6.7 and 7.6, 512
// 12.6 and 23.3; the rotation's launch, which writes the terms, 5.6 and 5.4, 6.1 and 5.3.
// Error against 64 bits (normal values): 27 tokens 1.5e-7 and 1.1e-7, 300 1.9e-7 and 1.6e-7, 1931 2.2e-7 and 2.3e-7;
// scores four times as large 2.3e-7 and 2.2e-7, 3.7e-7 and 3.6e-7, 5.3e-7 and 5.2e-7; a channel in 40 eight times as
// large 3.3e-7 and 4.0e-7, 6.5e-7 and 7.1e-7, 9.7e-7 and 1.1e-6.
#include "attn.h"
#include "attn_terms.h"

namespace bh {
namespace {

constexpr int kThreads = 512, kRows = 32, kWaves = kThreads / 64;
constexpr int kOutRow = kPromptD + 4;                // floats of a row in LDS
constexpr int kQueries = 2 * 8 * 1024;               // [term][step][lane][16 bytes]
constexpr int kLds = kQueries + kWaves * kRows * (kOutRow + 2) * 4;
// keys of which the scales fit where the sums go
constexpr int kMostKeys = (kLds - kQueries) / (int)sizeof(TileScales) * kTileKeys;
static_assert(kMostKeys >= kTermsMostKeys, "scales of the longest prompt");

struct TermsArgs {
  PromptFold f; // the operands, for rows that are to be computed again
  float *out;
  int64_t o_stride, o_hstride;
  int q_len, row_blocks;
};

__global__ void __launch_bounds__(kThreads)
attn_terms_kernel(const unsigned char *tiles, const float *q, int64_t q_stride, int64_t q_hstride, int per_head,
                  int group, int q_len, int row_blocks, float scale, TermsArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[]; // queries; scales, then sums and their weights
  __shared__ float scale_s[kRows];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, up = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // long ones first
  const int kvh = blockIdx.y, row0 = (row_blocks - 1 - (int)blockIdx.x) * kRows, last = q_len * group - 1;
  auto token_of = [&](int r) { return min(row0 + r, last) / group; };
  const int ntiles = token_of(kRows - 1) / kTileKeys + 1;

  // queries: sixteen threads to a row; this wavefront's first keys behind them
  const int qr = tid >> 4, g8 = tid & 15;
  const int qrow = min(row0 + qr, last), qtok = qrow / group;
  const float *src = q + (int64_t)qtok * q_stride + (int64_t)(kvh * group + qrow - qtok * group) * q_hstride + g8 * 8;
  const float4 x0 = *reinterpret_cast<const float4 *>(src), x1 = *reinterpret_cast<const float4 *>(src + 4);
  const unsigned char *head = tiles + (size_t)kvh * per_head * kTermTile;
  const unsigned at = lane * 16;
  // a scalar base: 64-bit addresses of every lane would take registers there are not
  auto operand = [&](const unsigned char *p) {
    const uintptr_t u = reinterpret_cast<uintptr_t>(p);
    const uintptr_t base = (uintptr_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)u) |
                           (uintptr_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(u >> 32)) << 32;
    const auto *from = (const __attribute__((address_space(1))) char *)base + at;
    return *(const __attribute__((address_space(1))) u32x4 *)from;
  };
  u32x4 kf[8][2];
  auto ask_keys = [&](int t, int half) {
    const unsigned char *p = head + (size_t)t * kTermTile;
#pragma unroll
    for (int s = 4 * half; s < 4 * half + 4; ++s)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        kf[s][c] = operand(p + c * kTermBytes + s * 1024);
  };
  ask_keys(min(wave, ntiles - 1), 0);
  ask_keys(min(wave, ntiles - 1), 1);
  // all tiles' scales, where the sums go at the end
  TileScales *scales = reinterpret_cast<TileScales *>(lds + kQueries);
  constexpr int kQuads = sizeof(TileScales) / 16;
  for (int i = tid; i < ntiles * kQuads; i += kThreads)
    reinterpret_cast<float4 *>(scales)[i] = *reinterpret_cast<const float4 *>(
        head + (size_t)(i / kQuads) * kTermTile + 4 * kTermBytes + i % kQuads * 16);
  {
    float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w}, undo;
    const unsigned e = key_scale(x, undo);
    if (g8 == 0)
      scale_s[qr] = undo * scale;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      x[i] *= pow2(e);
    uint4 term[2];
    split8(x, term);
#pragma unroll
    for (int p = 0; p < 2; ++p) // slots permuted by the step: writing by rows meets every bank
      *reinterpret_cast<uint4 *>(lds + ((p * 8 + (g8 >> 1)) * 64 + (g8 & 1) * 32 + (qr ^ g8)) * 16) = term[p];
  }
  __syncthreads();

  RowState r;
  r.m = kSeedM;
  r.l = 0.f;
  r.q_scale = scale_s[col];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    r.o[i] = f32x16{};
  const int qpos = token_of(col), pos_first = __builtin_amdgcn_readfirstlane(qpos);
  for (int t = wave; t < ntiles; t += kWaves) {
    const unsigned char *tile = head + (size_t)t * kTermTile;
    f32x16 s0{}, s1{}; // the small products by themselves
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      uint4 qf[2];
#pragma unroll
      for (int p = 0; p < 2; ++p)
        qf[p] = *reinterpret_cast<const uint4 *>(lds + (p * 8 + s) * 1024 + up * 512 + (col ^ (2 * s + up)) * 16);
      s1 = mma_f16(__builtin_bit_cast(uint4, kf[s][0]), qf[1], s1);
      s0 = mma_f16(__builtin_bit_cast(uint4, kf[s][0]), qf[0], s0);
      s1 = mma_f16(__builtin_bit_cast(uint4, kf[s][1]), qf[0], s1);
    }
    // values are asked for ahead of the weights
    u32x4 vf[2][2][4]; // [term][step][32 channels]
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int b = 0; b < 4; ++b)
          vf[c][s][b] = operand(tile + (2 + c) * kTermBytes + (b * 2 + s) * 1024);
    __builtin_amdgcn_sched_barrier(0);
    float w[16];
#pragma unroll
    for (int i = 0; i < 16; ++i)
      w[i] = s0[i] + s1[i];
    const int k0 = t * kTileKeys;
    uint4 pf[2][2];
    tile_weights(w, scales[t], up, k0 + kTileKeys - 1 > pos_first, qpos - k0, r, pf);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int c = 0; c < 3; ++c) // small ones first
#pragma unroll
        for (int b = 0; b < 4; ++b)
          r.o[b] = mma_f16(__builtin_bit_cast(uint4, vf[c == 0][s][b]), pf[s][c == 1], r.o[b]);
      __builtin_amdgcn_sched_barrier(0);
      ask_keys(min(t + kWaves, ntiles - 1), s); // into registers that those values leave
    }
  }

  // the wavefronts meet
  __syncthreads();
  const int waves = min(ntiles, kWaves);
  float *sums = reinterpret_cast<float *>(lds + kQueries), *ml = sums + kWaves * kRows * kOutRow;
  if (wave < waves) {
    float x, y;
    lane_pair<32>(r.l, x, y);
    float *dst = sums + (wave * kRows + col) * kOutRow + 4 * up;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<float4 *>(dst + b * 32 + 8 * j) =
            float4{r.o[b][4 * j], r.o[b][4 * j + 1], r.o[b][4 * j + 2], r.o[b][4 * j + 3]};
    if (up == 0)
      *reinterpret_cast<float2 *>(ml + (wave * kRows + col) * 2) = make_float2(r.m, x + y);
  }
  __syncthreads();
#pragma unroll 1
  for (int i = 0; i < kRows / 16; ++i) {
    const int rr = i * 16 + (tid >> 5), d = (tid & 31) * 4, row = row0 + rr;
    float m = kSeedM, l = 0.f, v[4] = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < waves; ++w)
      m = fmaxf(m, ml[(w * kRows + rr) * 2]);
    for (int w = 0; w < waves; ++w) {
      const float2 p = *reinterpret_cast<const float2 *>(ml + (w * kRows + rr) * 2);
      const float4 x = *reinterpret_cast<const float4 *>(sums + (w * kRows + rr) * kOutRow + d);
      const float f = __builtin_amdgcn_exp2f(p.x - m);
      l = fmaf(p.y, f, l);
      v[0] = fmaf(x.x, f, v[0]);
      v[1] = fmaf(x.y, f, v[1]);
      v[2] = fmaf(x.z, f, v[2]);
      v[3] = fmaf(x.w, f, v[3]);
    }
    if (row > last) // of half a wavefront together
      continue;
    const float inv = inverse_of(l);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] *= inv;
    const int tok = row / group, h = kvh * group + row - tok * group;
    repair4(a.f, tok, h, d, v);
    *reinterpret_cast<float4 *>(a.out + (int64_t)tok * a.o_stride + (int64_t)h * a.o_hstride + d) =
        make_float4(v[0], v[1], v[2], v[3]);
  }
}

} // namespace

BH_TILE_FAMILY(TermsFamily, "attn_terms_kernel");

int launch_attn_terms(const AttnPrefillArgs &in, const PromptTerms &terms, hipStream_t stream) {
  BH_REQUIRE(in.q && in.k && in.v && in.out && terms.tiles && !in.mask, "attn_terms: null pointer or mask");
  BH_REQUIRE(in.head_dim == kPromptD && in.kv_heads > 0 && in.kv_heads <= 65535 && in.heads % in.kv_heads == 0 &&
                 in.q_len > 0 && in.k_len == in.q_len && in.kv_stride >= in.k_len &&
                 in.k_len <= kTermsMostKeys && ceil_div(in.k_len, kTileKeys) <= terms.per_head,
             "attn_terms: heads=%d kv_heads=%d q_len=%d k_len=%d", in.heads, in.kv_heads, in.q_len, in.k_len);
  BH_REQUIRE(in.q_stride % 4 == 0 && in.q_hstride % 4 == 0 && in.o_stride % 4 == 0 && in.o_hstride % 4 == 0 &&
                 ((reinterpret_cast<uintptr_t>(in.q) | reinterpret_cast<uintptr_t>(in.k) |
                   reinterpret_cast<uintptr_t>(in.v) | reinterpret_cast<uintptr_t>(in.out) |
                   reinterpret_cast<uintptr_t>(terms.tiles)) & 15) == 0,
             "attn_terms: strides and pointers must keep 16-byte alignment");
  const int group = in.heads / in.kv_heads;
  BH_REQUIRE((int64_t)in.q_len * group < (1 << 30), "attn_terms: q_len %d too long", in.q_len);
  TermsArgs a;
  a.f.group = group;
  a.f.q = in.q;
  a.f.k = in.k;
  a.f.v = in.v;
  a.f.q_stride = in.q_stride;
  a.f.q_hstride = in.q_hstride;
  a.f.kv_stride = in.kv_stride;
  a.f.scale = (float)(in.scale * 1.4426950408889634);
  a.out = in.out;
  a.o_stride = in.o_stride;
  a.o_hstride = in.o_hstride;
  a.q_len = in.q_len;
  a.row_blocks = (int)ceil_div((int64_t)in.q_len * group, kRows);
  BH_NOTE_VARIANT(TermsFamily, kRows);
  static DynLdsOnce dyn_lds;
  BH_CHECK_HIP(ensure_dyn_lds(dyn_lds, reinterpret_cast<const void *>(attn_terms_kernel), kLds));
  hipLaunchKernelGGL(attn_terms_kernel, dim3((unsigned)a.row_blocks, (unsigned)in.kv_heads), dim3(kThreads), kLds,
                     stream, terms.tiles, in.q, in.q_stride, in.q_hstride, terms.per_head, group, in.q_len,
                     a.row_blocks, a.f.scale, a);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

} // namespace bh
