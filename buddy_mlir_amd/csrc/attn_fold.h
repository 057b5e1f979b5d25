// attn_fold.h -- partial results of a prompt's attention and their sum.
//
// The attention of a block of prompt tokens (attn_prompt.hip) takes the query heads of a
// KV head together: row r of a KV head is query r / group, head r % group of its group,
// and 256 consecutive rows are a block.  A block whose keys went to several workgroups
// leaves one partial result per workgroup in slots of a workspace.
#pragma once

#include "common.h"

#include <type_traits>

namespace bh {

constexpr int kPromptRows = 256;       // rows of a block
constexpr int kPromptD = 128;          // head size
constexpr int kPromptWorkgroups = 256; // at most, each with up to two partial results

// Where the parts of a block lie: part 0 in slot `first`, part j > 0 in slot
// 2 * (owner + j).  parts == 0: the finished rows are in the output already.
struct PromptBlock {
  int first, owner, parts, pad;
};
struct PromptFold {
  const float *out = nullptr;   // [tokens, heads, 128], finished rows of whole blocks
  const float *acc = nullptr;   // [slots][256 rows][128], sums of weight * value
  const float *ml = nullptr;    // [slots][256 rows][2]: max (of the scores times log2 e), sum of the weights
  const PromptBlock *blocks = nullptr; // [kv_heads][blocks]
  int group = 0, nblk = 0;
  // the operands, for rows that are to be computed again (f32_row)
  const float *q = nullptr, *k = nullptr, *v = nullptr;
  int64_t q_stride = 0, q_hstride = 0, kv_stride = 0;
  int q_offset = 0;
  float scale = 0.f; // of the scores, times log2 e
};

// Whether launch_attn_prompt and the fold behind it are to be taken for a session's prompt, or
// attn_prefill.hip and, if it `converts` its rows for the output product, the launch that does; or, of a prompt
// alone `on_terms`, attn_terms.hip.
bool attn_prompt_pays(int q_len, int q_offset, int heads, int kv_heads, bool converts, bool on_terms);

// Attention of a session's prompt tokens (no mask), on a workspace of
// attn_prompt_workspace_bytes for at least as many tokens and positions; what it leaves is
// described by `fold`.  `terms`: of a prompt alone, or none.
struct AttnPrefillArgs;
struct PromptTerms;
size_t attn_prompt_workspace_bytes(int q_len, int k_len, int heads, int kv_heads);
int launch_attn_prompt(const AttnPrefillArgs &a, const PromptTerms &terms, void *workspace, PromptFold &fold,
                       hipStream_t stream);
// the finished rows in `out`, [tokens, heads * 128], which may be fold.out ...
int launch_attn_fold_rows(const PromptFold &fold, int64_t o_stride, int heads, int tokens, float *out,
                          hipStream_t stream);
// ... as the bf16 terms of the matmul behind the attention (gemm_w8_mfma.hip) ...
int launch_attn_fold_to_terms(const PromptFold &fold, int64_t o_stride, int heads, int tokens, int terms,
                              unsigned short *staged, hipStream_t stream);
// ... or as its digit planes (gemm_w8_i8.hip)
int launch_attn_fold_to_digits(const PromptFold &fold, int64_t o_stride, int heads, int tokens, int digits,
                               void *staged, hipStream_t stream);

#if defined(__HIPCC__)
// The row of query head h at token t once more, in f32 sums, key after key: 32 lanes that
// hold four values each from d on.  A row comes to this when its sum of weights is NaN:
// because it is to be, or because the float16 terms of an operand do not exist (an
// infinity) or leave none to the row's other values (one far above them), a row of values is far from
// ordinary magnitudes (attn_terms.h), or a score's terms leave the range that the score itself is in.  An infinite
// score of -inf has no weight, and an infinite value makes its own channel infinite, as in the other attention
// kernels.  (1900 keys: some 0.4 ms.)
__device__ __forceinline__ void f32_row(const PromptFold &f, int t, int h, int d, float (&v)[4]) {
#pragma clang fp contract(off) // a score is rounded before the maximum is taken from it
  const int64_t head = (int64_t)(h / f.group) * f.kv_stride * kPromptD;
  const float *kp = f.k + head + d, *vp = f.v + head + d;
  const float4 q = *reinterpret_cast<const float4 *>(f.q + (int64_t)t * f.q_stride +
                                                     (int64_t)h * f.q_hstride + d);
  float m = -1.0e30f, l = 0.f;
  // a NaN in the query row itself: what was left is the result
  const unsigned long long nan = __ballot(q.x != q.x || q.y != q.y || q.z != q.z || q.w != q.w);
  if ((nan >> (threadIdx.x & 32)) & 0xffffffffu)
    return;
  v[0] = v[1] = v[2] = v[3] = 0.f;
#pragma unroll 1
  for (int key = 0; key <= f.q_offset + t; ++key) {
    const float4 k4 = *reinterpret_cast<const float4 *>(kp + (int64_t)key * kPromptD);
    const float4 v4 = *reinterpret_cast<const float4 *>(vp + (int64_t)key * kPromptD);
    float s = fmaf(q.w, k4.w, fmaf(q.z, k4.z, fmaf(q.y, k4.y, q.x * k4.x)));
#pragma unroll
    for (int o = 1; o < 32; o <<= 1)
      s += __shfl_xor(s, o, 64);
    s *= f.scale;
    const float mx = fmaxf(m, s), old = __builtin_amdgcn_exp2f(m - mx);
    const float w = __builtin_amdgcn_exp2f(s - mx);
    m = mx;
    l = fmaf(l, old, w);
    v[0] = fmaf(v4.x, w, v[0] * old);
    v[1] = fmaf(v4.y, w, v[1] * old);
    v[2] = fmaf(v4.z, w, v[2] * old);
    v[3] = fmaf(v4.w, w, v[3] * old);
    if (l != l) // the same in all lanes of the row
      break;
  }
  const float inv = 1.0f / l;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    v[e] *= inv;
}

// 1 / a row's sum of weights; NaN, so that the row is computed again, of one that is infinite
__device__ __forceinline__ float inverse_of(float sum) { return fmaf(sum, 0.f, 1.0f / sum); }

// Four values d .. d + 3 of query head h at token t, from where the launch left them; at most kMost parts
// asked for at once.  Sixteen take registers that leave a compute unit one workgroup of 512 threads: for as
// many tokens as make two rounds of those.  (1931 tokens 23 us so, four parts at once 14.2.)
constexpr int kFoldTokens = 512; // up to which sixteen are asked for
template <int kMost>
__device__ __forceinline__ void left4(const PromptFold &f, int64_t out_stride, int t, int h, int d,
                                      float (&v)[4]) {
  const int kvh = h / f.group, row = t * f.group + (h - kvh * f.group);
  const PromptBlock b = f.blocks[kvh * f.nblk + row / kPromptRows];
  if (b.parts == 0) {
    const float4 q = *reinterpret_cast<const float4 *>(f.out + (int64_t)t * out_stride +
                                                       (int64_t)h * kPromptD + d);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    return;
  }
  const int r = row % kPromptRows;
  auto slot = [&](int j) { return (size_t)(j ? 2 * (b.owner + j) : b.first) * kPromptRows + r; };
  float m = -INFINITY, l = 0.f, s[4] = {0.f, 0.f, 0.f, 0.f};
  // several parts in one trip to memory; past the last one it is asked for again and has
  // no weight
  auto add = [&](int j0, auto width) {
    constexpr int kWidth = decltype(width)::value;
    float2 ml[kWidth];
    float4 q[kWidth];
#pragma unroll
    for (int i = 0; i < kWidth; ++i) {
      const size_t at = slot(j0 + i < b.parts ? j0 + i : b.parts - 1);
      ml[i] = *reinterpret_cast<const float2 *>(f.ml + 2 * at);
      q[i] = *reinterpret_cast<const float4 *>(f.acc + at * kPromptD + d);
    }
    float mx = m;
#pragma unroll
    for (int i = 0; i < kWidth; ++i)
      mx = fmaxf(mx, ml[i].x);
    const float old = __builtin_amdgcn_exp2f(m - mx); // 0 the first time
    m = mx;
    l *= old;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      s[e] *= old;
#pragma unroll
    for (int i = 0; i < kWidth; ++i) {
      const float w = j0 + i < b.parts ? __builtin_amdgcn_exp2f(ml[i].x - m) : 0.f;
      l = fmaf(ml[i].y, w, l);
      s[0] = fmaf(q[i].x, w, s[0]);
      s[1] = fmaf(q[i].y, w, s[1]);
      s[2] = fmaf(q[i].z, w, s[2]);
      s[3] = fmaf(q[i].w, w, s[3]);
    }
  };
  if (kMost == 4 || b.parts <= 8)
    for (int j = 0; j < b.parts; j += 4)
      add(j, std::integral_constant<int, 4>{});
  else
    for (int j = 0; j < b.parts; j += kMost)
      add(j, std::integral_constant<int, kMost>{});
  const float inv = inverse_of(l);
#pragma unroll
  for (int e = 0; e < 4; ++e)
    v[e] = s[e] * inv;
}

// left4 leaves something that is not finite where a row is to be computed again.
__device__ __forceinline__ bool to_repair(const float (&v)[4]) {
  unsigned most = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    most = max(most, __float_as_uint(v[e]) & 0x7fffffffu);
  return most >= 0x7f800000u;
}
// ... which is done here, behind everything else (inside the loop over the heads: 600 tokens
// of 12 heads, all finite, 13.9 us; behind it 12.2; not at all 11.3).  Called by all 32 lanes
// of a row together, half a wavefront, with what left4 gave.
__device__ __forceinline__ void repair4(const PromptFold &f, int t, int h, int d, float (&v)[4]) {
  if ((__ballot(to_repair(v)) >> (threadIdx.x & 32)) & 0xffffffffu)
    f32_row(f, t, h, d, v);
}
#endif

} // namespace bh
