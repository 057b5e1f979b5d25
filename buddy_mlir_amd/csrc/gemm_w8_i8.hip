// gemm_w8_i8.hip -- the prefill matmul on the int8 matrix cores:
// C[M,N] (+)= A[M,K] . (int8 W[K,N] * scale[N]).
//
// Same contract as the bf16 kernels of gemm_w8_mfma.hip (the BLIS-style kernel
// of midend/lib/Conversion/MatMulOptimization/MatMulBlisVectorization.cpp:351-360,
// 398-986), another way to carry the f32 activations.  The int8 weights are used
// as they lie: a lane's 16 bytes of a packed 16 x 64 tile are an operand of
// v_mfma_i32_32x32x32_i8, so nothing is converted in the loop (the bf16 kernels
// spend more VALU time turning int8 into bf16 than the matrix cores spend on the
// products).  The activations become fixed point for that:
//   per row m a power-of-two step s[m] with |A[m,k]| / s[m] < 2^(8D-2),
//   X[m,k] = rint(A[m,k] / s[m])   (an integer of 8D-1 bits with its sign),
//   X = sum_j d_j 256^j with balanced digits d_j in [-128, 127] (each an int8;
//   the last one is what is left, at most 64 in magnitude),
// one integer matmul per digit plane with exact int32 sums, and
//   C[m,n] = s[m] * scale[n] * sum_j 256^j acc_j[m,n].
// The only rounding of the whole product is that of X: at most s/2 per element,
// i.e. 2^-(8D-1) of the row's largest magnitude (D = 3: 2^-23, the rounding an
// f32 sum of the same row makes when it adds the largest term; D = 2: 2^-15).
// The sums themselves are exact and do not depend on any order.  A row that
// holds a NaN or an infinity gets a NaN step, so every result of that row is
// NaN, as a NaN spreads through the reference's f32 multiply-add chain over the
// row (an infinity gives the reference +-inf or NaN per column; here NaN).
// |d q| <= 2^14, so K may not exceed 2^17.
//
// Digit planes lie in blocks of 32 rows x 64 k (plane_at), rows and k zero padded, followed
// by the row steps (f32 [rows_padded]): what a workgroup fetches at once is one run of
// memory.  (Rows of K bytes: a load instruction asks for half a cache line of each of 16
// rows.)  A lane's operand is 16 contiguous bytes of a row of a block.
//
// Workgroups take 32 rows x 128 or 256 channels, or one of the other tiles of kTiles1 to
// kTiles3, with the activation fragments shared through LDS.
#include "attn.h"
#include "attn_fold.h"
#include "attn_terms.h"
#include "digits_dev.h"
#include "gemm.h"
#include "tile_place.h"

#include <algorithm>
#include <cstdlib>
#include <map>
#include <mutex>
#include <type_traits>
#include <vector>

namespace bh {
namespace {

constexpr int kSlices = 4;    // wavefronts per workgroup

typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef int v2i32 __attribute__((ext_vector_type(2)));

// ---- f32 rows -> digit planes ------------------------------------------------

// smallest power of two s (not below 2^-126) with mx / s < 2^(8 D - 2)
__device__ __forceinline__ float digit_step(float mx, int D) {
  const int ex = (int)((__float_as_uint(mx) >> 23) & 0xffu) - 127; // floor(log2 mx)
  const int e = max(ex + 1 - (8 * D - 2), -126);
  return __uint_as_float((unsigned)(e + 127) << 23);
}

// Row sources: four consecutive values k0..k0+3 of the row (zero past its end).
__device__ __forceinline__ void load4(const float *p, int k0, int n, float (&v)[4]) {
  if (k0 + 3 < n && (reinterpret_cast<uintptr_t>(p + k0) & 15) == 0) {
    const float4 q = *reinterpret_cast<const float4 *>(p + k0);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = k0 + e < n ? p[k0 + e] : 0.f;
  }
}
struct PlainRow {
  static constexpr bool kRepairs = false;
  const float *a;
  int n;
  __device__ __forceinline__ void operator()(int k0, float (&v)[4]) const {
    load4(a, k0, n, v);
  }
};
struct NormRow { // w * (x * rs)
  static constexpr bool kRepairs = false;
  const float *x, *w;
  float rs;
  int n;
  __device__ __forceinline__ void operator()(int k0, float (&v)[4]) const {
    float xv[4], wv[4];
    load4(x, k0, n, xv);
    load4(w, k0, n, wv);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = wv[e] * (xv[e] * rs);
  }
};
// SiLU(g) * u with the one-instruction exp and reciprocal (1 ulp each)
__device__ __forceinline__ float silu_times(float g, float u) {
  const float sig = fast_rcp(1.0f + fast_exp(-g));
  return (g * sig) * u;
}
struct SiluMulRow { // silu(g) * u
  static constexpr bool kRepairs = false;
  const float *g, *u;
  int n;
  __device__ __forceinline__ void operator()(int k0, float (&v)[4]) const {
    float gv[4], uv[4];
    load4(g, k0, n, gv);
    load4(u, k0, n, uv);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = silu_times(gv[e], uv[e]);
  }
};

template <int kMost> struct FoldedRow { // the attention's output at one token, added up from its parts
  static constexpr bool kRepairs = true;
  const PromptFold &f;
  int64_t o_stride;
  int t, n;
  __device__ __forceinline__ void operator()(int k0, float (&v)[4]) const {
    v[0] = v[1] = v[2] = v[3] = 0.f;
    if (k0 < n)
      left4<kMost>(f, o_stride, t, k0 / kPromptD, k0 % kPromptD, v);
  }
  __device__ __forceinline__ void repair(int k0, float (&v)[4]) const {
    if (k0 < n)
      repair4(f, t, k0 / kPromptD, k0 % kPromptD, v);
  }
};

// Rows of up to this many values are kept in LDS between the pass that finds the
// row maximum and the pass that writes the digits; longer rows are computed twice.
constexpr int kRowCache = 12288;

constexpr int kRowThreads = 512; // threads of a producer workgroup (one row)

// One workgroup of kRowThreads threads writes row `row` of every plane and its step.
// A thread owns the same groups of four values in both passes.
template <class F>
__device__ __forceinline__ void row_to_digits(const F &f, int n, int row, int D, int Mp,
                                              int Kp, int8_t *planes, float *red,
                                              float *cache) {
  const bool cached = Kp <= kRowCache;
  // the row's largest magnitude as the largest bit pattern of |v|: a NaN or an
  // infinity is then the maximum (fmaxf would drop a NaN) and gives the row a
  // NaN step, so that every result of the row is NaN -- what the reference's f32
  // multiply-add chain makes of such a row (MatMulBlisVectorization.cpp:644-740)
  unsigned mb = 0;
  auto note = [&](const float (&v)[4]) {
    constexpr unsigned kAbs = 0x7fffffffu;
    mb = max(max(mb, max(__float_as_uint(v[0]) & kAbs, __float_as_uint(v[1]) & kAbs)),
             max(__float_as_uint(v[2]) & kAbs, __float_as_uint(v[3]) & kAbs));
  };
  auto row_max = [&]() {
    mb = wave_max_u32(mb);
    __syncthreads(); // red may still be read by the caller's own reduction
    if ((threadIdx.x & 63) == 0)
      red[threadIdx.x >> 6] = __uint_as_float(mb);
    __syncthreads();
    unsigned m2 = __float_as_uint(red[0]);
#pragma unroll
    for (int w = 1; w < kRowThreads / 64; ++w)
      m2 = max(m2, __float_as_uint(red[w]));
    mb = m2;
  };
#pragma unroll 3
  for (int k0 = threadIdx.x * 4; k0 < Kp; k0 += kRowThreads * 4) {
    float v[4];
    f(k0, v);
    note(v);
    if (cached)
      *reinterpret_cast<float4 *>(cache + k0) = make_float4(v[0], v[1], v[2], v[3]);
  }
  row_max();
  bool repaired = false; // once more where the source can do better than this
  if constexpr (F::kRepairs) {
    repaired = mb >= 0x7f800000u; // the same in all threads
    if (repaired) {
      mb = 0;
#pragma unroll 1
      for (int k0 = threadIdx.x * 4; k0 < Kp; k0 += kRowThreads * 4) {
        float v[4];
        f(k0, v);
        f.repair(k0, v);
        note(v);
        if (cached)
          *reinterpret_cast<float4 *>(cache + k0) = make_float4(v[0], v[1], v[2], v[3]);
      }
      row_max();
    }
  }
  const bool finite = mb < 0x7f800000u;
  const float step = finite ? digit_step(__uint_as_float(mb), D) : __uint_as_float(0x7fc00000u);
  // a power of two as well
  const float inv = finite ? 1.0f / step : 0.f;
  float *steps = reinterpret_cast<float *>(planes + (size_t)D * Mp * Kp);
  if (threadIdx.x == 0)
    steps[row] = step;
  for (int k0 = threadIdx.x * 4; k0 < Kp; k0 += kRowThreads * 4) {
    float v[4];
    if (cached) {
      const float4 q = *reinterpret_cast<const float4 *>(cache + k0);
      v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else {
      f(k0, v);
      if constexpr (F::kRepairs) {
        if (repaired)
          f.repair(k0, v);
      }
    }
    unsigned word[3];
    digits_of(v, inv, D, word);
    unsigned *dst = reinterpret_cast<unsigned *>(planes + plane_at(row, k0, 0, D, Kp));
    dst[0] = word[0];
    dst[kPlaneBlock / 4] = word[1];
    if (D == 3)
      dst[2 * (kPlaneBlock / 4)] = word[2];
  }
}

__device__ __forceinline__ void padding_to_digits(int row, int D, int Mp, int Kp, int8_t *planes) {
  for (int j = 0; j < D; ++j)
    for (int k0 = threadIdx.x * 4; k0 < Kp; k0 += (int)blockDim.x * 4)
      *reinterpret_cast<unsigned *>(planes + plane_at(row, k0, j, D, Kp)) = 0u;
  if (threadIdx.x == 0)
    reinterpret_cast<float *>(planes + (size_t)D * Mp * Kp)[row] = 1.0f;
}

// Two rows of a plane's block are a cache line: workgroups 8 apart, which run on one XCD, take them, so that its
// L2 writes the line whole (of the kernels that fold attention and add slices, too: 1931 rows 14.5 -> 13.8 us,
// 20.4 -> 19.7).  Of a grid of a multiple of 16.
__device__ __forceinline__ int row_of_workgroup() {
  const int b = blockIdx.x;
  return (b & ~15) | (b & 7) << 1 | (b >> 3 & 1);
}
inline unsigned row_workgroups(int64_t rows) { return (unsigned)round_up(rows, 16); }

// Rows of up to NV x 4 x kThreads values, a multiple of four, 16-byte aligned; NORM: RMSNorm(row) * w.  Everything is
// asked for at once and stays in registers: one trip to memory, and for many rows its bytes (1931 rows of 8960 values
// 121 MB at 5.6 TB/s).  us with rows in LDS or read twice, lines written by two XCDs, and so: 1931 rows of 8960
// 26.8 and 21.6, normed of 1536 8.9 and 6.2; 512 rows 7.2 and 6.9, 5.2 and 5.2.
template <int NV, bool NORM, int kThreads>
__global__ void __launch_bounds__(kThreads)
rows_to_digits_kernel(const float *A, int64_t lda, const float *w, int M, int K, float inv_n, float eps, int D, int Mp,
                      int Kp, int8_t *planes) {
  constexpr int kWaves = kThreads / 64;
  __shared__ float sums[kWaves];
  __shared__ unsigned most[kWaves];
  const int row = row_of_workgroup(), tid = threadIdx.x;
  if (row >= M) { // padding rows: zero digits, step 1 (where they are asked for)
    if (!NORM && row < Mp)
      padding_to_digits(row, D, Mp, Kp, planes);
    return;
  }
  const float *src = A + (int64_t)row * lda;
  float v[NV][4], nw[NORM ? NV : 1][4];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k0 = (i * kThreads + tid) * 4, at = min(k0, K - 4);
    const float4 q = *reinterpret_cast<const float4 *>(src + at);
    v[i][0] = q.x; v[i][1] = q.y; v[i][2] = q.z; v[i][3] = q.w;
    if constexpr (NORM) {
      const float4 u = *reinterpret_cast<const float4 *>(w + at);
      nw[i][0] = u.x; nw[i][1] = u.y; nw[i][2] = u.z; nw[i][3] = u.w;
    }
  }
  if constexpr (NORM) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if ((i * kThreads + tid) * 4 < K)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          s = fmaf(v[i][e], v[i][e], s);
    s = wave_sum(s);
    if ((tid & 63) == 0)
      sums[tid >> 6] = s;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int i = 0; i < kWaves; ++i)
      tot += sums[i];
    const float rs = 1.0f / sqrtf(tot * inv_n + eps);
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[i][e] = nw[i][e] * (v[i][e] * rs);
  }
  // values behind the row repeat its last ones; see row_to_digits for what a NaN does
  unsigned mb = 0;
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      mb = max(mb, __float_as_uint(v[i][e]) & 0x7fffffffu);
  mb = wave_max_u32(mb);
  if ((tid & 63) == 0)
    most[tid >> 6] = mb;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kWaves; ++i)
    mb = max(mb, most[i]);
  const bool finite = mb < 0x7f800000u;
  const float step = finite ? digit_step(__uint_as_float(mb), D) : __uint_as_float(0x7fc00000u);
  const float inv = finite ? 1.0f / step : 0.f;
  if (tid == 0)
    reinterpret_cast<float *>(planes + (size_t)D * Mp * Kp)[row] = step;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k0 = (i * kThreads + tid) * 4;
    if (k0 >= Kp)
      break;
    unsigned word[3] = {};
    if (k0 < K)
      digits_of(v[i], inv, D, word);
    unsigned *dst = reinterpret_cast<unsigned *>(planes + plane_at(row, k0, 0, D, Kp));
    dst[0] = word[0];
    dst[kPlaneBlock / 4] = word[1];
    if (D == 3)
      dst[2 * (kPlaneBlock / 4)] = word[2];
  }
}

__global__ void __launch_bounds__(kRowThreads)
activations_to_digits_kernel(const float *__restrict__ A, int64_t lda, int M, int K, int D,
                             int Mp, int Kp, int8_t *__restrict__ planes) {
  __shared__ float red[kRowThreads / 64];
  extern __shared__ __attribute__((aligned(16))) float row_cache[];
  const int row = blockIdx.x;
  if (row >= M) { // padding rows: zero digits, step 1
    padding_to_digits(row, D, Mp, Kp, planes);
    return;
  }
  row_to_digits(PlainRow{A + (int64_t)row * lda, K}, K, row, D, Mp, Kp, planes, red,
                row_cache);
}

template <int kMost>
__global__ void __launch_bounds__(kRowThreads, kMost == 4 ? 8 : 1)
attn_fold_to_digits_kernel(PromptFold f, int64_t o_stride, int M, int K, int D, int Mp, int Kp,
                           int8_t *__restrict__ planes) {
  __shared__ float red[kRowThreads / 64];
  extern __shared__ __attribute__((aligned(16))) float row_cache[];
  const int row = row_of_workgroup();
  if (row >= M) {
    padding_to_digits(row, D, Mp, Kp, planes);
    return;
  }
  row_to_digits(FoldedRow<kMost>{f, o_stride, row, K}, K, row, D, Mp, Kp, planes, red, row_cache);
}

__global__ void __launch_bounds__(kRowThreads)
rmsnorm_to_digits_kernel(const float *__restrict__ x, int64_t ldx,
                         const float *__restrict__ w, int n, float inv_n, float eps, int D,
                         int Mp, int Kp, int8_t *__restrict__ planes) {
  __shared__ float red[kRowThreads / 64];
  extern __shared__ __attribute__((aligned(16))) float row_cache[];
  const int row = blockIdx.x;
  const float *xr = x + (int64_t)row * ldx;
  float s = 0.f;
  for (int i = threadIdx.x; i < n; i += kRowThreads)
    s = fmaf(xr[i], xr[i], s);
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = s;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int w = 0; w < kRowThreads / 64; w += 2) // pairs first, as four wavefronts did
    tot += red[w] + red[w + 1];
  const float rs = 1.0f / sqrtf(tot * inv_n + eps);
  row_to_digits(NormRow{xr, w, rs, n}, n, row, D, Mp, Kp, planes, red, row_cache);
}

__global__ void __launch_bounds__(kRowThreads)
silu_mul_to_digits_kernel(const float *__restrict__ g, const float *__restrict__ u, int64_t ld,
                          int n, int D, int Mp, int Kp, int8_t *__restrict__ planes) {
  __shared__ float red[kRowThreads / 64];
  extern __shared__ __attribute__((aligned(16))) float row_cache[];
  const int row = blockIdx.x;
  row_to_digits(SiluMulRow{g + (size_t)row * ld, u + (size_t)row * ld, n}, n, row, D, Mp, Kp,
                planes, red, row_cache);
}

// ---- the matmul ----------------------------------------------------------------

struct GemmI8Args {
  const int8_t *planes; // blocks of plane_at
  const float *steps;   // [Mp]
  const int4 *W;
  const float *scale;
  const float *bias;
  float *C;
  int64_t ldc;
  int M, N, Mp, Kp, groups, chunks;
  int ncols, row_tiles, panel; // column tiles, row tiles, and how they are placed
  int span;      // channels per wavefront, where K is split
  int tile_rows; // rows per workgroup, where K is split
  // K split over `slices` workgroups per tile, chunks_per_slice chunks each
  // (the last may hold fewer, never none); partial is only used when slices > 1
  int slices, chunks_per_slice;
  float *partial;     // [tile][slice][wavefront][row][channel]
  int accumulate;
  int32_t *sums;      // one plane only: the int32 sums themselves, dense [M, N], or null
  int int_partials;   // one plane, K split: the slices leave their int32 sums as they are
  RopeKv rope;        // of q | k | v that the product itself rotates
};

// The finished value of one output.  One plane is the w8a8 matmul, whose result
// is f32(sum) * (s_a * s_w[n]) in exactly that order (linalg.py:12833-12845).
template <int D> __device__ __forceinline__ float scaled(float v, float step, float s) {
  return D == 1 ? v * (step * s) : (v * step) * s;
}

// A tile: 32 RB rows x 128 GP channels per workgroup (GP tiles of 32 channels per
// wavefront), every wavefront runs the whole K on v_mfma_i32_32x32x32_i8.  A wavefront
// that has its SIMD to itself issues that instruction at its full rate, the 16 x 16 x 64
// one at two thirds of it, and it reads half as many operands per product.  Its A operand
// is 32 channels x 32 k: the lanes take it from the tiles of two channel groups.  What
// bounds it: 1931 rows of gate | up run at 1.87 P operations/s (16 x 16 x 64: 1.57), half
// of what the instruction alone reaches; twice the rows per weight give no more (below).
//
// The digit planes' rows go through LDS, shared by the wavefronts; weights go from memory
// to registers to the matrix core.  Weights are asked for three chunks of 64 k
// ahead, rows five (two in LDS: step c multiplies buffer c % 3, whose first fragments were
// read during step c - 1, and fills buffer (c + 2) % 3, last read before the previous
// barrier).
//
// Matrices too narrow to fill the chip with such tiles split K over several
// workgroups per tile instead of shrinking the tile (a 64 x 64 tile reads its
// operands four times as often from L2, and that, not the matrix cores, is what
// bounds it).  Every slice writes its unscaled sums to a workspace and a second
// small kernel adds the slices in slice order, applies the scales and writes C.
// (Finishing a tile inside the kernel, by the workgroup that arrives last at a
// counter, needs device-scope fences; on this chip they write back and
// invalidate a whole L2 each time and slowed the running workgroups threefold.)
//
// PAIR: W holds two matrices of a.groups / 2 channel groups each, one behind the
// other; a tile is a group of the first and the same group of the second, so that a lane
// holds matching channels of both, and the result is SiLU(first) * second ([M, N / 2]).
typedef int v16i32 __attribute__((ext_vector_type(16)));
// Blocks of 32 rows of the tile of 256 channels that every launch of some size can use (of
// one plane, whose weights are otherwise used for too little: 512 rows, 1536 -> 8960, 31.2 us
// on blocks of one; of two 26, of three 25).
constexpr int wide_blocks(int D) { return D == 1 ? 2 : 1; }
constexpr int kWideRow = kTileK + 16; // bytes of a row in LDS: fragment reads meet every bank once

// sum_j 256^j acc_j as f32 (each int32 sum is exact; the conversions round to 24
// bits, like an f32 accumulator would)
template <int D> __device__ __forceinline__ float combine(const v16i32 (&acc)[D], int r) {
  float v = (float)acc[D - 1][r];
#pragma unroll
  for (int j = D - 2; j >= 0; --j)
    v = fmaf(v, 256.0f, (float)acc[j][r]);
  return v;
}

// sums 4 q .. 4 q + 3 as they are, carried as float bit patterns
__device__ __forceinline__ float4 int_bits(const v16i32 &acc, int q) {
  return make_float4(__int_as_float(acc[4 * q]), __int_as_float(acc[4 * q + 1]),
                     __int_as_float(acc[4 * q + 2]), __int_as_float(acc[4 * q + 3]));
}

constexpr int turn_floats(int span) { return span + 4; } // of a row of the epilogue's tile
constexpr int turned_bytes(int span) { return kSlices * 32 * turn_floats(span) * 4; }

// What follows q | k | v, for a tile whose finished values lie in LDS (32 rows of 4 x `kSpan` channels, whole
// heads): sixteen lanes take a head's row, four channels and their partners each, rotate it by angles that
// the prompt has as a table, and store queries to C, keys and values to the cache and, of a prompt alone, as
// terms; a tile of terms is these 32 rows.  A launch for it was 5.6 us behind 512 tokens' product and 10.1
// behind 1931's, most of which were its own and two more trips of the values; here 1 and 2.
template <int GP>
__device__ __forceinline__ void rotate_tile(const GemmI8Args &a, unsigned char *lds, int ctile, int m0) {
  constexpr int kSpan = 32 * GP, kTurn = turn_floats(kSpan), kHalf = kAttnHeadDim / 2, kPasses = 2 * GP;
  constexpr int kKeys = kTileKeys + 2; // of a channel in LDS: sixteen lanes' stores meet sixteen banks
  static_assert(kAttnHeadDim == 4 * 32 && 2 * kAttnHeadDim * kKeys * 2 <= turned_bytes(32), "a head a channel tile");
  const int tid = threadIdx.x, j = tid % 16 * 4;
  const RopeKv &r = a.rope;
  float lo[kPasses][4], hi[kPasses][4];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPasses; ++i) { // pass i: rows 16 (i % 2) + 0..15 of head i / 2
    const int row = i % 2 * 16 + tid / 16;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int ch = i / 2 * kAttnHeadDim + h * kHalf + j;
      const float4 v = *reinterpret_cast<const float4 *>(
          reinterpret_cast<const float *>(lds) + (ch / kSpan * 32 + row) * kTurn + ch % kSpan);
      float *to = h ? hi[i] : lo[i];
      to[0] = v.x; to[1] = v.y; to[2] = v.z; to[3] = v.w;
    }
  }
  __syncthreads(); // the values have been read: LDS is free
  auto store = [&](float *dst, const float (&l)[4], const float (&h)[4]) {
    *reinterpret_cast<float4 *>(dst) = make_float4(l[0], l[1], l[2], l[3]);
    *reinterpret_cast<float4 *>(dst + kHalf) = make_float4(h[0], h[1], h[2], h[3]);
  };
  unsigned short(*vt)[kAttnHeadDim][kKeys] = reinterpret_cast<unsigned short(*)[kAttnHeadDim][kKeys]>(lds);
#pragma unroll
  for (int i = 0; i < kPasses; ++i) {
    const int head = ctile * GP + i / 2, row = i % 2 * 16 + tid / 16, m = m0 + row, pos = r.start_pos + m;
    if (head * kAttnHeadDim >= a.N)
      break;
    const bool is = m < a.M;
    if (head < r.heads + r.kv_heads) {
      if (!is)
        continue;
      const float *turns = r.turns + (int64_t)m * kAttnHeadDim + j;
      const float4 c4 = *reinterpret_cast<const float4 *>(turns), s4 = *reinterpret_cast<const float4 *>(turns + kHalf);
      const float c[4] = {c4.x, c4.y, c4.z, c4.w}, s[4] = {s4.x, s4.y, s4.z, s4.w};
      float nlo[4], nhi[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        nlo[e] = lo[i][e] * c[e] + (-hi[i][e]) * s[e];
        nhi[e] = hi[i][e] * c[e] + lo[i][e] * s[e];
      }
      if (head < r.heads) {
        store(a.C + (int64_t)m * a.ldc + head * kAttnHeadDim + j, nlo, nhi);
      } else {
        const int kvh = head - r.heads;
        store(r.kcache + ((int64_t)kvh * r.max_len + pos) * kAttnHeadDim + j, nlo, nhi);
        if (r.terms.tiles)
          put_key_terms(r.terms, kvh, pos, j / 4, nlo, nhi);
      }
      continue;
    }
    const int kvh = head - r.heads - r.kv_heads;
    if (is)
      store(r.vcache + ((int64_t)kvh * r.max_len + pos) * kAttnHeadDim + j, lo[i], hi[i]);
    if (!r.terms.tiles)
      continue;
    uint4 term[2] = {}; // of rows behind the prompt: numbers
    if (is)
      value_terms(r.terms, kvh, pos, j / 4, lo[i], hi[i], term);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const unsigned w[4] = {term[p].x, term[p].y, term[p].z, term[p].w};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        vt[p][kHalf * (e / 4) + j + e % 4][row] = (unsigned short)(e & 1 ? w[e / 2] >> 16 : w[e / 2]);
    }
    if (i % 2 == 0)
      continue;
    __syncthreads();
    // sixteen bytes are keys 16 s + 4 half + 0..3 and the four 8 behind them, of a channel
    unsigned char *tile = terms_tile(r.terms, kvh, r.start_pos + m0);
#pragma unroll
    for (int u = 0; u < 2 * 4 * kAttnHeadDim / 256; ++u) {
      const int id = u * 256 + tid, c = id % kAttnHeadDim, key = id / kAttnHeadDim % 4 * 4, p = id / (4 * kAttnHeadDim);
      const int first = key / 8 * 16 + key % 8;
      const unsigned *from = reinterpret_cast<const unsigned *>(&vt[p][c][first]);
      *reinterpret_cast<uint4 *>(value_term_at(tile, first, c, p)) = uint4{from[0], from[1], from[4], from[5]};
    }
    if (i + 1 < kPasses)
      __syncthreads();
  }
}

// The way of a tile's sums out, behind the last barrier of the loop over K (`lds` is free).
template <int D, int RB, int GP, bool PAIR, bool ROPE = false>
__device__ __forceinline__ void finish_tile(const GemmI8Args &a, const v16i32 (&acc)[GP][RB][D], unsigned char *lds,
                                            const float *scale_s, const float *bias_s, const float *step_s,
                                            int ctile, int rbk, int slice, int g0, int m0, int wave, int lane) {
  constexpr int kWidth = PAIR ? 16 : 32, kSpan = kWidth * GP, kRows = 32 * RB;
  constexpr int kTurn = turn_floats(kSpan), kScales = kSlices * 32 * GP;
  const int col = lane & 31, up = lane >> 5;
  // A lane holds channels 8 q + 4 up + 0..3, q = 0..3, of row `col` of every tile: stored
  // as they are, a store instruction would write 32-byte pieces of 32 rows.  Each
  // wavefront turns its 32 rows around in its own part of LDS (free now: every wavefront
  // is past the last barrier of the loop) and writes whole row segments.
  float *tile = reinterpret_cast<float *>(lds) + wave * (32 * kTurn);
  const int n0 = g0 * kTileN;
  auto turn_in = [&](int g, int q, float4 v) {
    *reinterpret_cast<float4 *>(tile + col * kTurn + g * kWidth + 8 * q + 4 * up) = v;
  };
  constexpr int kQuads = kSpan / 4; // float4 of a row
  if (a.slices > 1) {
    // unscaled sums of this slice, [wavefront][row][channel]; the kernel that adds the
    // slices finishes the tile
    const size_t at = ((size_t)(rbk * a.ncols + ctile) * a.slices + slice) * kSlices + wave;
    float *part = a.partial + at * kRows * kSpan;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      if (rb > 0)
        lds_turn();
#pragma unroll
      for (int g = 0; g < GP; ++g)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const v16i32(&t)[D] = acc[g][rb];
          float4 o = make_float4(combine<D>(t, 4 * q), combine<D>(t, 4 * q + 1),
                                 combine<D>(t, 4 * q + 2), combine<D>(t, 4 * q + 3));
          if constexpr (D == 1) {
            if (a.int_partials) // exact beyond 2^24: the bits travel as they are
              o = int_bits(t[0], q);
          }
          turn_in(g, q, o);
        }
      lds_turn();
#pragma unroll
      for (int i = 0; i < kQuads / 2; ++i) {
        const int idx = lane + 64 * i, row = idx / kQuads, c4 = idx % kQuads;
        *reinterpret_cast<float4 *>(part + (size_t)(rb * 32 + row) * kSpan + c4 * 4) =
            *reinterpret_cast<const float4 *>(tile + row * kTurn + c4 * 4);
      }
    }
    return;
  }
  const bool vec = (a.ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(a.C) & 15) == 0;
  const float *scales = scale_s + wave * kSpan;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const float row_step = step_s[rb * 32 + col];
    if (rb > 0)
      lds_turn();
#pragma unroll
    for (int g = 0; g < GP; ++g)
#pragma unroll
      for (int q = 0; q < kWidth / 8; ++q) {
        const int ch = g * kWidth + 8 * q + 4 * up;
        const v16i32(&t)[D] = acc[g][rb];
        const float4 sc = *reinterpret_cast<const float4 *>(scales + ch);
        const float s[4] = {sc.x, sc.y, sc.z, sc.w};
        float o[4];
        if constexpr (PAIR) {
          const float4 su = *reinterpret_cast<const float4 *>(scales + kScales / 2 + ch);
          const float s2[4] = {su.x, su.y, su.z, su.w};
#pragma unroll
          for (int i = 0; i < 4; ++i)
            o[i] = silu_times(scaled<D>(combine<D>(t, 4 * q + i), row_step, s[i]),
                              scaled<D>(combine<D>(t, 4 * q + 8 + i), row_step, s2[i]));
        } else {
          const float4 bb = *reinterpret_cast<const float4 *>(bias_s + wave * kSpan + ch);
          const float b[4] = {bb.x, bb.y, bb.z, bb.w};
#pragma unroll
          for (int i = 0; i < 4; ++i)
            o[i] = b[i] + scaled<D>(combine<D>(t, 4 * q + i), row_step, s[i]);
        }
        turn_in(g, q, make_float4(o[0], o[1], o[2], o[3]));
      }
    if constexpr (ROPE) {
      static_assert(RB == 1 && !PAIR, "the rows of a tile of terms");
      rotate_tile<GP>(a, lds, ctile, m0);
      return;
    }
    lds_turn();
#pragma unroll
    for (int i = 0; i < kQuads / 2; ++i) {
      const int idx = lane + 64 * i, row = idx / kQuads, c4 = idx % kQuads;
      const float4 o = *reinterpret_cast<const float4 *>(tile + row * kTurn + c4 * 4);
      const int m = m0 + rb * 32 + row, n = n0 + c4 * 4;
      if (m >= a.M || n >= a.N)
        continue;
      float *cp = a.C + (int64_t)m * a.ldc + n;
      if (vec && n + 3 < a.N) {
        float4 q = o;
        if (a.accumulate) {
          const float4 p = *reinterpret_cast<const float4 *>(cp);
          q = make_float4(p.x + q.x, p.y + q.y, p.z + q.z, p.w + q.w);
        }
        *reinterpret_cast<float4 *>(cp) = q;
      } else {
        const float v[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < a.N)
            cp[r] = a.accumulate ? cp[r] + v[r] : v[r];
      }
    }
    if constexpr (D == 1) {
      if (a.sums) { // the same turn for the integer sums, carried as float bit patterns
        lds_turn();
#pragma unroll
        for (int g = 0; g < GP; ++g)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            turn_in(g, q, int_bits(acc[g][rb][0], q));
        lds_turn();
        const bool ivec = (a.N & 3) == 0 && (reinterpret_cast<uintptr_t>(a.sums) & 15) == 0;
#pragma unroll
        for (int i = 0; i < kQuads / 2; ++i) {
          const int idx = lane + 64 * i, row = idx / kQuads, c4 = idx % kQuads;
          const float4 q = *reinterpret_cast<const float4 *>(tile + row * kTurn + c4 * 4);
          const v4i32 o = {__float_as_int(q.x), __float_as_int(q.y), __float_as_int(q.z),
                           __float_as_int(q.w)};
          const int m = m0 + rb * 32 + row, n = n0 + c4 * 4;
          if (m >= a.M || n >= a.N)
            continue;
          int32_t *cp = a.sums + (int64_t)m * a.N + n;
          if (ivec) {
            *reinterpret_cast<v4i32 *>(cp) = o;
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (n + r < a.N)
                cp[r] = o[r];
          }
        }
      }
    }
  }
}

template <int D, int RB, int GP, bool PAIR, bool ROPE = false>
__device__ __forceinline__ void multiply_tile(const GemmI8Args &a, int unit, int rbk, int row0 = 0) {
  constexpr int kWidth = PAIR ? 16 : 32;    // channels of the result per tile
  constexpr int kSpan = kWidth * GP;        // ... and per wavefront
  constexpr int kRows = 32 * RB;            // rows of the tile
  constexpr int L = D * RB;                 // layers of 32 rows: plane l % D of row block l / D
  constexpr int kThreads = kSlices * kWave;
  // a thread's loads of a chunk's rows: 16 bytes of two layers at a time, 8 of an odd last one
  constexpr int kQuad = L / 2, kLoads = (L + 1) / 2;
  constexpr int kBuf = L * 32 * kWideRow;
  constexpr int kTurned = turned_bytes(kSpan);
  constexpr int kLds = 3 * kBuf > kTurned ? 3 * kBuf : kTurned;
  constexpr int kScales = kSlices * 32 * GP;
  // chunks of weights and of rows in registers
  constexpr int kRing = 4;
  constexpr int kFetches = 2 * GP + kLoads; // loads of a chunk
  // the first load issued with sub-step u
  auto first_fetch = [](int u) constexpr {
    if (D > 1 || L == 1)
      return u * kFetches / (2 * L);
    return u == 0 ? 0 : u <= 2 ? 2 * GP : kFetches;
  };
  __shared__ __attribute__((aligned(16))) unsigned char lds[kLds];
  // the epilogue's operands, asked for as the launch starts: scales (PAIR: of both
  // matrices), bias, row steps
  __shared__ __attribute__((aligned(16))) float scale_s[kScales], bias_s[PAIR ? 4 : kScales];
  __shared__ float step_s[kRows];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, up = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ctile = unit % a.ncols, slice = unit / a.ncols;
  const int m0 = row0 + rbk * kRows;
  const int half_groups = a.groups / 2; // PAIR only
  const int glast = PAIR ? half_groups - 1 : a.groups - 1;
  const int g0 = (ctile * kSlices + wave) * (kSpan / 16); // first channel group of this wavefront
  const int cb = slice * a.chunks_per_slice;
  const int nch = min(a.chunks_per_slice, a.chunks - cb); // chunks of this slice, >= 1

  const v4i32 *wp[GP];
#pragma unroll
  for (int g = 0; g < GP; ++g) { // groups past the end repeat the last one
    const int second = (lane >> 4) & 1; // group of the tile
    const int gg =
        PAIR ? min(g0 + g, glast) + second * half_groups : min(g0 + 2 * g + second, glast);
    wp[g] = reinterpret_cast<const v4i32 *>(a.W) + ((size_t)gg * a.chunks + cb) * 64 + up * 16 +
            (lane & 15);
  }
  const int8_t *src[kLoads];
  int lds_at[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int run = i < kQuad ? 16 : 8, at = tid * run; // of layers 2 i and 2 i + 1
    const int l = 2 * i + at / kPlaneBlock, r = at % kPlaneBlock / kTileK, k = at % kTileK;
    const int block = min(m0 / 32 + l / D, a.Mp / 32 - 1);
    src[i] = a.planes + (((size_t)block * a.chunks + cb) * D + l % D) * kPlaneBlock + r * kTileK + k;
    lds_at[i] = (l * 32 + r) * kWideRow + k;
  }
  struct Rows {
    v4i32 q[kQuad ? kQuad : 1];
    v2i32 h;
  };
  v4i32 wr[kRing][GP * 2];
  Rows xr[kRing];
  auto fetch_w = [&](int c, v4i32 (&w)[GP * 2]) {
    const size_t cc = (size_t)min(c, nch - 1) * 64;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int g = 0; g < GP; ++g)
        w[g * 2 + h] = wp[g][cc + h * 32];
  };
  auto fetch_run = [&](int i, size_t cc, Rows &x) {
    if (i < kQuad)
      x.q[i] = *reinterpret_cast<const v4i32 *>(src[i] + cc);
    else
      x.h = *reinterpret_cast<const v2i32 *>(src[i] + cc);
  };
  auto put_run = [&](int i, const Rows &x, unsigned char *buf) {
    if (i < kQuad)
      *reinterpret_cast<v4i32 *>(buf + lds_at[i]) = x.q[i];
    else
      *reinterpret_cast<v2i32 *>(buf + lds_at[i]) = x.h;
  };
  auto fetch_x = [&](int c, Rows &x) {
    const size_t cc = (size_t)min(c, nch - 1) * (D * kPlaneBlock);
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      fetch_run(i, cc, x);
  };
  auto put_x = [&](const Rows &x, unsigned char *buf) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      put_run(i, x, buf);
  };
  fetch_x(0, xr[0]);
  fetch_x(1, xr[1]);
#pragma unroll
  for (int u = 0; u < kRing - 1; ++u) {
    fetch_w(u, wr[u]);
    if (u + 2 < kRing)
      fetch_x(u + 2, xr[u + 2]);
  }
  if (a.slices == 1) {
    const int n0 = ctile * kSlices * kSpan;
    for (int i = tid; i < kScales; i += kThreads) {
      const int mtx = PAIR ? i / (kScales / 2) : 0, n = n0 + (PAIR ? i % (kScales / 2) : i);
      scale_s[i] = n < a.N ? a.scale[(size_t)mtx * a.N + n] : 0.f;
      if constexpr (!PAIR)
        bias_s[i] = a.bias && n < a.N ? a.bias[n] : 0.f;
    }
    for (int i = tid; i < kRows; i += kThreads)
      step_s[i] = m0 + i < a.M ? a.steps[m0 + i] : 0.f;
  }

  v16i32 acc[GP][RB][D];
#pragma unroll
  for (int g = 0; g < GP; ++g)
#pragma unroll
    for (int l = 0; l < L; ++l)
      acc[g][l / D][l % D] = v16i32{};

  unsigned char *cur = lds, *next = lds + kBuf, *fill = lds + 2 * kBuf;
  put_x(xr[0], cur);
  put_x(xr[1], next);
  fetch_x(kRing, xr[0]);
  __syncthreads();
  const int frag_at = col * kWideRow + up * 16;
  v4i32 frag[4];
  // sub-step u of a chunk: layer u % L, k half u / L
  auto load_frag = [&](const unsigned char *buf, int u, v4i32 &f) {
    f = *reinterpret_cast<const v4i32 *>(buf + frag_at + u % L * 32 * kWideRow + u / L * 32);
  };
  load_frag(cur, 0, frag[0]);
  load_frag(cur, 1, frag[1]);
  // f: the slot of sub-step 0's fragments
  auto step = [&](int c, int f, v4i32 (&w)[GP * 2], v4i32 (&w_new)[GP * 2], const Rows &x,
                  Rows &x_new) {
    const size_t wc = (size_t)min(c + kRing - 1, nch - 1) * 64;
    const size_t xc = (size_t)min(c + kRing + 1, nch - 1) * (D * kPlaneBlock);
#pragma unroll
    for (int u = 0; u < 2 * L; ++u) {
      // fragments are asked for two sub-steps ahead of their products (one takes less than
      // the way through LDS), and stay there: left to itself the scheduler moves them to
      // their use
      load_frag(u + 2 < 2 * L ? cur : next, (u + 2) % (2 * L), frag[(f + u + 2) & 3]);
      // a chunk's loads, weights first: evenly between its products (all at its start: 171
      // against 167 us for gate | up of 1931 rows), for one plane, which has a third of the
      // products, at the start (19.2 against 21)
#pragma unroll
      for (int i = first_fetch(u); i < first_fetch(u + 1); ++i) {
        if (i < 2 * GP)
          w_new[i % GP * 2 + i / GP] = wp[i % GP][wc + i / GP * 32];
        else
          fetch_run(i - 2 * GP, xc, x_new);
      }
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        if (u == (i + 1 < 2 * L - 2 ? i + 1 : 1))
          put_run(i, x, fill);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < GP; ++g)
        acc[g][u % L / D][u % D] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
            w[g * 2 + u / L], frag[(f + u) & 3], acc[g][u % L / D][u % D], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    unsigned char *t = cur;
    cur = next;
    next = fill;
    fill = t;
  };
  // step c: weights from slot c, new ones into slot c - 1; rows c + 2 go to LDS, new ones
  // into slot c + 1 (all modulo kRing)
  auto turn = [&](int c0, auto slot) {
    constexpr int u = slot;
    step(c0 + u, (u * 2 * L) & 3, wr[u], wr[(u + kRing - 1) % kRing], xr[(u + 2) % kRing],
         xr[(u + 1) % kRing]);
  };
  // No branch within a round of the ring: where paths of fewer steps join, the compiler waits
  // for all loads but those of the shortest path ahead of any register it uses again.
  using std::integral_constant;
  int c0 = 0;
  for (; c0 + kRing <= nch; c0 += kRing) {
    turn(c0, integral_constant<int, 0>{});
    turn(c0, integral_constant<int, 1>{});
    turn(c0, integral_constant<int, 2>{});
    turn(c0, integral_constant<int, 3>{});
  }
  static_assert(kRing == 4, "a round is written out");
  if (c0 < nch) {
    turn(c0, integral_constant<int, 0>{});
    if (c0 + 1 < nch) {
      turn(c0, integral_constant<int, 1>{});
      if (c0 + 2 < nch)
        turn(c0, integral_constant<int, 2>{});
    }
  }

  finish_tile<D, RB, GP, PAIR, ROPE>(a, acc, lds, scale_s, bias_s, step_s, ctile, rbk, slice, g0, m0, wave, lane);
}

// The same product for tiles of many sums, two workgroups to a compute unit: two wavefronts on a
// SIMD have 256 registers each, of which the sums of 64 rows x 64 channels in three planes are
// 192, so the rows come from memory to LDS past the registers, three chunks ahead, and the weights
// half a chunk at a time, three of them ahead.  One workgroup loads and stores beside the
// products of the other.
//
// What bounds it: power.  gate | up of 1931 rows with three planes takes 146 us (the same tile
// alone on its compute unit, rows through registers, 180; 32 rows x 256 channels two to a compute
// unit 170), and 108 where rows and weights are zero: the clock falls from 2.3 to below 1.8 GHz
// with what the matrix cores draw.  Conflicts in LDS (a third of its cycles with pieces permuted by
// r / 2) or none, and either order of the products of a fragment, made no difference.
//
// A plane's block lies in LDS as it lies in memory but for the four 16-byte pieces of a row, which
// are permuted by the row's number: piece p of row r is where p ^ (r / 4 % 4) would be, and the
// fragment reads of sixteen rows in a line meet every bank once.
//
// Every step issues kDma loads into LDS and 2 GP of weights in that order.

// the tiles of gemm_w8_i8_tall_kernel that go this way
constexpr bool tall_shares(int D, int GP) { return D >= 2 && GP == 2; }
// A lane reaches its group of a pair's second matrix by 32 bits from a group of the first: matrices of
// fewer than 2^22 tiles (1 KiB each).  Larger ones go by multiply_tile, whose lanes have 64-bit addresses.
inline bool pair_in_reach(int64_t channels, int64_t chunks) { return ceil_div(channels, kTileN) * chunks < (1 << 22); }

template <int D, int RB, int GP, bool PAIR>
__device__ __forceinline__ void multiply_block(const GemmI8Args &a, int unit, int rbk) {
  constexpr int kWidth = PAIR ? 16 : 32, kSpan = kWidth * GP, kRows = 32 * RB, L = D * RB;
  constexpr int kThreads = kSlices * kWave;
  constexpr int kRing = 4;                    // chunks of rows in LDS, half chunks of weights in registers
  constexpr int kBuf = L * kPlaneBlock;
  constexpr int kDma = 2 * L / kSlices;       // a wavefront's loads of 1 KiB of a chunk's rows
  static_assert(2 * L % kSlices == 0 && (2 * L) % 4 == 0, "every wavefront brings as much; fragment slots repeat");
  // landed<> counts GP loads of weights in each half of a chunk, behind its loads into LDS
  static_assert(kDma + GP <= L, "a half of a chunk has room for its loads of weights");
  constexpr int kLds = kRing * kBuf > turned_bytes(kSpan) ? kRing * kBuf : turned_bytes(kSpan);
  constexpr int kScales = kSlices * 32 * GP;
  __shared__ __attribute__((aligned(16))) unsigned char lds[kLds];
  __shared__ __attribute__((aligned(16))) float scale_s[kScales], bias_s[PAIR ? 4 : kScales];
  __shared__ float step_s[kRows];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, up = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ctile = unit % a.ncols, slice = unit / a.ncols;
  const int m0 = rbk * kRows;
  const int half_groups = a.groups / 2; // PAIR only
  const int glast = PAIR ? half_groups - 1 : a.groups - 1;
  const int g0 = (ctile * kSlices + wave) * (kSpan / 16);
  const int cb = slice * a.chunks_per_slice;
  const int nch = min(a.chunks_per_slice, a.chunks - cb);

  // weights: a base per channel tile, and how far from it this lane's group lies
  const char *wb[GP];
  unsigned woff[GP];
#pragma unroll
  for (int g = 0; g < GP; ++g) {
    const int second = (lane >> 4) & 1, first = min(PAIR ? g0 + g : g0 + 2 * g, glast);
    const int gg = PAIR ? first + second * half_groups : min(g0 + 2 * g + second, glast);
    wb[g] = reinterpret_cast<const char *>(a.W) + ((size_t)first * a.chunks + cb) * 1024;
    woff[g] = (unsigned)(gg - first) * (unsigned)a.chunks * 1024u + (unsigned)(up * 16 + (lane & 15)) * 16u;
  }
  v4i32 wr[kRing][GP];
  auto fetch_w = [&](int c, int half, int g, v4i32 &w) {
    // a scalar base: 64-bit addresses of every lane would take registers there are not
    const uintptr_t at = reinterpret_cast<uintptr_t>(wb[g]) + (size_t)min(c, nch - 1) * 1024 + half * 512;
    const uintptr_t base = (uintptr_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)at) |
                           (uintptr_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(at >> 32)) << 32;
    w = *(const __attribute__((address_space(1))) v4i32 *)((const __attribute__((address_space(1))) char *)base + woff[g]);
  };
  // rows: 1 KiB `i` of this wavefront is rows 16 (j % 2) .. + 15 of layer j / 2, j = 4 i + wave
  const unsigned lds0 = (unsigned)__builtin_amdgcn_readfirstlane(
      (int)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds);
  const unsigned row_off = (unsigned)(lane >> 2) * kTileK + (unsigned)((lane & 3) ^ (lane >> 4)) * 16u;
  const int8_t *rows_at[kDma];
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int j = i * kSlices + wave, l = j / 2;
    const int block = min(m0 / 32 + l / D, a.Mp / 32 - 1);
    rows_at[i] = a.planes + (((size_t)block * a.chunks + cb) * D + l % D) * kPlaneBlock + j % 2 * 1024;
  }
  auto bring = [&](int c, int buf, int i) {
    load_1k_to_lds(rows_at[i] + (size_t)min(c, nch - 1) * (D * kPlaneBlock), row_off,
                   lds0 + buf * kBuf + (i * kSlices + wave) * 1024);
  };
#pragma unroll
  for (int c = 0; c < kRing - 1; ++c)
#pragma unroll
    for (int i = 0; i < kDma; ++i)
      bring(c, c, i);
#pragma unroll
  for (int h = 0; h < kRing - 1; ++h)
#pragma unroll
    for (int g = 0; g < GP; ++g)
      fetch_w(h / 2, h % 2, g, wr[h][g]);
  if (a.slices == 1) {
    const int n0 = ctile * kSlices * kSpan;
    for (int i = tid; i < kScales; i += kThreads) {
      const int mtx = PAIR ? i / (kScales / 2) : 0, n = n0 + (PAIR ? i % (kScales / 2) : i);
      scale_s[i] = n < a.N ? a.scale[(size_t)mtx * a.N + n] : 0.f;
      if constexpr (!PAIR)
        bias_s[i] = a.bias && n < a.N ? a.bias[n] : 0.f;
    }
    for (int i = tid; i < kRows; i += kThreads)
      step_s[i] = m0 + i < a.M ? a.steps[m0 + i] : 0.f;
  }

  v16i32 acc[GP][RB][D];
#pragma unroll
  for (int g = 0; g < GP; ++g)
#pragma unroll
    for (int l = 0; l < L; ++l)
      acc[g][l / D][l % D] = v16i32{};

  landed<(kRing - 1) * GP + kDma>(); // chunks 0 and 1
  __syncthreads();
  const int frag_at[2] = {col * kTileK + (up ^ ((col >> 2) & 3)) * 16,
                          col * kTileK + ((2 + up) ^ ((col >> 2) & 3)) * 16};
  v4i32 frag[4];
  // sub-step u of a chunk: layer u % L, k half u / L
  auto load_frag = [&](int buf, int u, v4i32 &f) {
    f = *reinterpret_cast<const v4i32 *>(lds + buf * kBuf + u % L * kPlaneBlock + frag_at[u / L]);
  };
  load_frag(0, 0, frag[0]);
  load_frag(0, 1, frag[1]);
  // step c = c0 + slot: chunk c in buffer `slot`, chunk c + 3 into the one before it
  auto step = [&](int c0, auto slot) {
    constexpr int sl = slot;
    const int c = c0 + sl;
#pragma unroll
    for (int u = 0; u < 2 * L; ++u) {
      load_frag(u + 2 < 2 * L ? sl : (sl + 1) % kRing, (u + 2) % (2 * L), frag[(u + 2) & 3]);
      const int h = u / L, ahead = h + kRing - 1;
      if (u < kDma)
        bring(c + kRing - 1, (sl + kRing - 1) % kRing, u);
      const int g = u - kDma - h * (L - kDma); // behind those
      if (g >= 0 && g < GP)
        fetch_w(c + ahead / 2, ahead % 2, g, wr[(2 * sl + ahead) % kRing][g]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < GP; ++g)
        acc[g][u % L / D][u % D] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wr[(2 * sl + h) % kRing][g], frag[u & 3],
                                                                         acc[g][u % L / D][u % D], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    landed<4 * GP + kDma>(); // chunk c + 2, issued at the start of step c - 1
    __syncthreads();
  };
  using std::integral_constant;
  int c0 = 0;
  for (; c0 + kRing <= nch; c0 += kRing) {
    step(c0, integral_constant<int, 0>{});
    step(c0, integral_constant<int, 1>{});
    step(c0, integral_constant<int, 2>{});
    step(c0, integral_constant<int, 3>{});
  }
  static_assert(kRing == 4, "a round is written out");
  if (c0 < nch) {
    step(c0, integral_constant<int, 0>{});
    if (c0 + 1 < nch) {
      step(c0, integral_constant<int, 1>{});
      if (c0 + 2 < nch)
        step(c0, integral_constant<int, 2>{});
    }
  }
  landed<0>(); // of the chunks asked for beyond the last: the tile's way out goes through their LDS
  __syncthreads();
  finish_tile<D, RB, GP, PAIR>(a, acc, lds, scale_s, bias_s, step_s, ctile, rbk, slice, g0, m0, wave, lane);
}

// What a wavefront needs before its first fetch arrives in SGPRs (this file is built
// with -amdgpu-kernarg-preload-count); the rest is loaded behind the fetch.
#define BH_I8_LEADING                                                                              \
  const int8_t *planes, const int4 *W, int Mp, int Kp, int groups, int chunks, int ncols,          \
      int slices, int chunks_per_slice, int row_tiles, int panel, GemmI8Args a
#define BH_I8_TAKE                                                                                 \
  a.planes = planes;                                                                               \
  a.W = W;                                                                                         \
  a.Mp = Mp;                                                                                       \
  a.Kp = Kp;                                                                                       \
  a.groups = groups;                                                                               \
  a.chunks = chunks;                                                                               \
  a.ncols = ncols;                                                                                 \
  a.slices = slices;                                                                               \
  a.chunks_per_slice = chunks_per_slice;                                                           \
  a.row_tiles = row_tiles;                                                                         \
  a.panel = panel;

// 32 rows x 128 channels per workgroup; 256 channels; the others of kTiles
template <int D, bool PAIR, bool ROPE = false>
__global__ void __launch_bounds__(kSlices *kWave) gemm_w8_i8_kernel(BH_I8_LEADING) {
  BH_I8_TAKE
  int unit, rbk;
  if (!place_tile(a.ncols * a.slices, a.row_tiles, a.panel, unit, rbk))
    return;
  multiply_tile<D, 1, 1, PAIR, ROPE>(a, unit, rbk);
}
template <int D, bool PAIR, bool ROPE = false>
__global__ void __launch_bounds__(kSlices *kWave, ROPE ? 2 : 1) gemm_w8_i8_wide_kernel(BH_I8_LEADING) {
  BH_I8_TAKE
  int unit, rbk;
  if (!place_tile(a.ncols * a.slices, a.row_tiles, a.panel, unit, rbk))
    return;
  multiply_tile<D, wide_blocks(D), 2, PAIR, ROPE>(a, unit, rbk);
}
template <int D, int RB, int GP, bool PAIR>
__global__ void __launch_bounds__(kSlices *kWave, tall_shares(D, GP) ? 2 : 1)
gemm_w8_i8_tall_kernel(BH_I8_LEADING) {
  BH_I8_TAKE
  int unit, rbk;
  if (!place_tile(a.ncols * a.slices, a.row_tiles, a.panel, unit, rbk))
    return;
  if constexpr (tall_shares(D, GP))
    multiply_block<D, RB, GP, PAIR>(a, unit, rbk);
  else
    multiply_tile<D, RB, GP, PAIR>(a, unit, rbk);
}

// Row tiles of 64 x 256 as far as they make whole rounds of two to a compute unit, the rows behind
// them in tiles of 32 x 128, which start as the last round ends: what a few large tiles of one more
// round would keep a part of the chip on for two thirds of a round, small ones spread over all of it.
// gate | up of three planes, 1536 -> 2 x 8960: 512 rows (560 large tiles for 512 places) 47.3 us, so 44.0;
// prompts of 449, 512, 960 and 1408 tokens 3.6, 1.5, 2.3 and 1.2 % shorter.  (Of two planes, whose tiles
// have more shapes, no prompt was shorter.)
__global__ void __launch_bounds__(kSlices *kWave, 2)
gemm_w8_i8_tailed_kernel(BH_I8_LEADING, int tail_from, int tail_cols) {
  BH_I8_TAKE
  int unit, rbk;
  if ((int)blockIdx.x < tail_from) {
    if (place_tile(a.ncols, a.row_tiles, a.panel, unit, rbk))
      multiply_block<3, 2, 2, true>(a, unit, rbk);
    return;
  }
  const int id = blockIdx.x - tail_from, ids = (tail_cols + 7) & ~7; // a column's tiles on one XCD
  rbk = id / ids;
  unit = id - rbk * ids;
  if (unit >= tail_cols)
    return;
  const int row0 = a.row_tiles * 64;
  a.ncols = tail_cols;
  multiply_tile<3, 1, 1, true>(a, unit, rbk, row0);
}

// ---- few f32 rows as they come -------------------------------------------------------
// The output and down products of a short prompt: up to 128 rows that no kernel before has as
// digits.  A launch that turns them into planes takes 2 to 5 us, most of which is the launch; here
// every workgroup turns its own slice of 32 rows into digits, each row with the step of its largest
// magnitude in the slice, which is never coarser than that of the whole row, and its sums leave
// scaled.  (A NaN or an infinity gives its slice a NaN step and the row's sums with it.)
//
// What bounds it: one trip to memory.  A workgroup takes 32 rows x 128 channels x C chunks of 64 k
// and asks for all of its rows and then all of its weights at once; the digits are made while the
// weights are on their way, and there is one barrier.  27 rows of 8960 -> 1536: 9.8 us, and
// 5.2 + 7.1 as two launches; of 1536 -> 1536 4.3, and 2.8 + 4.3.
template <int D, int C>
__global__ void __launch_bounds__(kSlices *kWave)
gemm_w8_i8_rows_kernel(const float *A, const int4 *W, int lda, int M, int K, int groups, int chunks, int ncols,
                       int slices, float *partial) {
  constexpr int kTurn = turn_floats(32);
  __shared__ __attribute__((aligned(16))) unsigned char planes[C * D * kPlaneBlock];
  __shared__ __attribute__((aligned(16))) float turned[kSlices * 32 * kTurn];
  __shared__ float step_s[32];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, up = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ctile = blockIdx.x, slice = blockIdx.y, m0 = blockIdx.z * 32;
  const int cb = slice * C, nch = min(C, chunks - cb); // chunks of this slice, >= 1

  // eight threads to a row, each with every eighth run of four values
  const int r = tid >> 3, j = tid & 7;
  float v[2 * C][4];
  const float *row = A + (int64_t)min(m0 + r, M - 1) * lda;
  const int k0 = cb * kTileK + j * 4;
#pragma unroll
  for (int i = 0; i < 2 * C; ++i) {
    const float4 q = *reinterpret_cast<const float4 *>(row + min(k0 + i * 32, K - 4));
    v[i][0] = q.x; v[i][1] = q.y; v[i][2] = q.z; v[i][3] = q.w;
  }
  const v4i32 *wp = reinterpret_cast<const v4i32 *>(W) +
                    ((size_t)min((ctile * kSlices + wave) * 2 + ((lane >> 4) & 1), groups - 1) * chunks + cb) * 64 +
                    up * 16 + (lane & 15);
  v4i32 w[C][2];
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      w[c][h] = wp[(size_t)min(c, nch - 1) * 64 + h * 32];
  __builtin_amdgcn_sched_barrier(0); // all of them before the first value is looked at

  // (Values beyond K repeat the row's last ones, and weights are zero there; rows beyond M repeat the
  // last row, and nobody reads their sums.)
  unsigned mb = 0;
#pragma unroll
  for (int i = 0; i < 2 * C; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      mb = max(mb, __float_as_uint(v[i][e]) & 0x7fffffffu);
#pragma unroll
  for (int o = 1; o < 8; o <<= 1)
    mb = max(mb, (unsigned)__shfl_xor((int)mb, o, 64));
  const bool finite = mb < 0x7f800000u;
  const float step = finite ? digit_step(__uint_as_float(mb), D) : __uint_as_float(0x7fc00000u);
  const float inv = finite ? 1.0f / step : 0.f;
  if (j == 0)
    step_s[r] = step;
  // pieces of 16 bytes permuted by the row's number, as in multiply_block
#pragma unroll
  for (int i = 0; i < 2 * C; ++i) {
    unsigned word[3];
    digits_of(v[i], inv, D, word);
    const int k4 = (i & 1) * 8 + j;
    unsigned char *dst = planes + (i / 2) * (D * kPlaneBlock) + r * kTileK + ((k4 >> 2) ^ (r >> 2 & 3)) * 16 + (k4 & 3) * 4;
#pragma unroll
    for (int p = 0; p < D; ++p)
      *reinterpret_cast<unsigned *>(dst + p * kPlaneBlock) = word[p];
  }
  __syncthreads();

  v16i32 acc[D];
#pragma unroll
  for (int p = 0; p < D; ++p)
    acc[p] = v16i32{};
#pragma unroll
  for (int c = 0; c < C; ++c)
    if (c < nch) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int p = 0; p < D; ++p) {
          const v4i32 f = *reinterpret_cast<const v4i32 *>(planes + (c * D + p) * kPlaneBlock + col * kTileK +
                                                           ((2 * h + up) ^ (col >> 2 & 3)) * 16);
          acc[p] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[c][h], f, acc[p], 0, 0, 0);
        }
    }

  // out as finish_tile leaves the sums of a slice, but scaled
  float *tile = turned + wave * (32 * kTurn);
  const float s = step_s[col];
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<float4 *>(tile + col * kTurn + 8 * q + 4 * up) =
        make_float4(combine<D>(acc, 4 * q) * s, combine<D>(acc, 4 * q + 1) * s, combine<D>(acc, 4 * q + 2) * s,
                    combine<D>(acc, 4 * q + 3) * s);
  const size_t at = ((size_t)(blockIdx.z * ncols + ctile) * slices + slice) * kSlices + wave;
  float *part = partial + at * 32 * 32;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int idx = lane + 64 * i, rr = idx / 8, c4 = idx % 8;
    *reinterpret_cast<float4 *>(part + rr * 32 + c4 * 4) =
        *reinterpret_cast<const float4 *>(tile + rr * kTurn + c4 * 4);
  }
}

// Where the sums of row m, channels n.. of the first K slice lie.
template <class Args> // GemmI8Args, SliceSums
__device__ __forceinline__ const float *first_slice(const Args &a, int m, int n) {
  const int tile = m / a.tile_rows * a.ncols + n / (kSlices * a.span), wave = n / a.span % kSlices;
  const size_t row =
      ((size_t)tile * a.slices * kSlices + wave) * a.tile_rows + m % a.tile_rows;
  return a.partial + row * a.span + n % a.span;
}

// Sum of a float4 over the K slices, in slice order, eight loads in flight at a
// time (slices past the end repeat the last one and are not added).
__device__ __forceinline__ void sum_slices(const float *p, size_t slice_stride, int slices,
                                           float (&v)[4]) {
  v[0] = v[1] = v[2] = v[3] = 0.f;
  for (int sl = 0; sl < slices; sl += 8) {
    float4 q[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      q[u] = *reinterpret_cast<const float4 *>(p + (size_t)min(sl + u, slices - 1) * slice_stride);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (sl + u < slices) {
        v[0] += q[u].x; v[1] += q[u].y; v[2] += q[u].z; v[3] += q[u].w;
      }
  }
}

// What finishes four neighbouring outputs: scales, bias and (accumulating) the old
// values, asked for in one go before the slices are summed -- loaded at their
// use, each was an L2 round trip of its own behind the sum.
struct FinishOperands {
  float scale[4], bias[4], old[4];
};
__device__ __forceinline__ FinishOperands load_finish_operands(const GemmI8Args &a, const float *c,
                                                              int n) {
  FinishOperands f;
  load4(a.scale, n, a.N, f.scale);
  f.bias[0] = f.bias[1] = f.bias[2] = f.bias[3] = 0.f;
  f.old[0] = f.old[1] = f.old[2] = f.old[3] = 0.f;
  if (a.bias)
    load4(a.bias, n, a.N, f.bias);
  if (a.accumulate)
    load4(c - n, n, a.N, f.old);
  return f;
}

// C (+)= step[m] * scale[n] * sum over slices of the unscaled sums, slice order (no steps: 1).
__global__ void __launch_bounds__(256)
reduce_slices_kernel(GemmI8Args a) {
  const int n4 = (a.N + 3) / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)a.M * n4)
    return;
  const int m = (int)(i / n4), n = (int)(i % n4) * 4;
  const size_t slice_stride = (size_t)kSlices * a.tile_rows * a.span;
  const float *p = first_slice(a, m, n);
  const float step = a.steps ? a.steps[m] : 1.0f;
  float *c = a.C + (int64_t)m * a.ldc + n;
  const FinishOperands f = load_finish_operands(a, c, n);
  float v[4];
  sum_slices(p, slice_stride, a.slices, v);
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (n + r < a.N) {
      const float o = f.bias[r] + (v[r] * step) * f.scale[r];
      c[r] = a.accumulate ? f.old[r] + o : o;
    }
}

// The same where C is q | k | v and what follows it is the rotation and the cache rows: a
// thread has four channels of a head and their partners 64 further on.
// Its angles are worked out while its loads are on their way (27 rows of 2048 channels: 4.7 us
// and 3.4 in a launch behind it, 5.4 in this one; prompts of 3 to 100 tokens 2 to 5 % shorter).
// Small workgroups: a short prompt's few loads then come in through many compute units.
constexpr int kRopeThreads = 64;
__global__ void __launch_bounds__(kRopeThreads)
reduce_slices_rope_kernel(SliceSums a, RopeKv r, float *C, int64_t ldc, int M) {
  constexpr int kHalf = kAttnHeadDim / 2;
  const int turned = r.heads + r.kv_heads, per_row = (turned + r.kv_heads) * (kHalf / 4);
  const int64_t i = (int64_t)blockIdx.x * kRopeThreads + threadIdx.x;
  if (i >= (int64_t)M * per_row)
    return;
  const int m = (int)(i / per_row), t = (int)(i % per_row), pos = r.start_pos + m;
  const size_t slice_stride = (size_t)kSlices * a.tile_rows * a.span;
  const float step = a.steps ? a.steps[m] : 1.0f;
  float *row = C + (int64_t)m * ldc;
  // a quad's first eight slices and its operands
  struct Quad {
    float4 q[8];
    float scale[4], bias[4];
    const float *p;
  };
  auto request = [&](int n, Quad &x) {
    x.p = first_slice(a, m, n);
    load4(a.scale, n, a.N, x.scale);
    x.bias[0] = x.bias[1] = x.bias[2] = x.bias[3] = 0.f;
    if (a.bias)
      load4(a.bias, n, a.N, x.bias);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      x.q[u] = *reinterpret_cast<const float4 *>(x.p + (size_t)min(u, a.slices - 1) * slice_stride);
  };
  auto finish = [&](Quad &x, float (&v)[4]) {
    v[0] = v[1] = v[2] = v[3] = 0.f;
    for (int sl = 0;;) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (sl + u < a.slices) {
          v[0] += x.q[u].x; v[1] += x.q[u].y; v[2] += x.q[u].z; v[3] += x.q[u].w;
        }
      sl += 8;
      if (sl >= a.slices)
        break;
#pragma unroll
      for (int u = 0; u < 8; ++u)
        x.q[u] = *reinterpret_cast<const float4 *>(x.p + (size_t)min(sl + u, a.slices - 1) * slice_stride);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = x.bias[e] + (v[e] * step) * x.scale[e];
  };
  const int head = t / (kHalf / 4), j = t % (kHalf / 4) * 4, n = head * kAttnHeadDim + j;
  Quad x, y;
  request(n, x);
  request(n + kHalf, y);
  const bool is_v = head >= turned;
  float s[4], c[4], lo[4], hi[4];
  if (!is_v) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      sincosf(r.inv_freq[j + e] * (float)pos, &s[e], &c[e]);
  }
  finish(x, lo);
  finish(y, hi);
  if (is_v) {
    const int kvh = head - turned;
    float *dst = r.vcache + ((int64_t)kvh * r.max_len + pos) * kAttnHeadDim + j;
    *reinterpret_cast<float4 *>(dst) = make_float4(lo[0], lo[1], lo[2], lo[3]);
    *reinterpret_cast<float4 *>(dst + kHalf) = make_float4(hi[0], hi[1], hi[2], hi[3]);
    if (r.terms.tiles) // all sixteen lanes of a head's row
      put_value_terms(r.terms, kvh, pos, j / 4, lo, hi);
    return;
  }
  float nlo[4], nhi[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    nlo[e] = lo[e] * c[e] + (-hi[e]) * s[e];
    nhi[e] = hi[e] * c[e] + lo[e] * s[e];
  }
  float *dst = head < r.heads ? row + n
                              : r.kcache + ((int64_t)(head - r.heads) * r.max_len + pos) * kAttnHeadDim + j;
  *reinterpret_cast<float4 *>(dst) = make_float4(nlo[0], nlo[1], nlo[2], nlo[3]);
  *reinterpret_cast<float4 *>(dst + kHalf) = make_float4(nhi[0], nhi[1], nhi[2], nhi[3]);
  if (r.terms.tiles && head >= r.heads)
    put_key_terms(r.terms, head - r.heads, pos, j / 4, nlo, nhi);
}

// One plane (the w8a8 matmul): the slices hold int32 sums, added exactly; then
// C = f32(sum) * (step * scale[n]) in that order (linalg.py:12833-12845), and the
// sums themselves where the caller asked for them.
__global__ void __launch_bounds__(256)
reduce_slices_i32_kernel(GemmI8Args a) {
  const int n4 = (a.N + 3) / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)a.M * n4)
    return;
  const int m = (int)(i / n4), n = (int)(i % n4) * 4;
  const size_t slice_stride = (size_t)kSlices * a.tile_rows * a.span;
  const float *p = first_slice(a, m, n);
  int v[4] = {0, 0, 0, 0};
  for (int sl = 0; sl < a.slices; sl += 4) {
    v4i32 q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      q[u] = *reinterpret_cast<const v4i32 *>(p + (size_t)min(sl + u, a.slices - 1) * slice_stride);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (sl + u < a.slices) {
        v[0] += q[u][0]; v[1] += q[u][1]; v[2] += q[u][2]; v[3] += q[u][3];
      }
  }
  const float step = a.steps[m];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (n + r < a.N) {
      a.C[(int64_t)m * a.ldc + n + r] = scaled<1>((float)v[r], step, a.scale[n + r]);
      if (a.sums)
        a.sums[(int64_t)m * a.N + n + r] = v[r];
    }
}

// The same, one workgroup per row, which then holds the finished row and goes on
// to write RMSNorm(row) * w as the digit planes of the next matmul's input (what
// rmsnorm_to_digits_kernel would read back from C): lds = [Kp2] norm weights, then cache
// of row_to_digits, then [Kp2] the row.  A thread owns the same quads throughout.
//
// A chain of waits bounds it: everything in memory, the norm weights too, is asked for
// at the start, and the two sums over the row are the only barriers (27 rows
// of 1536: 8.0 -> 6.4 us, 512 rows 9.0 -> 8.0, 1931 rows 23.5 -> 17.6).
__global__ void __launch_bounds__(kRowThreads)
reduce_slices_norm_kernel(const float *p_partial, const float *p_steps, int p_N, int p_ncols,
                          int p_slices, int p_span, int p_tile_rows, GemmI8Args rest,
                          const float *__restrict__ norm_w, float inv_n, float eps, int D,
                          int Mp2, int Kp2, int8_t *__restrict__ planes) {
  GemmI8Args a = rest; // the leading parameters arrive in SGPRs, ahead of the first load
  a.partial = const_cast<float *>(p_partial);
  a.steps = p_steps;
  a.N = p_N;
  a.ncols = p_ncols;
  a.slices = p_slices;
  a.span = p_span;
  a.tile_rows = p_tile_rows;
  __shared__ float red[kRowThreads / 64];
  extern __shared__ __attribute__((aligned(16))) float row_lds[];
  float *xrow = row_lds + Kp2;
  const int m = row_of_workgroup();
  if (m >= rest.M)
    return;
  const int n4 = (a.N + 3) / 4;
  const size_t slice_stride = (size_t)kSlices * a.tile_rows * a.span;
  const float step = a.steps ? a.steps[m] : 1.0f;
  float s = 0.f;
  for (int q4 = threadIdx.x; q4 < n4; q4 += kRowThreads) {
    const int n = q4 * 4;
    const float *p = first_slice(a, m, n);
    float *c = a.C + (int64_t)m * a.ldc + n;
    const FinishOperands f = load_finish_operands(a, c, n);
    float v[4], w[4];
    load4(norm_w, n, a.N, w);
    sum_slices(p, slice_stride, a.slices, v);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[r] = f.bias[r] + (v[r] * step) * f.scale[r];
      if (a.accumulate)
        v[r] += f.old[r];
      if (n + r >= a.N)
        v[r] = 0.f;
      s = fmaf(v[r], v[r], s);
    }
    if (n + 3 < a.N && (reinterpret_cast<uintptr_t>(c) & 15) == 0) {
      *reinterpret_cast<float4 *>(c) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < a.N)
          c[r] = v[r];
    }
    *reinterpret_cast<float4 *>(row_lds + n) = make_float4(w[0], w[1], w[2], w[3]);
    *reinterpret_cast<float4 *>(xrow + n) = make_float4(v[0], v[1], v[2], v[3]);
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = s;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int w = 0; w < kRowThreads / 64; w += 2)
    tot += red[w] + red[w + 1];
  const float rs = 1.0f / sqrtf(tot * inv_n + eps);
  row_to_digits(NormRow{xrow, row_lds, rs, a.N}, a.N, m, D, Mp2, Kp2, planes, red, row_lds);
}

BH_VARIANT_FAMILY(WideFamily, "gemm_w8_i8_wide_kernel");
BH_VARIANT_FAMILY(NarrowFamily, "gemm_w8_i8_kernel");
BH_TILE_FAMILY(NarrowPairFamily, "gemm_w8_i8_kernel pair");
BH_TILE_FAMILY(TallFamily, "gemm_w8_i8_tall_kernel");
BH_TILE_FAMILY(TailedFamily, "gemm_w8_i8_tailed_kernel");
BH_TILE_FAMILY(RotatesFamily, "gemm_w8_i8 rotates"); // planes, channel tiles per wavefront

template <class Kernel>
int launch_tiles(Kernel kernel, const GemmI8Args &a, unsigned blocks, hipStream_t stream) {
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kSlices * kWave), 0, stream, a.planes, a.W, a.Mp,
                     a.Kp, a.groups, a.chunks, a.ncols, a.slices, a.chunks_per_slice,
                     a.row_tiles, a.panel, a);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

template <int D, bool PAIR>
int launch_wide(const GemmI8Args &a, unsigned blocks, hipStream_t stream) {
  BH_NOTE_VARIANT(WideFamily, D, (int)PAIR);
  return launch_tiles(gemm_w8_i8_wide_kernel<D, PAIR>, a, blocks, stream);
}

template <int D, bool PAIR>
int launch_narrow(const GemmI8Args &a, unsigned blocks, hipStream_t stream) {
  if constexpr (PAIR)
    BH_NOTE_VARIANT(NarrowPairFamily, D);
  else
    BH_NOTE_VARIANT(NarrowFamily, D);
  return launch_tiles(gemm_w8_i8_kernel<D, PAIR>, a, blocks, stream);
}

// `blocks` large tiles, as place_tile has them, and the tail
int launch_tailed(const GemmI8Args &a, unsigned blocks, hipStream_t stream) {
  BH_NOTE_VARIANT(TailedFamily, 3);
  const int cols = (int)ceil_div(a.N, kSlices * 16);
  const unsigned tail = (unsigned)round_up(cols, 8) * (unsigned)ceil_div(a.M - 64 * a.row_tiles, 32);
  hipLaunchKernelGGL(gemm_w8_i8_tailed_kernel, dim3(blocks + tail), dim3(kSlices * kWave), 0, stream, a.planes,
                     a.W, a.Mp, a.Kp, a.groups, a.chunks, a.ncols, a.slices, a.chunks_per_slice, a.row_tiles,
                     a.panel, a, (int)blocks, cols);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

template <int D, int RB, int GP, bool PAIR>
int launch_tall(const GemmI8Args &a, unsigned blocks, hipStream_t stream) {
  BH_NOTE_VARIANT(TallFamily, D, RB, GP, (int)PAIR);
  return launch_tiles(gemm_w8_i8_tall_kernel<D, RB, GP, PAIR>, a, blocks, stream);
}

} // namespace

namespace {
size_t row_cache_bytes(int cols_padded) {
  return cols_padded <= kRowCache ? sizeof(float) * (size_t)cols_padded : 0;
}
} // namespace

namespace {
// The rows in registers where they can be read 16 bytes at a time and are not longer; *done stays false
// elsewhere.
template <bool NORM>
int launch_rows_to_digits(const float *A, int64_t lda, const float *w, int64_t M, int64_t K, float eps, int digits,
                          void *staged, bool *done, hipStream_t stream) {
  const GemmStagingLayout l = gemm_staging_layout(M, K);
  const int nv = (int)ceil_div(K, kRowThreads * 4);
  if (K % 4 || lda % 4 || nv > (NORM ? 3 : 7) ||
      ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(w)) & 15) != 0)
    return BUDDY_HIP_OK;
  auto launch = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(row_workgroups(NORM ? M : (int64_t)l.rows_padded)), dim3(threads), 0, stream, A,
                       lda, w, (int)M, (int)K, 1.0f / (float)K, eps, digits, l.rows_padded, l.cols_padded,
                       static_cast<int8_t *>(staged));
  };
  if (nv == 1) // (on 64, 128 and 512 threads 6.6, 6.2 and 7.5 us for 1931 normed rows of 1536, 6.2 so)
    launch(rows_to_digits_kernel<2, NORM, 256>, 256);
  else if (nv == 2)
    launch(rows_to_digits_kernel<2, NORM, 512>, 512);
  else if (nv == 3)
    launch(rows_to_digits_kernel<3, NORM, 512>, 512);
  if constexpr (!NORM) {
    if (nv == 4 || nv == 5) // (on 256 threads 23.6 us for 1931 rows of 8960, 21.6 so)
      launch(rows_to_digits_kernel<5, false, 512>, 512);
    else if (nv >= 6)
      launch(rows_to_digits_kernel<7, false, 512>, 512);
  }
  BH_CHECK_HIP(hipGetLastError());
  *done = true;
  return BUDDY_HIP_OK;
}
} // namespace

int launch_activations_to_digits(const float *A, int64_t lda, int64_t M, int64_t K,
                                 int digits, void *staged, hipStream_t stream) {
  BH_REQUIRE(A && staged && M > 0 && K > 0 && digits >= 2 && digits <= 3 && lda >= K,
             "activations_to_digits: bad argument");
  bool done = false;
  if (int rc = launch_rows_to_digits<false>(A, lda, nullptr, M, K, 0.f, digits, staged, &done, stream))
    return rc;
  if (done)
    return BUDDY_HIP_OK;
  const GemmStagingLayout l = gemm_staging_layout(M, K);
  hipLaunchKernelGGL(activations_to_digits_kernel, dim3((unsigned)l.rows_padded), dim3(kRowThreads),
                     row_cache_bytes(l.cols_padded), stream, A, lda, (int)M, (int)K, digits,
                     l.rows_padded, l.cols_padded, static_cast<int8_t *>(staged));
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

int launch_attn_fold_to_digits(const PromptFold &fold, int64_t o_stride, int heads, int tokens,
                               int digits, void *staged, hipStream_t stream) {
  const int64_t K = (int64_t)heads * kPromptD;
  BH_REQUIRE(fold.blocks && staged && tokens > 0 && (digits == 2 || digits == 3),
             "attn_fold_to_digits: bad argument");
  const GemmStagingLayout l = gemm_staging_layout(tokens, K);
  hipLaunchKernelGGL(tokens > kFoldTokens ? attn_fold_to_digits_kernel<4> : attn_fold_to_digits_kernel<16>,
                     dim3((unsigned)l.rows_padded), dim3(kRowThreads),
                     row_cache_bytes(l.cols_padded), stream, fold, o_stride, tokens, (int)K, digits,
                     l.rows_padded, l.cols_padded, static_cast<int8_t *>(staged));
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

int launch_rmsnorm_to_digits(const float *x, int64_t ldx, const float *w, int rows, int n,
                             float eps, int digits, void *staged, hipStream_t stream) {
  BH_REQUIRE(x && w && staged && rows > 0 && n > 0 && ldx >= n && digits >= 2 && digits <= 3,
             "rmsnorm_to_digits: bad argument");
  bool done = false;
  if (int rc = launch_rows_to_digits<true>(x, ldx, w, rows, n, eps, digits, staged, &done, stream))
    return rc;
  if (done)
    return BUDDY_HIP_OK;
  const GemmStagingLayout l = gemm_staging_layout(rows, n);
  hipLaunchKernelGGL(rmsnorm_to_digits_kernel, dim3(rows), dim3(kRowThreads),
                     row_cache_bytes(l.cols_padded), stream, x, ldx, w, n,
                     1.0f / (float)n, eps, digits, l.rows_padded, l.cols_padded,
                     static_cast<int8_t *>(staged));
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

int launch_silu_mul_to_digits(const float *g, const float *u, int64_t ld, int rows, int n,
                              int digits, void *staged, hipStream_t stream) {
  BH_REQUIRE(g && u && staged && rows > 0 && n > 0 && ld >= n && digits >= 2 && digits <= 3,
             "silu_mul_to_digits: bad argument");
  const GemmStagingLayout l = gemm_staging_layout(rows, n);
  hipLaunchKernelGGL(silu_mul_to_digits_kernel, dim3(rows), dim3(kRowThreads),
                     row_cache_bytes(l.cols_padded), stream, g, u, ld, n,
                     digits, l.rows_padded, l.cols_padded, static_cast<int8_t *>(staged));
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

namespace {

// Split-K workspace: one grow-only device buffer per stream (calls on one stream
// are ordered; calls on different streams must not share it).
struct Workspace {
  char *ptr = nullptr;
  size_t bytes = 0;
  bool recorded = false;    // a capture was given ptr
  std::vector<char *> held; // outgrown ones that captures were given
};
std::mutex g_workspace_mutex;
std::map<hipStream_t, Workspace> g_workspace;

bool captures(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return status != hipStreamCaptureStatusNone;
}

} // namespace

int gemm_slices_workspace(hipStream_t stream, size_t bytes, char **out) {
  std::lock_guard<std::mutex> lock(g_workspace_mutex);
  Workspace &w = g_workspace[stream];
  const bool capturing = captures(stream);
  *out = nullptr;
  if (w.bytes < bytes) {
    if (capturing)
      return BUDDY_HIP_OK;
    if (w.ptr && w.recorded) {
      // a graph may hold it; at least twice as much next, so that all that are held
      // together stay below the one in use
      bytes = std::max(bytes, 2 * w.bytes);
      w.held.push_back(w.ptr);
    } else if (w.ptr) {
      BH_CHECK_HIP(hipStreamSynchronize(stream)); // an earlier matmul may still use it
      BH_CHECK_HIP(hipFree(w.ptr));
    }
    w.ptr = nullptr;
    w.bytes = 0;
    w.recorded = false;
    BH_CHECK_HIP(hipMalloc(reinterpret_cast<void **>(&w.ptr), bytes));
    w.bytes = bytes;
  }
  w.recorded |= capturing;
  *out = w.ptr;
  return BUDDY_HIP_OK;
}

namespace {

// Tile and K slices for a launch, by an estimate of its time in microseconds.  An XCD (32
// compute units) works on 64 workgroups at a time, two to a compute unit, or on 32 where a
// tile's registers leave room for one.  A chunk of 64 k takes a workgroup that has its
// compute unit to itself `alone`, two that share one `both`, each beside a fixed part; a last
// round that fills less than half runs at the former.  Fitted to
// launches of 27 to 1931 rows of 1536, 4096, 8960 and 14336 k, every tile with every K split: over
// 120 such products, conversion and slices included, the picks are 0.4 (three planes) and 0.9 % (two)
// off the best on average.
// Microseconds of a product with three planes in a prompt (in brackets with tiles of 64 x 256 that
// fill a compute unit alone, which then were the pick for down at 512 rows only):
//   gate | up, 1536 -> 2 x 8960: 27 rows 12.4, 512: 47.3 [52.4] (44.0 with a tail), 1931: 146 [164]
//   down, 8960 -> 1536: 27 rows 5.7, 512: 24.7 [24.9], 1931: 71.5 [78.5]
//   q|k|v, 1536 -> 2048: 512 rows 11.6
//   one plane, 1536 -> 8960: 512 rows 19.1
// (gate | up of 28 rows with weights from memory: two channel tiles 15.4, one 11.4, for which twice
// the compute units ask.)
// 64 x 256 and 96 x 256 use an operand more often: long sums and many rows; 32 x 640: row counts for
// which it comes to a whole round and the others to a little more than one.
struct TileShape {
  int rb, gp;           // blocks of 32 rows; tiles of 32 channels per wavefront
  bool shares;          // two workgroups to a compute unit
  double alone, alone0; // us per chunk and beside that
  double both, both0;
};
constexpr TileShape kTiles1[] = {{1, 1, true, 0.21, 4.5, 0.285, 4.5},
                                 {wide_blocks(1), 2, true, 0.33, 5.0, 0.54, 4.0},
                                 {3, 2, true, 0.39, 5.0, 0.66, 4.0}};
constexpr TileShape kTiles2[] = {{1, 1, true, 0.194, 4.15, 0.379, 3.85},
                                 {wide_blocks(2), 2, true, 0.303, 5.0, 0.51, 6.05},
                                 {2, 2, true, 0.493, 6.2, 0.969, 2.28},
                                 {1, 3, true, 0.428, 6.0, 0.913, 10.0},
                                 {3, 2, true, 0.656, 5.56, 1.259, 3.1}};
constexpr TileShape kTiles3[] = {{1, 1, true, 0.216, 3.2, 0.455, 4.5},
                                 {wide_blocks(3), 2, true, 0.35, 4.7, 0.676, 4.0},
                                 {2, 2, true, 0.546, 5.29, 1.002, 6.81},
                                 {1, 5, false, 0.855, 7.0, 0, 0}};

struct TilePlan {
  int rb = 0, gp = 0, slices = 1;
  int tail = 0; // row tiles in front of a tail of small ones (gemm_w8_i8_tailed_kernel)
  double us = 0;
};
template <int D, bool PAIR>
TilePlan plan_tiles(int64_t M, int64_t channels, int chunks, bool may_split, double norm_us,
                    double split_norm_us, int64_t sum_wgs) {
  TilePlan best;
  const bool in_reach = !PAIR || pair_in_reach(channels, chunks);
  auto consider = [&](const TileShape &t) {
    const bool brings = tall_shares(D, t.gp) && t.rb != wide_blocks(D); // multiply_block
    if (!in_reach && brings)
      return;
    const int64_t ncols = ceil_div(channels, kSlices * t.gp * (PAIR ? 16 : 32));
    const int64_t rows = ceil_div(M, 32 * t.rb);
    for (int s = 1; s <= (may_split ? 16 : 1); ++s) {
      const int64_t per_xcd = ceil_div(ncols * s * rows, 8);
      if (s > 1 && per_xcd > 256)
        break;
      const int64_t cps = ceil_div(chunks, s);
      if (ceil_div(chunks, cps) != s)
        continue; // the last slice would be empty
      const double store = s > 1 ? 2.0 : 0.0; // of the partial sums
      // (With three planes, one that brings its rows and has K whole takes 2 us more in prompts than in a row
      // of its own kind, where nothing beside it hides its way in and out.  o of Qwen2-1.5B at 1931 rows 27.4
      // us, and 25.0 on 32 x 256 tiles; prompts of 1100 to 2000 tokens 0.4 to 1.3 % shorter with those.)
      const double alone_us =
          t.alone * (double)cps + t.alone0 + store + (!PAIR && s == 1 && D == 3 && brings ? 2.0 : 0.0);
      double us;
      if (t.shares) {
        const double both_us = t.both * (double)cps + t.both0 + store;
        const int64_t left = per_xcd % 64;
        us = (double)(per_xcd / 64) * both_us + (left == 0 ? 0.0 : left <= 32 ? alone_us : both_us);
      } else {
        us = (double)ceil_div(per_xcd, 32) * alone_us;
      }
      if (s > 1) // the kernel that adds the slices: 3 us and its bytes
        us += 3.0 + 4.0 * (double)(M * s) * (double)(ncols * 128 * t.gp) / 4e6 +
              0.002 * (double)sum_wgs + split_norm_us;
      else
        us += norm_us;
      if (!best.gp || us < best.us - 1e-9)
        best = {t.rb, t.gp, s, 0, us};
    }
  };
  if constexpr (D == 1)
    for (const TileShape &t : kTiles1)
      consider(t);
  else if constexpr (D == 2)
    for (const TileShape &t : kTiles2)
      consider(t);
  else
    for (const TileShape &t : kTiles3)
      consider(t);
  if constexpr (D == 3 && PAIR) {
    // Whole rounds of 64 x 256, then small tiles: alone on their compute units and 4.5 us beside (each
    // begins with two trips to memory), more from 30 on an XCD on.  512 rows of gate | up have 32 and
    // 44.0 us (47.3), 1931 rows 50 and 2 us more than with large tiles only.
    const TileShape &t = kTiles3[2], &small = kTiles3[0];
    const int64_t ncols = ceil_div(channels, kSlices * 16 * t.gp), rows = ceil_div(M, 32 * t.rb);
    const int64_t rounds = ncols * rows / 512, large = rounds ? std::min(512 * rounds / ncols, rows - 1) : 0;
    if (large > 0 && in_reach) {
      const int64_t tail = ceil_div(channels, kSlices * 16) * ceil_div(M - 32 * t.rb * large, 32);
      const double beside = (double)(tail - (512 * rounds - ncols * large)) / 8;
      const double us = (double)rounds * (t.both * chunks + t.both0) + small.alone * chunks + small.alone0 + 4.5 +
                        0.35 * std::max(0.0, beside - 30) + norm_us;
      if (beside <= 64 && us < best.us)
        best = {t.rb, t.gp, 1, (int)large, us};
    }
  }
  return best;
}

// Whether the product rotates q | k | v itself: tiles of 32 rows and whole heads with K whole.
bool rotates(const TilePlan &plan, const GemmI8Args &a) {
  return a.rope.turns && plan.slices == 1 && !plan.tail && plan.rb == 1 && plan.gp <= 2;
}

// a.partial stays null where K was to be split and no workspace could be had: the caller
// comes back with a plan that leaves K whole.
template <int D, bool PAIR>
int launch_plan(const TilePlan &plan, GemmI8Args &a, hipStream_t stream) {
  a.ncols = (int)ceil_div(a.N, kSlices * (PAIR ? 16 : 32) * plan.gp);
  a.tile_rows = 32 * plan.rb;
  a.span = 32 * plan.gp;
  a.row_tiles = (int)ceil_div(a.M, a.tile_rows);
  a.slices = plan.slices;
  a.chunks_per_slice = (int)ceil_div(a.chunks, plan.slices);
  if (plan.slices > 1) {
    const size_t tile_floats = (size_t)a.tile_rows * kSlices * a.span;
    const size_t bytes = sizeof(float) * tile_floats * plan.slices * (size_t)a.ncols * a.row_tiles;
    char *ws = nullptr;
    if (int rc = gemm_slices_workspace(stream, bytes, &ws))
      return rc;
    if (!ws)
      return BUDDY_HIP_OK;
    a.partial = reinterpret_cast<float *>(ws);
  }
  if (plan.tail)
    a.row_tiles = plan.tail;
  const int64_t units = (int64_t)a.ncols * a.slices;
  a.panel = panel_for(units, a.row_tiles, D > 1);
  const int64_t tiles = (a.panel ? units : round_up(units, 8)) * a.row_tiles;
  BH_REQUIRE(tiles < (1u << 31), "gemm_w8: %lld tiles", (long long)tiles);
  const unsigned blocks = (unsigned)tiles;
  if constexpr (D > 1 && !PAIR) {
    if (rotates(plan, a)) {
      if (plan.gp == 1) {
        BH_NOTE_VARIANT(RotatesFamily, D, 1);
        return launch_tiles(gemm_w8_i8_kernel<D, false, true>, a, blocks, stream);
      }
      BH_NOTE_VARIANT(RotatesFamily, D, 2);
      return launch_tiles(gemm_w8_i8_wide_kernel<D, false, true>, a, blocks, stream);
    }
  }
  if (plan.tail)
    return launch_tailed(a, blocks, stream);
  if (plan.gp == 1)
    return launch_narrow<D, PAIR>(a, blocks, stream);
  if (plan.gp == 2 && plan.rb == wide_blocks(D))
    return launch_wide<D, PAIR>(a, blocks, stream);
  if constexpr (D == 3) {
    if (plan.gp == 2)
      return launch_tall<D, 2, 2, PAIR>(a, blocks, stream);
    return launch_tall<D, 1, 5, PAIR>(a, blocks, stream);
  } else if constexpr (D == 2) {
    if (plan.gp == 3)
      return launch_tall<D, 1, 3, PAIR>(a, blocks, stream);
    if (plan.rb == 2)
      return launch_tall<D, 2, 2, PAIR>(a, blocks, stream);
    return launch_tall<D, 3, 2, PAIR>(a, blocks, stream);
  } else {
    return launch_tall<D, 3, 2, PAIR>(a, blocks, stream);
  }
}

} // namespace

void release_gemm_i8_workspace(hipStream_t stream) {
  std::lock_guard<std::mutex> lock(g_workspace_mutex);
  auto it = g_workspace.find(stream);
  if (it == g_workspace.end())
    return;
  Workspace &w = it->second;
  if (w.ptr || !w.held.empty())
    (void)hipStreamSynchronize(stream);
  if (w.ptr)
    (void)hipFree(w.ptr);
  for (char *p : w.held)
    (void)hipFree(p);
  g_workspace.erase(it);
}

BH_TILE_FAMILY(SlicesRopeFamily, "reduce_slices_rope_kernel"); // trips for eight slices: one, more

int launch_slices_rope(const SliceSums &sums, const RopeKv &r, float *C, int64_t ldc, int M,
                       hipStream_t stream) {
  if (sums.slices <= 8)
    BH_NOTE_VARIANT(SlicesRopeFamily, 1);
  else
    BH_NOTE_VARIANT(SlicesRopeFamily, 2);
  const int64_t quads = (int64_t)M * (r.heads + 2 * r.kv_heads) * (kAttnHeadDim / 8);
  hipLaunchKernelGGL(reduce_slices_rope_kernel, dim3((unsigned)ceil_div(quads, kRopeThreads)),
                     dim3(kRopeThreads), 0, stream, sums, r, C, ldc, M);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

// `planes` holds the digit planes and row steps of the activations (written by
// one of the producers above for exactly this M, K and digit count).
namespace {
// The RMSNorm of the finished rows into digit planes, or the rotation of q | k | v, where the caller
// asked for it and no kernel of the matmul holds whole rows.
int norm_behind(const GemmW8Args &in, hipStream_t stream) {
  if (in.then_rope) {
    const RopeKv &r = *in.then_rope;
    return launch_rope_kv_write(in.C, in.ldc, r, (int)in.M, stream);
  }
  if (!in.then_norm_w)
    return BUDDY_HIP_OK;
  return launch_rmsnorm_to_digits(in.C, in.ldc, in.then_norm_w, (int)in.M, (int)in.N,
                                  in.then_norm_eps, in.digits, in.then_norm_staged, stream);
}

// What follows a product whose K is in slices: their sum, and what the caller wants behind it.
int add_slices(const GemmW8Args &in, const GemmI8Args &a, hipStream_t stream) {
  const GemmStagingLayout next = gemm_staging_layout(in.M, in.N);
  if (in.then_norm_w && next.cols_padded <= kRowCache) {
    // the kernel that adds the slices holds whole rows: it writes the planes too
    const size_t row_lds = 2 * sizeof(float) * (size_t)next.cols_padded;
    if (row_lds > 48 * 1024) { // up to 96 KiB at kRowCache columns
      static DynLdsOnce dyn_lds;
      BH_CHECK_HIP(ensure_dyn_lds(dyn_lds,
                                  reinterpret_cast<const void *>(reduce_slices_norm_kernel),
                                  (int)(2 * sizeof(float) * kRowCache)));
    }
    hipLaunchKernelGGL(reduce_slices_norm_kernel, dim3(row_workgroups(a.M)), dim3(kRowThreads),
                       row_lds, stream, a.partial, a.steps, a.N, a.ncols, a.slices, a.span,
                       a.tile_rows, a, in.then_norm_w, 1.0f / (float)in.N, in.then_norm_eps,
                       in.digits, next.rows_padded, next.cols_padded,
                       static_cast<int8_t *>(in.then_norm_staged));
    BH_CHECK_HIP(hipGetLastError());
    return BUDDY_HIP_OK;
  }
  if (in.then_rope)
    return launch_slices_rope({a.partial, a.steps, a.scale, a.bias, a.slices, a.span, a.tile_rows, a.ncols, a.N},
                              *in.then_rope, a.C, a.ldc, a.M, stream);
  const int64_t threads = (int64_t)a.M * ((a.N + 3) / 4);
  hipLaunchKernelGGL(reduce_slices_kernel, dim3((unsigned)ceil_div(threads, 256)), dim3(256), 0,
                     stream, a);
  BH_CHECK_HIP(hipGetLastError());
  return norm_behind(in, stream);
}

template <int D>
int launch_gemm_w8_digits_d(const GemmW8Args &in, const void *planes, hipStream_t stream) {
  GemmI8Args a;
  const GemmStagingLayout layout = gemm_staging_layout(in.M, in.K);
  a.Mp = layout.rows_padded;
  a.Kp = layout.cols_padded;
  a.planes = static_cast<const int8_t *>(planes);
  a.steps = reinterpret_cast<const float *>(a.planes + (size_t)in.digits * a.Mp * a.Kp);
  a.W = reinterpret_cast<const int4 *>(in.W);
  a.scale = in.scale;
  a.bias = in.bias;
  a.C = in.C;
  a.ldc = in.ldc;
  a.M = (int)in.M;
  a.N = (int)in.N;
  a.groups = (int)ceil_div(in.N, kTileN);
  a.chunks = (int)ceil_div(in.K, kTileK);
  a.accumulate = in.accumulate ? 1 : 0;
  a.partial = nullptr;
  a.sums = nullptr;
  a.int_partials = 0;
  a.slices = 1;
  if (in.silu_pair) {
    // two matrices of N / 2 channels, result SiLU(first) * second: whole K per workgroup
    BH_REQUIRE(!in.then_norm_w, "gemm_w8: no norm after the SiLU pair");
    BH_REQUIRE(in.N % (2 * kTileN) == 0 && !in.accumulate && !in.bias,
               "gemm_w8: the SiLU pair needs two matrices of a multiple of 16 channels, no "
               "bias, no accumulation");
    a.N = (int)(in.N / 2);
    return launch_plan<D, true>(plan_tiles<D, true>(in.M, a.N, a.chunks, false, 0.0, 0.0, 0), a, stream);
  }
  if (in.then_rope && in.then_rope->turns && !in.accumulate && in.ldc % 4 == 0 &&
      in.N == (int64_t)(in.then_rope->heads + 2 * in.then_rope->kv_heads) * kAttnHeadDim &&
      ((reinterpret_cast<uintptr_t>(in.C) | reinterpret_cast<uintptr_t>(in.then_rope->turns) |
        reinterpret_cast<uintptr_t>(in.then_rope->kcache) | reinterpret_cast<uintptr_t>(in.then_rope->vcache)) & 15) == 0)
    a.rope = *in.then_rope;
  // A norm that is to follow (then_norm_w) costs a launch of its own, about
  // 5 us, unless the kernel that adds K slices writes its planes (it holds whole
  // rows, up to kRowCache columns).
  const bool slices_fuse_norm = gemm_staging_layout(in.M, in.N).cols_padded <= kRowCache;
  // The rotation behind q | k | v likewise: 4 us, in the kernel that adds slices 0.5 and what the
  // angles take, which every head works out for itself there.  In the product itself (see `rotates`) it
  // takes one or two; what is said here is where prompts become shorter with K whole (three planes, 64 tokens
  // 1771 and 1765 us, 128 2157 and 2120, 160 2321 and 2242; two, 128 2057 and 1985).
  const double turn_us = !a.rope.turns ? 4.0 : D == 3 ? 2.9 : 3.3;
  const double norm_us = in.then_norm_w ? 5.0 : in.then_rope ? turn_us : 0.0;
  const double split_norm_us = in.then_rope ? 0.5 + 0.004 * (double)in.M : slices_fuse_norm ? 0.0 : norm_us;
  TilePlan plan = plan_tiles<D, false>(in.M, in.N, a.chunks, true, norm_us, split_norm_us, 0);
  if (int rc = launch_plan<D, false>(plan, a, stream))
    return rc;
  if (plan.slices > 1 && !a.partial) {
    plan = plan_tiles<D, false>(in.M, in.N, a.chunks, false, norm_us, 0.0, 0);
    if (int rc = launch_plan<D, false>(plan, a, stream))
      return rc;
  }
  if (plan.slices == 1)
    return rotates(plan, a) ? BUDDY_HIP_OK : norm_behind(in, stream);
  return add_slices(in, a, stream);
}
} // namespace

int launch_gemm_w8_digits(const GemmW8Args &in, const void *planes, hipStream_t stream) {
  return in.digits == 2 ? launch_gemm_w8_digits_d<2>(in, planes, stream)
                        : launch_gemm_w8_digits_d<3>(in, planes, stream);
}

namespace {
BH_TILE_FAMILY(RowsFamily, "gemm_w8_i8_rows_kernel"); // planes, chunks of a slice

// Chunks of 64 k to a slice: the fewest that leave at most sixteen slices, whose sums have to be
// added, and at most a workgroup per compute unit, whose loads are one trip; 0: no such cut.
// (8960 -> 1536 has one up to 64 rows, 1536 -> 1536 up to 128.)  Rows are read 16 bytes at a time.
// Beyond 128 (three planes: 129 rows 2426 -> 2335 us a prompt, 256 the same; two: 180 rows 1 % longer) a
// launch for the digits is a small part.
int rows_chunks(int64_t M, int64_t K, int64_t N, int64_t lda) {
  if (M > 128 || ((K | lda) & 3) != 0 || lda >= (1 << 30))
    return 0;
  const int64_t chunks = ceil_div(K, kTileK), tiles = ceil_div(N, kSlices * 32) * ceil_div(M, 32);
  for (int c : {2, 3, 5, 9, 14})
    if (ceil_div(chunks, c) <= 16 && ceil_div(chunks, c) * tiles <= 256)
      return c;
  return 0;
}

template <int D, int C> int launch_rows(const GemmW8Args &in, const GemmI8Args &a, hipStream_t stream) {
  BH_NOTE_VARIANT(RowsFamily, D, C);
  hipLaunchKernelGGL((gemm_w8_i8_rows_kernel<D, C>), dim3(a.ncols, a.slices, a.row_tiles), dim3(kSlices * kWave), 0,
                     stream, in.A, a.W, (int)in.lda, a.M, (int)in.K, a.groups, a.chunks, a.ncols, a.slices, a.partial);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}
template <int D> int launch_rows_of(int c, const GemmW8Args &in, const GemmI8Args &a, hipStream_t stream) {
  switch (c) {
  case 2:
    return launch_rows<D, 2>(in, a, stream);
  case 3:
    return launch_rows<D, 3>(in, a, stream);
  case 5:
    return launch_rows<D, 5>(in, a, stream);
  case 9:
    return launch_rows<D, 9>(in, a, stream);
  default:
    return launch_rows<D, 14>(in, a, stream);
  }
}
} // namespace

bool gemm_w8_takes_rows(int64_t M, int64_t K, int64_t N, int64_t lda) { return rows_chunks(M, K, N, lda) != 0; }

int launch_gemm_w8_digits_rows(const GemmW8Args &in, bool *done, hipStream_t stream) {
  *done = false;
  BH_REQUIRE(in.A && in.W && in.scale && in.C && in.M > 0 && in.K > 0 && in.N > 0 && in.lda >= in.K && in.ldc >= in.N &&
                 (in.digits == 2 || in.digits == 3) && !in.staged && !in.silu_pair && !in.then_rope,
             "gemm_w8: rows as they come");
  const int c = (reinterpret_cast<uintptr_t>(in.A) & 15) == 0 ? rows_chunks(in.M, in.K, in.N, in.lda) : 0;
  if (!c)
    return BUDDY_HIP_OK;
  GemmI8Args a{};
  a.W = reinterpret_cast<const int4 *>(in.W);
  a.scale = in.scale;
  a.bias = in.bias;
  a.C = in.C;
  a.ldc = in.ldc;
  a.M = (int)in.M;
  a.N = (int)in.N;
  a.groups = (int)ceil_div(in.N, kTileN);
  a.chunks = (int)ceil_div(in.K, kTileK);
  a.accumulate = in.accumulate ? 1 : 0;
  a.ncols = (int)ceil_div(in.N, kSlices * 32);
  a.row_tiles = (int)ceil_div(in.M, 32);
  a.tile_rows = a.span = 32;
  a.chunks_per_slice = c;
  a.slices = (int)ceil_div(a.chunks, c);
  const size_t bytes = sizeof(float) * 32 * kSlices * 32 * (size_t)a.slices * a.ncols * a.row_tiles;
  char *ws = nullptr;
  if (int rc = gemm_slices_workspace(stream, bytes, &ws))
    return rc;
  if (!ws) // under capture, and none of this size
    return BUDDY_HIP_OK;
  a.partial = reinterpret_cast<float *>(ws);
  if (int rc = in.digits == 2 ? launch_rows_of<2>(c, in, a, stream) : launch_rows_of<3>(c, in, a, stream))
    return rc;
  *done = true;
  return add_slices(in, a, stream);
}

// The w8a8 matmul for more than 16 rows: `plane` holds the int8 activations as
// one plane ([rows_padded][cols_padded], zero padded) followed by the row steps,
// every one of them the per-tensor activation scale.  The int32 sums are exact
// whether K stays within one workgroup or is split over several (K <= 2^17:
// 2^17 * 127 * 128 is below 2^31).
int launch_gemm_w8a8_plane(const void *plane, const int8_t *W, const float *wscale, float *C,
                           int32_t *sums, int64_t M, int64_t K, int64_t N,
                           hipStream_t stream) {
  BH_REQUIRE(K <= (1 << 17), "w8a8 matmul: K=%lld above 131072", (long long)K);
  GemmI8Args a;
  const GemmStagingLayout layout = gemm_staging_layout(M, K);
  a.Mp = layout.rows_padded;
  a.Kp = layout.cols_padded;
  a.planes = static_cast<const int8_t *>(plane);
  a.steps = reinterpret_cast<const float *>(a.planes + (size_t)a.Mp * a.Kp);
  a.W = reinterpret_cast<const int4 *>(W);
  a.scale = wscale;
  a.bias = nullptr;
  a.C = C;
  a.ldc = N;
  a.M = (int)M;
  a.N = (int)N;
  a.groups = (int)ceil_div(N, kTileN);
  a.chunks = (int)ceil_div(K, kTileK);
  a.accumulate = 0;
  a.partial = nullptr;
  a.sums = sums;
  a.int_partials = 0;
  // the cost model of the digit-plane launch with one plane; K slices leave int32
  // sums in the workspace (f32 ones would round above 2^24) and a second kernel
  // adds them exactly
  const int64_t reduce_wgs = ceil_div(M * ceil_div(N, 4), 256);
  TilePlan plan = plan_tiles<1, false>(M, N, a.chunks, true, 0.0, 0.0, reduce_wgs);
  a.int_partials = plan.slices > 1;
  if (int rc = launch_plan<1, false>(plan, a, stream))
    return rc;
  if (plan.slices > 1 && !a.partial) {
    plan = plan_tiles<1, false>(M, N, a.chunks, false, 0.0, 0.0, reduce_wgs);
    a.int_partials = 0;
    if (int rc = launch_plan<1, false>(plan, a, stream))
      return rc;
  }
  if (plan.slices > 1) {
    hipLaunchKernelGGL(reduce_slices_i32_kernel, dim3((unsigned)reduce_wgs), dim3(256), 0, stream,
                       a);
    BH_CHECK_HIP(hipGetLastError());
  }
  return BUDDY_HIP_OK;
}

} // namespace bh

extern "C" int buddy_hip_gemm_w8_digits_plan(int64_t M, int64_t K, int64_t N, unsigned flags,
                                             buddy_hip_digits_plan *out) try {
  BH_REQUIRE(out, "gemm_w8_digits_plan: null result");
  BH_REQUIRE(M > 0 && N > 0 && K > 0 && M < (1 << 24) && N < (1 << 24) && K <= (1 << 17),
             "gemm_w8_digits_plan: bad shape M=%lld K=%lld N=%lld", (long long)M, (long long)K, (long long)N);
  const bool pair = flags & BUDDY_HIP_GEMM_SILU_PAIR, two = flags & BUDDY_HIP_GEMM_TWO_DIGITS;
  const int chunks = (int)bh::ceil_div(K, bh::kTileK);
  const bh::TilePlan p = pair ? two ? bh::plan_tiles<2, true>(M, N, chunks, false, 0, 0, 0)
                                    : bh::plan_tiles<3, true>(M, N, chunks, false, 0, 0, 0)
                              : two ? bh::plan_tiles<2, false>(M, N, chunks, true, 0, 0, 0)
                                    : bh::plan_tiles<3, false>(M, N, chunks, true, 0, 0, 0);
  *out = {p.rb, p.gp, p.slices, p.tail};
  return BUDDY_HIP_OK;
} BH_CATCH_INT("buddy_hip_gemm_w8_digits_plan")
