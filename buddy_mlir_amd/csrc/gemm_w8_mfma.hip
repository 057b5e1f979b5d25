// gemm_w8_mfma.hip -- prefill matmul: C[M,N] (+)= A[M,K] . (int8 W[K,N] * scale)
// on the bf16 matrix cores.
//
// Replaces the BLIS-style kernel with dequantisation fused into B packing that
// midend/lib/Conversion/MatMulOptimization/MatMulBlisVectorization.cpp:351-360,
// 398-986 generates for M > 1.
//
// Shape of the kernel:
//  * the weights are read from the same wave-tile packed copy the decode GEMV
//    streams (one resident copy serves prefill and decode).  A lane takes the runs of 16
//    k of one channel that make up its operands of v_mfma_f32_32x32x16_bf16 (32 channels
//    = two tiles): they go from global memory to registers, are converted to bf16
//    (|q| <= 128 is exact) and fed to the matrix core.  No LDS on the way;
//  * the activations are converted once per call to bf16 terms (one term =
//    "activations cast to bf16"; three terms carry all 24 significand bits of
//    the f32 input) in a [term][row][k] buffer, whose rows the wavefronts of a
//    workgroup share through LDS;
//  * workgroups take 32 or 64 rows x 128 or 256 channels, and K is split over
//    several of them where a matrix is too narrow to fill the chip;
//  * workgroup ids are laid out so that the row tiles of one column tile run
//    on the same XCD and share the weight tiles in its L2 (tile_place.h);
//  * the per-channel scale is applied once to the f32 accumulators, where the
//    reference multiplies every element before the FMA.
#include "attn.h"
#include "attn_fold.h"
#include "gemm.h"
#include "tile_place.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>

namespace bh {
namespace {

constexpr int kWaves = 4; // wavefronts per workgroup

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned short u16;
typedef int v4i32 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ u16 bf16_rne(float x) {
  unsigned u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (u16)(u >> 16);
}
__device__ __forceinline__ float bf16_to_f32(u16 b) {
  return __uint_as_float((unsigned)b << 16);
}
__device__ __forceinline__ unsigned pack2(u16 lo, u16 hi) {
  return (unsigned)lo | ((unsigned)hi << 16);
}
// two int8 (bytes j, j+1 of v) -> two exact bf16
__device__ __forceinline__ unsigned q2_to_bf16x2(int v, int j) {
  const float a = (float)(signed char)(v >> (8 * j));
  const float b = (float)(signed char)(v >> (8 * j + 8));
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ bf16x8 frag_from(int lo, int hi) {
  union {
    uint4 u;
    bf16x8 v;
  } x;
  x.u = make_uint4(q2_to_bf16x2(lo, 0), q2_to_bf16x2(lo, 2), q2_to_bf16x2(hi, 0),
                   q2_to_bf16x2(hi, 2));
  return x.v;
}
// A[M, K] f32 -> terms x [Mp, Kp] bf16, zero padded; term t holds the bf16
// rounding of what the terms before it left over.
__global__ void __launch_bounds__(256)
activations_to_bf16(const float *__restrict__ A, int64_t lda, int M, int K, int Mp,
                    int Kp, int terms, u16 *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; // 8 k per thread
  const int kq = Kp / 8;
  if (i >= (int64_t)Mp * kq)
    return;
  const int m = (int)(i / kq), k0 = (int)(i % kq) * 8;
  float r[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    r[e] = (m < M && k0 + e < K) ? A[(int64_t)m * lda + k0 + e] : 0.f;
  for (int t = 0; t < terms; ++t) {
    u16 h[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      h[e] = bf16_rne(r[e]);
      r[e] -= bf16_to_f32(h[e]);
    }
    *reinterpret_cast<uint4 *>(out + ((size_t)t * Mp + m) * Kp + k0) =
        make_uint4(pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]),
                   pack2(h[6], h[7]));
  }
}

// 8 consecutive values of a row -> `terms` bf16 terms in the staging layout
__device__ __forceinline__ void store_terms(float (&r)[8], int terms, u16 *out,
                                            size_t term_stride) {
  for (int t = 0; t < terms; ++t) {
    u16 h[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      h[e] = bf16_rne(r[e]);
      r[e] -= bf16_to_f32(h[e]);
    }
    *reinterpret_cast<uint4 *>(out + t * term_stride) =
        make_uint4(pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]),
                   pack2(h[6], h[7]));
  }
}

// the same for four
__device__ __forceinline__ void store_terms4(const float (&v)[4], int terms, u16 *out, size_t term_stride) {
  float r[4] = {v[0], v[1], v[2], v[3]};
  for (int t = 0; t < terms; ++t) {
    u16 h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h[e] = bf16_rne(r[e]);
      r[e] -= bf16_to_f32(h[e]);
    }
    *reinterpret_cast<uint2 *>(out + t * term_stride) = make_uint2(pack2(h[0], h[1]), pack2(h[2], h[3]));
  }
}

__device__ __forceinline__ float silu_times(float g, float u) {
  const float sig = 1.0f / (1.0f + expf(-g));
  return (g * sig) * u;
}

// The attention's output, added up from its parts, as the terms of the matmul behind it (in f32 rows and
// a conversion: 8.7 + 4.4 us for 150 tokens).  A workgroup per token and four heads: few tokens then come in through
// all compute units (twelve heads to a workgroup: 150 tokens of 37 parts 8.6 us, so 8.2).
constexpr int kFoldThreads = 128;
template <int kMost>
__global__ void __launch_bounds__(kFoldThreads, kMost == 4 ? 8 : 1)
attn_fold_to_terms_kernel(PromptFold f, int64_t o_stride, int n, int terms, int Mp, u16 *__restrict__ out) {
  const int t = blockIdx.x, i = (blockIdx.y * kFoldThreads + threadIdx.x) * 4;
  if (i >= n) // of a head together
    return;
  u16 *row = out + (size_t)t * n;
  const size_t term_stride = (size_t)Mp * n;
  float v[4];
  left4<kMost>(f, o_stride, t, i / kPromptD, i % kPromptD, v);
  repair4(f, t, i / kPromptD, i % kPromptD, v);
  store_terms4(v, terms, row + i, term_stride);
}

// The same rows in f32, for few tokens, whose output product reads them so: two heads a workgroup, since one
// compute unit takes in a token's parts at some 40 bytes a nanosecond.  9 tokens behind 1500, a layer: one
// workgroup a token that makes digits of them, and the prompt's product, 8.9 + 9.2 us; so 5.8 + 5.5.
constexpr int kFoldRowsThreads = 64;
__global__ void __launch_bounds__(kFoldRowsThreads)
attn_fold_rows_kernel(PromptFold f, int64_t o_stride, int n, float *out) {
  const int t = blockIdx.x, i = (blockIdx.y * kFoldRowsThreads + threadIdx.x) * 4;
  if (i >= n)
    return;
  float v[4];
  left4<16>(f, o_stride, t, i / kPromptD, i % kPromptD, v);
  repair4(f, t, i / kPromptD, i % kPromptD, v);
  *reinterpret_cast<float4 *>(out + (int64_t)t * o_stride + i) = make_float4(v[0], v[1], v[2], v[3]);
}

// One workgroup per row: y = w * (x * rsqrt(sum(x^2) / n + eps)) -> staging
__global__ void __launch_bounds__(256)
rmsnorm_to_staging_kernel(const float *__restrict__ x, const float *__restrict__ w, int n,
                          float inv_n, float eps, int terms, int Mp, int Kp,
                          u16 *__restrict__ out) {
  __shared__ float red[4];
  const int row = blockIdx.x;
  const float *xr = x + (size_t)row * n;
  float s = 0.f;
  for (int i = threadIdx.x; i < n; i += 256)
    s = fmaf(xr[i], xr[i], s);
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = s;
  __syncthreads();
  const float tot = (red[0] + red[1]) + (red[2] + red[3]);
  const float rs = 1.0f / sqrtf(tot * inv_n + eps);
  for (int k0 = threadIdx.x * 8; k0 < Kp; k0 += 256 * 8) {
    float r[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      r[e] = k0 + e < n ? w[k0 + e] * (xr[k0 + e] * rs) : 0.f;
    store_terms(r, terms, out + (size_t)row * Kp + k0, (size_t)Mp * Kp);
  }
}

__global__ void __launch_bounds__(256)
silu_mul_to_staging_kernel(const float *__restrict__ g, const float *__restrict__ u,
                           int64_t ld, int rows, int n, int terms, int Mp, int Kp,
                           u16 *__restrict__ out) {
  const int kq = Kp / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)rows * kq)
    return;
  const int row = (int)(i / kq), k0 = (int)(i % kq) * 8;
  float r[8], gv[8], uv[8];
  const float *gr = g + (size_t)row * ld + k0, *ur = u + (size_t)row * ld + k0;
  if (k0 + 7 < n && ((reinterpret_cast<uintptr_t>(gr) | reinterpret_cast<uintptr_t>(ur)) & 15) == 0) {
    const float4 g0 = *reinterpret_cast<const float4 *>(gr), g1 = *reinterpret_cast<const float4 *>(gr + 4);
    const float4 u0 = *reinterpret_cast<const float4 *>(ur), u1 = *reinterpret_cast<const float4 *>(ur + 4);
    gv[0] = g0.x; gv[1] = g0.y; gv[2] = g0.z; gv[3] = g0.w;
    gv[4] = g1.x; gv[5] = g1.y; gv[6] = g1.z; gv[7] = g1.w;
    uv[0] = u0.x; uv[1] = u0.y; uv[2] = u0.z; uv[3] = u0.w;
    uv[4] = u1.x; uv[5] = u1.y; uv[6] = u1.z; uv[7] = u1.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      gv[e] = k0 + e < n ? gr[e] : 0.f;
      uv[e] = k0 + e < n ? ur[e] : 0.f;
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e)
    r[e] = k0 + e < n ? silu_times(gv[e], uv[e]) : 0.f;
  store_terms(r, terms, out + (size_t)row * Kp + k0, (size_t)Mp * Kp);
}

struct GemmArgs {
  const u16 *Abf; // [terms][Mp][Kp]
  const int4 *W;
  const float *scale;
  const float *bias;
  float *C;
  int64_t ldc;
  int M, N, Mp, Kp, groups, chunks;
  int ncols; // column tiles
  // K split over `slices` workgroups per tile, chunks_per_slice chunks of 64 each (the last
  // may hold fewer, never none)
  int slices, chunks_per_slice;
  int row_tiles, panel;      // and how the tiles are placed
  float *partial;            // [tile][slice][wavefront][row][channel], where K is split
  int span, tile_rows;       // channels per wavefront, rows per workgroup
  int accumulate;
  u16 *pair_out; // PAIR: the result's terms [terms][Mp][pair_Kp]
  int pair_Kp;
};

// A tile of 32 RB rows x 128 GP channels, on v_mfma_f32_32x32x16_bf16 (GP tiles of 32 channels per wavefront); every
// wavefront runs the workgroup's whole share of K.  What bounds it: gate | up of 1931 rows, one
// term, takes 126 us in a prompt, 0.84 PFLOP/s and half of what the instruction alone reaches, with
// the conversion of the weights and the way of the rows through LDS in the wavefronts' stream of
// instructions.
//
// Rows go through LDS, weights from memory to registers.  Weights are asked for three
// chunks of 64 k ahead, rows five (two of them in LDS: step c multiplies buffer c % 3, whose
// first fragments were read during step c - 1, and fills buffer (c + 2) % 3, last read before
// the previous barrier).  The weights of a quarter of a chunk are converted while the
// quarter before it is multiplied.
//
// A round of the ring has no branch: where paths of fewer chunks join, the compiler waits for
// all loads but those of the shortest path ahead of any register it uses again.
//
// PAIR: W holds two matrices of a.groups / 2 channel groups each, one behind the other; a tile
// of 32 channels is a group of the first and the same group of the second, and what is stored
// is SiLU(first) * second as the terms of the next matmul's input (as f32 and a launch that
// reads it back: 22.9 + 5.3 us for 150 rows of 1536 -> 2 x 8960, 19.9 now).
constexpr int kRing = 4;               // chunks in registers
constexpr int kRowBytes = 2 * kTileK + 16; // of a row in LDS: reads meet every bank once

template <int TERMS, int RB, int GP, bool PAIR>
__device__ __forceinline__ void multiply_tile(const GemmArgs &a) {
  constexpr int L = TERMS * RB; // layers of 32 rows: term l % TERMS of row block l / TERMS
  constexpr int kWidth = PAIR ? 16 : 32; // channels of the result per tile
  constexpr int kRows = 32 * RB, kSpan = kWidth * GP, kThreads = kWaves * kWave;
  constexpr int kScales = kWaves * 32 * GP;
  constexpr int kBuf = L * 32 * kRowBytes;
  constexpr int kTurn = kSpan + 4; // floats of a row of the epilogue's tile
  constexpr int kTurned = kWaves * 32 * kTurn * 4;
  constexpr int kLds = 3 * kBuf > kTurned ? 3 * kBuf : kTurned;
  __shared__ __attribute__((aligned(16))) unsigned char lds[kLds];
  __shared__ __attribute__((aligned(16))) float scale_s[kScales], bias_s[PAIR ? 4 : kScales];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, up = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int unit, rbk;
  if (!place_tile(a.ncols * a.slices, a.row_tiles, a.panel, unit, rbk))
    return;
  const int ctile = unit % a.ncols, slice = unit / a.ncols;
  const int m0 = rbk * kRows;
  const int g0 = (ctile * kWaves + wave) * (kSpan / 16); // first channel group of this wavefront
  const int cb = slice * a.chunks_per_slice;
  const int nch = min(a.chunks_per_slice, a.chunks - cb); // chunks of this slice, >= 1
  const int half_groups = a.groups / 2; // PAIR only

  const v4i32 *wp[GP];
#pragma unroll
  for (int g = 0; g < GP; ++g) { // groups past the end repeat the last one
    const int second = (lane >> 4) & 1; // group of the tile
    const int gg = PAIR ? min(g0 + g, half_groups - 1) + second * half_groups
                        : min(g0 + 2 * g + second, a.groups - 1);
    wp[g] = reinterpret_cast<const v4i32 *>(a.W) + ((size_t)gg * a.chunks + cb) * 64 + up * 16 +
            (lane & 15);
  }
  const u16 *src[L];
#pragma unroll
  for (int l = 0; l < L; ++l) // 8 threads per row, 32 rows per layer
    src[l] = a.Abf +
             ((size_t)(l % TERMS) * a.Mp + min(m0 + l / TERMS * 32 + tid / 8, a.Mp - 1)) * a.Kp +
             (size_t)cb * kTileK + (tid & 7) * 8;
  const int lds_at = tid / 8 * kRowBytes + (tid & 7) * 16;
  v4i32 wr[kRing][GP * 2], xr[kRing][L];
  constexpr int kFetches = 2 * GP + L; // loads of a chunk
  auto fetch_w = [&](int c, v4i32 (&w)[GP * 2]) {
    const size_t cc = (size_t)min(c, nch - 1) * 64;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int g = 0; g < GP; ++g)
        w[g * 2 + h] = wp[g][cc + h * 32];
  };
  auto fetch_x = [&](int c, v4i32 (&x)[L]) {
    const size_t cc = (size_t)min(c, nch - 1) * kTileK;
#pragma unroll
    for (int l = 0; l < L; ++l)
      x[l] = *reinterpret_cast<const v4i32 *>(src[l] + cc);
  };
  auto put_x = [&](const v4i32 (&x)[L], unsigned char *buf) {
#pragma unroll
    for (int l = 0; l < L; ++l)
      *reinterpret_cast<v4i32 *>(buf + l * 32 * kRowBytes + lds_at) = x[l];
  };
  // quarter t of a chunk: 8 of the 16 k of run t / 2
  auto convert = [&](const v4i32 (&w)[GP * 2], int t, int g) {
    const v4i32 &q = w[g * 2 + t / 2];
    return t % 2 == 0 ? frag_from(q[0], q[1]) : frag_from(q[2], q[3]);
  };
  fetch_x(0, xr[0]);
  fetch_x(1, xr[1]);
#pragma unroll
  for (int u = 0; u < kRing - 1; ++u) {
    fetch_w(u, wr[u]);
    if (u + 2 < kRing)
      fetch_x(u + 2, xr[u + 2]);
  }
  if (a.slices == 1)
    for (int i = tid; i < kScales; i += kThreads) {
      const int mtx = PAIR ? i / (kScales / 2) : 0, n = ctile * kWaves * kSpan + (PAIR ? i % (kScales / 2) : i);
      scale_s[i] = n < a.N ? a.scale[(size_t)mtx * a.N + n] : 0.f;
      if constexpr (!PAIR)
        bias_s[i] = a.bias && n < a.N ? a.bias[n] : 0.f;
    }

  f32x16 acc[GP][RB];
#pragma unroll
  for (int g = 0; g < GP; ++g)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
      acc[g][rb] = f32x16{};

  unsigned char *cur = lds, *next = lds + kBuf, *fill = lds + 2 * kBuf;
  put_x(xr[0], cur);
  put_x(xr[1], next);
  fetch_x(kRing, xr[0]);
  __syncthreads();
  v4i32 frag[4];
  bf16x8 wf[2][GP];
  // sub-step u of a chunk: layer u % L, quarter u / L
  auto load_frag = [&](const unsigned char *buf, int u, v4i32 &f) {
    f = *reinterpret_cast<const v4i32 *>(buf + col * kRowBytes + up * 32 +
                                         u % L * 32 * kRowBytes + u / L / 2 * 64 + u / L % 2 * 16);
  };
  load_frag(cur, 0, frag[0]);
  load_frag(cur, 1, frag[1]);
#pragma unroll
  for (int g = 0; g < GP; ++g)
    wf[0][g] = convert(wr[0], 0, g);
  auto step = [&](int c, const v4i32 (&w)[GP * 2], const v4i32 (&w_next)[GP * 2],
                  v4i32 (&w_new)[GP * 2], v4i32 (&x)[L], v4i32 (&x_new)[L]) {
    const size_t wc = (size_t)min(c + kRing - 1, nch - 1) * 64;
    const size_t xc = (size_t)min(c + kRing + 1, nch - 1) * kTileK;
#pragma unroll
    for (int u = 0; u < 4 * L; ++u) {
      const int t = u / L, l = u % L;
      // fragments are asked for two sub-steps ahead of their products (one takes less than
      // the way through LDS), and stay there: left to itself the scheduler moves them to
      // their use
      load_frag(u + 2 < 4 * L ? cur : next, (u + 2) % (4 * L), frag[(u + 2) & 3]);
      // the chunk's loads evenly between its products, weights first
#pragma unroll
      for (int i = u * kFetches / (4 * L); i < (u + 1) * kFetches / (4 * L); ++i) {
        if (i < 2 * GP)
          w_new[i % GP * 2 + i / GP] = wp[i % GP][wc + i / GP * 32];
        else
          x_new[i - 2 * GP] = *reinterpret_cast<const v4i32 *>(src[i - 2 * GP] + xc);
      }
      if (u >= 1 && u <= L)
        *reinterpret_cast<v4i32 *>(fill + (u - 1) * 32 * kRowBytes + lds_at) = x[u - 1];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < GP; ++g) {
        union {
          v4i32 i;
          bf16x8 v;
        } f;
        f.i = frag[u & 3];
        acc[g][l / TERMS] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[t & 1][g], f.v,
                                                                    acc[g][l / TERMS], 0, 0, 0);
        // behind a product that takes 32 cycles: a piece of the next quarter's weights
        if (g % L == l)
          wf[(t + 1) & 1][g] = t < 3 ? convert(w, t + 1, g) : convert(w_next, 0, g);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    unsigned char *b = cur;
    cur = next;
    next = fill;
    fill = b;
  };
  // step c: weights from slot c, new ones into slot c - 1; rows c + 2 go to LDS, new ones
  // into slot c + 1 (all modulo kRing)
  auto turn = [&](int c0, auto slot) {
    constexpr int u = slot;
    step(c0 + u, wr[u], wr[(u + 1) % kRing], wr[(u + kRing - 1) % kRing], xr[(u + 2) % kRing],
         xr[(u + 1) % kRing]);
  };
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

  // ---- epilogue: a lane holds channels 8 q + 4 up + 0..3, q = 0..3, of row `col` of every
  // tile; the wavefront turns 32 rows around in its own part of LDS (free now: every
  // wavefront is past the last barrier of the loop) and writes whole row segments
  float *tile = reinterpret_cast<float *>(lds) + wave * (32 * kTurn);
  const int n0 = g0 * kTileN; // (PAIR: groups of 16 channels of the result as well)
  constexpr int kQuads = kSpan / 4; // float4 of a row
  if constexpr (PAIR) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
      for (int g = 0; g < GP; ++g)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int ch = g * 16 + 8 * q + 4 * up;
          const float *sg = scale_s + wave * kSpan + ch, *su = sg + kScales / 2;
          float o[4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            o[i] = silu_times(acc[g][rb][4 * q + i] * sg[i], acc[g][rb][4 * q + 8 + i] * su[i]);
          *reinterpret_cast<float4 *>(tile + col * kTurn + ch) = make_float4(o[0], o[1], o[2], o[3]);
        }
#pragma unroll
      for (int i = 0; i < kQuads / 2; ++i) {
        const int idx = lane + 64 * i, row = idx / kQuads, c4 = idx % kQuads;
        const float4 o = *reinterpret_cast<const float4 *>(tile + row * kTurn + c4 * 4);
        const int m = m0 + rb * 32 + row, n = n0 + c4 * 4;
        if (m >= a.M || n >= a.pair_Kp)
          continue;
        // a.N is a multiple of 16: four channels are in the result or in its padding
        const float v[4] = {o.x, o.y, o.z, o.w}, none[4] = {0.f, 0.f, 0.f, 0.f};
        store_terms4(n < a.N ? v : none, TERMS, a.pair_out + (size_t)m * a.pair_Kp + n,
                     (size_t)a.Mp * a.pair_Kp);
      }
    }
    return;
  }
  const size_t at = ((size_t)(rbk * a.ncols + ctile) * a.slices + slice) * kWaves + wave;
  float *part = a.partial + at * kRows * kSpan;
  const bool vec = (a.ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(a.C) & 15) == 0;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
    for (int g = 0; g < GP; ++g)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ch = g * 32 + 8 * q + 4 * up;
        float4 o = make_float4(acc[g][rb][4 * q], acc[g][rb][4 * q + 1], acc[g][rb][4 * q + 2],
                               acc[g][rb][4 * q + 3]);
        if (a.slices == 1) {
          const float4 s = *reinterpret_cast<const float4 *>(scale_s + wave * kSpan + ch);
          const float4 b = *reinterpret_cast<const float4 *>(bias_s + wave * kSpan + ch);
          o = make_float4(b.x + o.x * s.x, b.y + o.y * s.y, b.z + o.z * s.z, b.w + o.w * s.w);
        }
        *reinterpret_cast<float4 *>(tile + col * kTurn + ch) = o;
      }
#pragma unroll
    for (int i = 0; i < kQuads / 2; ++i) {
      const int idx = lane + 64 * i, row = idx / kQuads, c4 = idx % kQuads;
      const float4 o = *reinterpret_cast<const float4 *>(tile + row * kTurn + c4 * 4);
      if (a.slices > 1) {
        *reinterpret_cast<float4 *>(part + (size_t)(rb * 32 + row) * kSpan + c4 * 4) = o;
        continue;
      }
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
  }
}

// What a wavefront needs before its first fetch arrives in SGPRs (this file is built
// with -amdgpu-kernarg-preload-count); the rest is loaded behind the fetch.
#define BH_BF16_LEADING                                                                            \
  const u16 *Abf, const int4 *W, int Mp, int Kp, int groups, int chunks, int ncols, int slices,    \
      int chunks_per_slice, int row_tiles, int panel, GemmArgs a
#define BH_BF16_TAKE                                                                               \
  a.Abf = Abf;                                                                                     \
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

// Blocks of 32 rows per workgroup.
constexpr int row_blocks(int terms, int gp) { return terms == 1 && gp == 2 ? 2 : 1; }

// 128 channels per workgroup, and 256
template <int TERMS, bool PAIR>
__global__ void __launch_bounds__(kWaves *kWave) gemm_w8_bf16_kernel(BH_BF16_LEADING) {
  BH_BF16_TAKE
  multiply_tile<TERMS, 1, 1, PAIR>(a);
}
template <int TERMS, bool PAIR>
__global__ void __launch_bounds__(kWaves *kWave) gemm_w8_bf16_wide_kernel(BH_BF16_LEADING) {
  BH_BF16_TAKE
  multiply_tile<TERMS, row_blocks(TERMS, 2), 2, PAIR>(a);
}

// C (+)= scale[n] * sum over the K slices, in slice order (+ bias); four loads are in flight
// at a time (slices past the end repeat the last one and are not added).
__global__ void __launch_bounds__(256) add_slices_kernel(GemmArgs a) {
  const int n4 = (a.N + 3) / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)a.M * n4)
    return;
  const int m = (int)(i / n4), n = (int)(i % n4) * 4;
  const int tile = m / a.tile_rows * a.ncols + n / (kWaves * a.span), wave = n / a.span % kWaves;
  const size_t row = ((size_t)tile * a.slices * kWaves + wave) * a.tile_rows + m % a.tile_rows;
  const size_t stride = (size_t)kWaves * a.tile_rows * a.span;
  const float *p = a.partial + row * a.span + n % a.span;
  float *c = a.C + (int64_t)m * a.ldc + n;
  float s[4], b[4], v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const bool in = n + r < a.N;
    s[r] = in ? a.scale[n + r] : 0.f;
    b[r] = !in ? 0.f : a.accumulate ? c[r] : a.bias ? a.bias[n + r] : 0.f;
  }
  for (int sl = 0; sl < a.slices; sl += 4) {
    float4 q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      q[u] = *reinterpret_cast<const float4 *>(p + (size_t)min(sl + u, a.slices - 1) * stride);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (sl + u < a.slices) {
        v[0] += q[u].x;
        v[1] += q[u].y;
        v[2] += q[u].z;
        v[3] += q[u].w;
      }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (n + r < a.N)
      c[r] = b[r] + v[r] * s[r];
}

// The same, one workgroup per row, which then writes RMSNorm(row) * w as the terms of the next
// matmul's input.  lds: [Kp2] the row, [Kp2] norm weights.  Everything in memory is asked for
// ahead of the row's one sum (150 rows of 1536 in five slices: 4.2 + 4.9 us in two launches,
// 5.1 in this one).
constexpr int kNormThreads = 512;
constexpr int kNormColumns = 12288; // 96 KB of LDS
__global__ void __launch_bounds__(kNormThreads)
add_slices_norm_kernel(GemmArgs a, const float *__restrict__ norm_w, float inv_n, float eps, int terms,
                       int Kp2, u16 *__restrict__ out) {
  __shared__ float red[kNormThreads / 64];
  extern __shared__ __attribute__((aligned(16))) float xrow[];
  float *wrow = xrow + Kp2;
  const int m = blockIdx.x;
  const size_t stride = (size_t)kWaves * a.tile_rows * a.span;
  float *c = a.C + (int64_t)m * a.ldc;
  float ss = 0.f;
  for (int n = threadIdx.x * 4; n < Kp2; n += kNormThreads * 4) {
    float s[4], b[4], w[4], v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const bool in = n + r < a.N;
      s[r] = in ? a.scale[n + r] : 0.f;
      b[r] = !in ? 0.f : a.accumulate ? c[n + r] : a.bias ? a.bias[n + r] : 0.f;
      w[r] = in ? norm_w[n + r] : 0.f;
    }
    if (n < a.N) {
      const int tile = m / a.tile_rows * a.ncols + n / (kWaves * a.span), wave = n / a.span % kWaves;
      const size_t row = ((size_t)tile * a.slices * kWaves + wave) * a.tile_rows + m % a.tile_rows;
      const float *p = a.partial + row * a.span + n % a.span;
      for (int sl = 0; sl < a.slices; sl += 4) {
        float4 q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          q[u] = *reinterpret_cast<const float4 *>(p + (size_t)min(sl + u, a.slices - 1) * stride);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (sl + u < a.slices) {
            v[0] += q[u].x;
            v[1] += q[u].y;
            v[2] += q[u].z;
            v[3] += q[u].w;
          }
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[r] = n + r < a.N ? b[r] + v[r] * s[r] : 0.f;
      if (n + r < a.N)
        c[n + r] = v[r];
      ss = fmaf(v[r], v[r], ss);
    }
    *reinterpret_cast<float4 *>(xrow + n) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4 *>(wrow + n) = make_float4(w[0], w[1], w[2], w[3]);
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int i = 0; i < kNormThreads / 64; i += 2)
    tot += red[i] + red[i + 1];
  const float rs = 1.0f / sqrtf(tot * inv_n + eps);
  for (int n = threadIdx.x * 4; n < Kp2; n += kNormThreads * 4) { // the thread's own values
    const float4 x = *reinterpret_cast<const float4 *>(xrow + n), w = *reinterpret_cast<const float4 *>(wrow + n);
    const float v[4] = {w.x * (x.x * rs), w.y * (x.y * rs), w.z * (x.z * rs), w.w * (x.w * rs)};
    store_terms4(v, terms, out + (size_t)m * Kp2 + n, (size_t)a.Mp * Kp2);
  }
}

// bf16 staging of the activations: one grow-only device buffer per stream, so
// that calls on different streams do not share it.  Calls on one stream are
// ordered, and the buffer is only read by the matmul that follows the
// conversion on that stream.
struct Staging {
  u16 *ptr = nullptr;
  size_t bytes = 0;
};
std::mutex g_staging_mutex;
std::map<hipStream_t, Staging> g_staging;

int staging_for(hipStream_t stream, size_t bytes, u16 **out) {
  std::lock_guard<std::mutex> lock(g_staging_mutex);
  Staging &s = g_staging[stream];
  if (s.bytes < bytes) {
    if (s.ptr) {
      BH_CHECK_HIP(hipStreamSynchronize(stream)); // an earlier matmul may still read it
      BH_CHECK_HIP(hipFree(s.ptr));
      s.ptr = nullptr;
      s.bytes = 0;
    }
    BH_CHECK_HIP(hipMalloc(reinterpret_cast<void **>(&s.ptr), bytes));
    s.bytes = bytes;
  }
  *out = s.ptr;
  return BUDDY_HIP_OK;
}

BH_VARIANT_FAMILY(WideFamily, "gemm_w8_bf16_wide_kernel");
BH_VARIANT_FAMILY(NarrowFamily, "gemm_w8_bf16_kernel");
BH_TILE_FAMILY(PairFamily, "gemm_w8_bf16_kernel pair"); // terms, channel tiles per wavefront
BH_TILE_FAMILY(SlicesNormFamily, "add_slices_norm_kernel"); // more LDS than a launch gets unasked
BH_TILE_FAMILY(NormBehindFamily, "add_slices_kernel and a norm behind it"); // 1

template <class Kernel>
int launch_tiles(Kernel kernel, const GemmArgs &a, unsigned blocks, hipStream_t stream) {
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kWaves * kWave), 0, stream, a.Abf, a.W, a.Mp, a.Kp,
                     a.groups, a.chunks, a.ncols, a.slices, a.chunks_per_slice, a.row_tiles, a.panel, a);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

// Channel tiles per wavefront and K slices for a launch, by an estimate of its time in
// microseconds.  An XCD (32 compute units) works on 64 workgroups at a time, two to a compute
// unit.  A chunk of 64 k on L layers of 32 rows (terms, blocks of rows) takes a compute unit
// with two workgroups 0.20 + 0.38 L us, one that has its compute unit to itself 0.29 + 0.14 L
// us (with one channel tile 0.20 + 0.185 L and 0.17 + 0.073 L); a last round that fills less
// than half runs at the latter.  Fitted to launches of 20 to 1931 rows of 1536, 4096, 8960 and
// 14336 k, both tiles with every K split.  Of 528 launches of 17 to 2048 rows under the profiler its
// pick is 2.1 (one term) and 1.1 % (three) off the best on average.
// Microseconds of a product in a prompt of 150 rows, one term (in brackets with a branch at every
// chunk and its loads at the chunk's start): 1536 -> 2048 10.9 [14.1], 1536 -> 2 x 8960 19.9
// [22.9], 8960 -> 1536 11.6 [13.0] without the adding of its slices.
struct TilePlan {
  int gp = 0, slices = 1;
  double us = 0;
};
// A norm of the finished rows is a launch of its own, 5 us, unless the kernel that adds the
// slices does it; the rotation of q and k 4 us, there 0.5 and what its angles
// take, which every head works out for itself.
TilePlan plan_tiles(int64_t M, int64_t channels, int chunks, int terms, bool may_split, bool pair,
                    double norm_us, double split_norm_us) {
  TilePlan best;
  for (int gp = 1; gp <= 2; ++gp) {
    const int layers = terms * row_blocks(terms, gp);
    const int64_t rows = ceil_div(M, 32 * row_blocks(terms, gp));
    const int64_t ncols = ceil_div(channels, kWaves * (pair ? 16 : 32) * gp);
    const double alone = gp == 2 ? 0.291 + 0.141 * layers : 0.172 + 0.073 * layers;
    const double full = gp == 2 ? 0.203 + 0.38 * layers : 0.20 + 0.185 * layers;
    for (int s = 1; s <= (may_split ? 16 : 1); ++s) {
      const int64_t per_xcd = ceil_div(ncols * s * rows, 8);
      if (s > 1 && per_xcd > 256)
        break;
      const int64_t cps = ceil_div(chunks, s);
      if (ceil_div(chunks, cps) != s)
        continue; // the last slice would be empty
      const double store = s > 1 ? 2.0 : 0.0; // of the partial sums
      const double full_us = full * (double)cps + 5.95 + store;
      const double alone_us = alone * (double)cps + 4.15 + store;
      const int64_t left = per_xcd % 64;
      double us = (double)(per_xcd / 64) * full_us +
                  (left == 0 ? 0.0 : 2 * left <= 64 ? alone_us : full_us);
      if (s > 1) // the kernel that adds the slices: 4 us and its bytes
        us += 4.0 + 4.0 * (double)(M * s) * (double)(ncols * 128 * gp) / 5e6 + split_norm_us;
      else
        us += norm_us;
      if (!best.gp || us < best.us - 1e-9)
        best = {gp, s, us};
    }
  }
  return best;
}

template <int GP, bool PAIR>
int launch_width(const GemmArgs &a, int terms, unsigned blocks, hipStream_t stream) {
  auto run = [&](auto t) {
    constexpr int T = t;
    if constexpr (PAIR)
      BH_NOTE_VARIANT(PairFamily, T, GP);
    else if constexpr (GP == 1)
      BH_NOTE_VARIANT(NarrowFamily, T);
    else
      BH_NOTE_VARIANT(WideFamily, T);
    if constexpr (GP == 1)
      return launch_tiles(gemm_w8_bf16_kernel<T, PAIR>, a, blocks, stream);
    else
      return launch_tiles(gemm_w8_bf16_wide_kernel<T, PAIR>, a, blocks, stream);
  };
  return terms == 1 ? run(std::integral_constant<int, 1>{}) : run(std::integral_constant<int, 3>{});
}

int launch_plan(const TilePlan &plan, GemmArgs &a, const GemmW8Args &in, hipStream_t stream) {
  const int terms = in.terms;
  const GemmStagingLayout next = gemm_staging_layout(in.M, in.N);
  const bool fuses = next.cols_padded <= kNormColumns;
  a.tile_rows = 32 * row_blocks(terms, plan.gp);
  a.span = 32 * plan.gp;
  a.ncols = (int)ceil_div(a.N, kWaves * (a.pair_out ? a.span / 2 : a.span));
  a.row_tiles = (int)ceil_div(a.M, a.tile_rows);
  a.slices = plan.slices;
  a.chunks_per_slice = (int)ceil_div(a.chunks, plan.slices);
  a.partial = nullptr;
  if (a.slices > 1) {
    const size_t tile_floats = (size_t)a.tile_rows * kWaves * a.span;
    char *ws = nullptr;
    if (int rc = gemm_slices_workspace(
            stream, sizeof(float) * tile_floats * a.slices * (size_t)a.ncols * a.row_tiles, &ws))
      return rc;
    if (!ws) // under capture: K whole
      return launch_plan(plan_tiles(a.M, a.N, a.chunks, terms, false, false, 0.0, 0.0), a, in, stream);
    a.partial = reinterpret_cast<float *>(ws);
  }
  const int64_t units = (int64_t)a.ncols * a.slices;
  a.panel = panel_for(units, a.row_tiles, false);
  const int64_t tiles = (a.panel ? units : round_up(units, 8)) * a.row_tiles;
  BH_REQUIRE(tiles < (1u << 31), "gemm_w8: %lld tiles", (long long)tiles);
  const unsigned blocks = (unsigned)tiles;
  int rc;
  if (a.pair_out)
    return plan.gp == 1 ? launch_width<1, true>(a, terms, blocks, stream)
                        : launch_width<2, true>(a, terms, blocks, stream);
  rc = plan.gp == 1 ? launch_width<1, false>(a, terms, blocks, stream)
                    : launch_width<2, false>(a, terms, blocks, stream);
  if (rc)
    return rc;
  u16 *normed = static_cast<u16 *>(in.then_norm_staged);
  if (a.slices > 1 && in.then_norm_w && fuses) {
    const size_t lds = 2 * sizeof(float) * (size_t)next.cols_padded;
    if (lds <= 48 * 1024) {
      BH_NOTE_VARIANT(SlicesNormFamily, 0);
    } else {
      BH_NOTE_VARIANT(SlicesNormFamily, 1);
      static DynLdsOnce once;
      BH_CHECK_HIP(ensure_dyn_lds(once, reinterpret_cast<const void *>(add_slices_norm_kernel),
                                  (int)(2 * sizeof(float) * kNormColumns)));
    }
    hipLaunchKernelGGL(add_slices_norm_kernel, dim3((unsigned)a.M), dim3(kNormThreads), lds, stream, a,
                       in.then_norm_w, 1.0f / (float)a.N, in.then_norm_eps, terms, next.cols_padded, normed);
    BH_CHECK_HIP(hipGetLastError());
    return BUDDY_HIP_OK;
  }
  if (in.then_rope) {
    const RopeKv &r = *in.then_rope;
    if (a.slices > 1)
      return launch_slices_rope({a.partial, nullptr, a.scale, a.bias, a.slices, a.span, a.tile_rows, a.ncols, a.N},
                                r, a.C, a.ldc, a.M, stream);
    return launch_rope_kv_write(a.C, a.ldc, r, a.M, stream);
  }
  if (a.slices > 1) {
    if (in.then_norm_w)
      BH_NOTE_VARIANT(NormBehindFamily, 1);
    const int64_t threads = (int64_t)a.M * ceil_div(a.N, 4);
    hipLaunchKernelGGL(add_slices_kernel, dim3((unsigned)ceil_div(threads, 256)), dim3(256), 0,
                       stream, a);
    BH_CHECK_HIP(hipGetLastError());
  }
  return in.then_norm_w ? launch_rmsnorm_to_staging(a.C, in.then_norm_w, a.M, a.N, in.then_norm_eps, terms,
                                                    normed, stream)
                        : BUDDY_HIP_OK;
}

} // namespace

GemmStagingLayout gemm_staging_layout(int64_t M, int64_t K) {
  GemmStagingLayout l;
  l.rows_padded = (int)round_up(M, 32); // rows of a tile beyond these repeat the last
  l.cols_padded = (int)round_up(K, kTileK);
  return l;
}

int launch_rmsnorm_to_staging(const float *x, const float *w, int rows, int n, float eps,
                              int terms, unsigned short *staged, hipStream_t stream) {
  BH_REQUIRE(x && w && staged && rows > 0 && n > 0 && terms >= 1 && terms <= 3,
             "rmsnorm_to_staging: bad argument");
  const GemmStagingLayout l = gemm_staging_layout(rows, n);
  hipLaunchKernelGGL(rmsnorm_to_staging_kernel, dim3(rows), dim3(256), 0, stream, x, w, n,
                     1.0f / (float)n, eps, terms, l.rows_padded, l.cols_padded, staged);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

int launch_attn_fold_to_terms(const PromptFold &fold, int64_t o_stride, int heads, int tokens, int terms,
                              unsigned short *staged, hipStream_t stream) {
  const int64_t K = (int64_t)heads * kPromptD;
  BH_REQUIRE(fold.blocks && staged && tokens > 0 && terms >= 1 && terms <= 3, "attn_fold_to_terms: bad argument");
  const GemmStagingLayout l = gemm_staging_layout(tokens, K); // K is a multiple of 64: no padding
  hipLaunchKernelGGL(tokens > kFoldTokens ? attn_fold_to_terms_kernel<4> : attn_fold_to_terms_kernel<16>,
                     dim3(tokens, (unsigned)ceil_div(K, 4 * kFoldThreads)), dim3(kFoldThreads), 0, stream, fold,
                     o_stride, (int)K, terms, l.rows_padded, staged);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

int launch_attn_fold_rows(const PromptFold &fold, int64_t o_stride, int heads, int tokens, float *out,
                          hipStream_t stream) {
  BH_REQUIRE(fold.blocks && out && tokens > 0 && o_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0,
             "attn_fold_rows: bad argument");
  const int n = heads * kPromptD;
  hipLaunchKernelGGL(attn_fold_rows_kernel, dim3(tokens, (unsigned)ceil_div(n, 4 * kFoldRowsThreads)),
                     dim3(kFoldRowsThreads), 0, stream, fold, o_stride, n, out);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

int launch_silu_mul_to_staging(const float *g, const float *u, int64_t ld, int rows, int n, int terms,
                               unsigned short *staged, hipStream_t stream) {
  BH_REQUIRE(g && u && staged && rows > 0 && n > 0 && terms >= 1 && terms <= 3,
             "silu_mul_to_staging: bad argument");
  const GemmStagingLayout l = gemm_staging_layout(rows, n);
  const int64_t threads = (int64_t)rows * (l.cols_padded / 8);
  hipLaunchKernelGGL(silu_mul_to_staging_kernel, dim3((unsigned)ceil_div(threads, 256)),
                     dim3(256), 0, stream, g, u, ld, rows, n, terms, l.rows_padded,
                     l.cols_padded, staged);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

int launch_gemm_w8(const GemmW8Args &in, hipStream_t stream) {
  BH_REQUIRE((in.A || in.staged) && in.W && in.scale && (in.C || (in.silu_staged && !in.digits)),
             "gemm_w8: null pointer");
  BH_REQUIRE(in.M > 0 && in.K > 0 && in.N > 0 && in.M < (1 << 24) &&
                 in.K < (1 << 24) && in.N < (1 << 24),
             "gemm_w8: bad shape M=%lld K=%lld N=%lld", (long long)in.M,
             (long long)in.K, (long long)in.N);
  BH_REQUIRE((in.staged || in.lda >= in.K) && (!in.C || in.ldc >= (in.silu_pair ? in.N / 2 : in.N)),
             "gemm_w8: row stride below row length");
  BH_REQUIRE(!in.silu_pair || in.digits || (in.silu_staged && in.staged && in.N % (2 * kTileN) == 0 && !in.bias &&
                                            !in.accumulate && !in.then_norm_w),
             "gemm_w8: the SiLU pair of bfloat16 terms needs staged rows, two matrices of a multiple of 16 "
             "channels and a buffer for its terms");
  BH_REQUIRE(!in.then_norm_w || (in.then_norm_staged && (in.digits || in.ldc == in.N)),
             "gemm_w8: a following norm needs a buffer for its rows");
  if (in.then_rope) {
    const RopeKv &r = *in.then_rope;
    BH_REQUIRE(!in.silu_pair && !in.accumulate && !in.then_norm_w && in.ldc == in.N && r.inv_freq &&
                   r.kcache && r.vcache && r.heads > 0 && r.kv_heads > 0 &&
                   in.N == (int64_t)(r.heads + 2 * r.kv_heads) * kAttnHeadDim && r.start_pos >= 0 &&
                   r.start_pos + in.M <= r.max_len &&
                   ((reinterpret_cast<uintptr_t>(in.C) | reinterpret_cast<uintptr_t>(r.kcache) |
                     reinterpret_cast<uintptr_t>(r.vcache)) & 15) == 0,
               "gemm_w8: q | k | v with what follows it");
  }
  // one bf16 term (activations cast to bf16) or three (every f32 bit); three
  // digit planes (23 bits below the row's maximum) or two (15 bits: the fixed
  // point counterpart of the bf16 cast, for the same third less matrix work)
  BH_REQUIRE(in.terms == 1 || in.terms == 3, "gemm_w8: terms=%d (1 or 3)", in.terms);
  BH_REQUIRE(in.digits == 0 || in.digits == 2 || in.digits == 3,
             "gemm_w8: digits=%d (0, 2 or 3)", in.digits);
  BH_REQUIRE(in.digits == 0 || in.K <= (1 << 17),
             "gemm_w8: K=%lld beyond 2^17 would overflow the int32 sums of the digit planes",
             (long long)in.K);
  BH_REQUIRE(!(in.bias && in.accumulate), "gemm_w8: bias with accumulate");
  BH_REQUIRE((reinterpret_cast<uintptr_t>(in.W) & 15) == 0,
             "gemm_w8: packed weights must be 16-byte aligned");
  GemmArgs a;
  a.W = reinterpret_cast<const int4 *>(in.W);
  a.scale = in.scale;
  a.bias = in.bias;
  a.C = in.C;
  a.ldc = in.ldc;
  a.M = (int)in.M;
  a.N = (int)in.N;
  a.groups = (int)ceil_div(in.N, kTileN);
  a.chunks = (int)ceil_div(in.K, kTileK);
  const GemmStagingLayout layout = gemm_staging_layout(in.M, in.K);
  a.Mp = layout.rows_padded;
  a.Kp = layout.cols_padded;
  a.accumulate = in.accumulate ? 1 : 0;
  u16 *abf = static_cast<u16 *>(const_cast<void *>(in.staged));
  const bool staged = in.staged != nullptr;
  const size_t staging_bytes =
      in.digits ? layout.bytes_digits(in.digits) : layout.bytes(in.terms);
  int rc = staged ? BUDDY_HIP_OK : staging_for(stream, staging_bytes, &abf);
  if (rc)
    return rc;
  if (in.digits) {
    if (!staged &&
        (rc = launch_activations_to_digits(in.A, in.lda, in.M, in.K, in.digits, abf, stream)))
      return rc;
    return launch_gemm_w8_digits(in, abf, stream);
  }
  a.Abf = abf;
  if (!staged) {
    const int64_t threads = (int64_t)a.Mp * (a.Kp / 8);
    hipLaunchKernelGGL(activations_to_bf16, dim3((unsigned)ceil_div(threads, 256)),
                       dim3(256), 0, stream, in.A, in.lda, a.M, (int)in.K, a.Mp, a.Kp,
                       in.terms, abf);
    BH_CHECK_HIP(hipGetLastError());
  }
  a.pair_out = nullptr;
  if (in.silu_pair) {
    a.N = (int)(in.N / 2);
    a.pair_out = static_cast<u16 *>(in.silu_staged);
    a.pair_Kp = gemm_staging_layout(in.M, a.N).cols_padded;
    return launch_plan(plan_tiles(in.M, a.N, a.chunks, in.terms, false, true, 0.0, 0.0), a, in, stream);
  }
  const double norm_us = in.then_norm_w ? 5.0 : in.then_rope ? 4.0 : 0.0;
  const bool fuses = gemm_staging_layout(in.M, in.N).cols_padded <= kNormColumns;
  const double split_norm_us = in.then_rope ? 0.5 + 0.004 * (double)in.M : fuses ? 0.0 : norm_us;
  return launch_plan(plan_tiles(in.M, in.N, a.chunks, in.terms, true, false, norm_us, split_norm_us), a, in,
                     stream);
}

void release_gemm_staging(hipStream_t stream) {
  release_gemm_i8_workspace(stream);
  std::lock_guard<std::mutex> lock(g_staging_mutex);
  auto it = g_staging.find(stream);
  if (it == g_staging.end())
    return;
  if (it->second.ptr) {
    (void)hipStreamSynchronize(stream);
    (void)hipFree(it->second.ptr);
  }
  g_staging.erase(it);
}

} // namespace bh

extern "C" {

int buddy_hip_gemm_w8a32(const float *A, const int8_t *packed, const float *scale,
                         float *C, int64_t M, int64_t K, int64_t N,
                         unsigned flags, buddy_hip_stream stream) try {
  bh::GemmW8Args a;
  a.A = A;
  a.lda = K;
  a.W = packed;
  a.scale = scale;
  a.C = C;
  a.ldc = N;
  a.M = M;
  a.K = K;
  a.N = N;
  a.accumulate = (flags & BUDDY_HIP_GEMV_ACCUMULATE) != 0;
  a.terms = (flags & BUDDY_HIP_GEMM_A_F32_EXACT) ? 3 : 1;
  a.digits = (flags & BUDDY_HIP_GEMM_A_I8_DIGITS) ? ((flags & BUDDY_HIP_GEMM_TWO_DIGITS) ? 2 : 3) : 0;
  BH_REQUIRE(a.digits || !(flags & BUDDY_HIP_GEMM_TWO_DIGITS),
             "gemm_w8a32: BUDDY_HIP_GEMM_TWO_DIGITS needs BUDDY_HIP_GEMM_A_I8_DIGITS");
  if (flags & BUDDY_HIP_GEMM_SILU_PAIR) {
    BH_REQUIRE(a.digits, "gemm_w8a32: BUDDY_HIP_GEMM_SILU_PAIR needs BUDDY_HIP_GEMM_A_I8_DIGITS");
    a.silu_pair = true;
    a.N = 2 * N; // both matrices; the result has N channels
  }
  return bh::launch_gemm_w8(a, bh::as_stream(stream));
} BH_CATCH_INT("buddy_hip_gemm_w8a32")
}
