// gemv_w8a8.hip -- w8a8 matmul: dynamic per-tensor int8 activations times int8
// weights with exact int32 partial sums.
//
// Replaces quantized_matmul_op / _quantize_activation_i8
// (frontend/Python/ops/linalg.py:12728-12847):
//   s_a  = max(absmax(x) * (1/127), 1e-10)            (:12737-12760)
//   x_q  = clamp(f32(i32(x * (1/s_a))), -128, 127)     (:12761-12792; the TOSA
//          f32 -> i32 cast rounds to nearest even)
//   acc  = x_q (i8) . W (i8) -> i32                    (:12814-12831)
//   y    = f32(acc) * (s_a * s_w[n])                   (:12833-12845)
// The int8 weights are the same wave-tile packed copy the w8a32 kernels read, and
// the partial sums are exact integers whatever the order.
//
// Few rows are quantised by the workgroups that multiply them (w8a8_rows_kernel): one launch where a
// workgroup's rows are all there are, else partial maxima over the tensor ahead of it and, where K goes
// to several workgroups, a launch behind it that adds their int32 sums.
//
// More rows run on the int8 matrix cores of the prefill matmul (the i8 x i8 -> i32
// branch of the reference's BLIS kernel,
// midend/lib/Conversion/MatMulOptimization/MatMulBlisVectorization.cpp:668-724):
// the quantised activations are written as one plane in the layout it
// reads, by two launches (partial maxima over the tensor, then one
// workgroup per row), and the prefill kernel multiplies it; where K goes to several
// workgroups, their int32 sums are added as integers.  Above 16 rows that is also
// the way of rows that cannot be read 16 bytes at a time, up to 16 v_dot4_i32_i8 behind one workgroup
// that quantises.
#include "common.h"
#include <algorithm>
#include <type_traits>
#include "gemm.h"

namespace bh {
namespace {

// absmax over the whole activation tensor, one workgroup
__global__ void __launch_bounds__(1024)
w8a8_quantize_kernel(const float *__restrict__ x, int64_t n, int M, int K, int Kp,
                     int8_t *__restrict__ xq, float *__restrict__ scale_out) {
  __shared__ float red[16];
  __shared__ float s_inv;
  float m = 0.f;
  for (int64_t i = threadIdx.x; i < n; i += 1024)
    m = fmaxf(m, fabsf(x[i]));
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = red[0];
    for (int w = 1; w < 16; ++w)
      t = fmaxf(t, red[w]);
    const float r127 = 1.0f / 127.0f;
    float s = t * r127;
    s = fmaxf(s, 1e-10f);
    *scale_out = s;
    s_inv = 1.0f / s;
  }
  __syncthreads();
  const float inv = s_inv;
  // rows are padded to Kp (a multiple of 64) with zeros
  for (int64_t i = threadIdx.x; i < (int64_t)M * Kp; i += 1024) {
    const int m_ = (int)(i / Kp), k = (int)(i % Kp);
    float r = 0.f;
    if (k < K) {
      r = rintf(x[(int64_t)m_ * K + k] * inv);
      r = fminf(fmaxf(r, -128.0f), 127.0f);
    }
    xq[i] = (int8_t)r;
  }
}


// stage 1 of the quantisation of many rows: workgroup g leaves the largest
// magnitude of its share of the tensor in part[g]
__global__ void __launch_bounds__(256)
w8a8_absmax_parts_kernel(const float *__restrict__ x, int64_t n, float *__restrict__ part) {
  __shared__ float red[4];
  float m = 0.f;
  const int64_t stride = (int64_t)gridDim.x * 256, first = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) { // 16 bytes per load, the tail one by one
    const int64_t n4 = n / 4;
    for (int64_t i = first; i < n4; i += stride) {
      const float4 v = reinterpret_cast<const float4 *>(x)[i];
      m = fmaxf(fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
    }
    for (int64_t i = 4 * n4 + first; i < n; i += stride)
      m = fmaxf(m, fabsf(x[i]));
  } else {
    for (int64_t i = first; i < n; i += stride)
      m = fmaxf(m, fabsf(x[i]));
  }
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0)
    part[blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

template <int M>
__global__ void __launch_bounds__(256)
w8a8_gemv_kernel(const int4 *__restrict__ W, const int8_t *__restrict__ xq,
                 const float *__restrict__ a_scale, const float *__restrict__ wscale,
                 float *__restrict__ C, int32_t *__restrict__ acc_out, int rows,
                 int N, int groups, int chunks, int Kp) {
  // 4 wavefronts split the k range of one channel group
  __shared__ int red[4][M][16];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int g = blockIdx.x;
  const int per = (chunks + 3) / 4;
  const int t0 = min(wave * per, chunks), t1 = min(t0 + per, chunks);
  // the two scales of the result: asked for with the first loads, not at the
  // very end of the launch behind the meeting of the wavefronts
  const float comb = *a_scale * wscale[min(g * 16 + (lane & 15), N - 1)];
  int acc[M];
#pragma unroll
  for (int m = 0; m < M; ++m)
    acc[m] = 0;
  const int4 *w = W + ((size_t)g * chunks) * 64 + lane;
  const int kg = lane >> 4;
  for (int t = t0; t < t1; ++t) {
    const int4 wv = w[(size_t)t * 64];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      if (m < rows) {
        const int4 xv = *reinterpret_cast<const int4 *>(xq + (size_t)m * Kp + t * 64 + kg * 16);
        int a = acc[m];
        a = __builtin_amdgcn_sdot4(wv.x, xv.x, a, false);
        a = __builtin_amdgcn_sdot4(wv.y, xv.y, a, false);
        a = __builtin_amdgcn_sdot4(wv.z, xv.z, a, false);
        a = __builtin_amdgcn_sdot4(wv.w, xv.w, a, false);
        acc[m] = a;
      }
    }
  }
#pragma unroll
  for (int m = 0; m < M; ++m) {
    acc[m] += __shfl_xor(acc[m], 16, 64);
    acc[m] += __shfl_xor(acc[m], 32, 64);
  }
  if (lane < 16) {
#pragma unroll
    for (int m = 0; m < M; ++m)
      red[wave][m][lane] = acc[m];
  }
  __syncthreads();
  if (wave == 0 && lane < 16) {
    const int n = g * 16 + lane;
    if (n < N) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        if (m < rows) {
          const int tot = red[0][m][lane] + red[1][m][lane] + red[2][m][lane] + red[3][m][lane];
          if (acc_out)
            acc_out[(size_t)m * N + n] = tot;
          C[(size_t)m * N + n] = (float)tot * comb;
        }
      }
    }
  }
}

// ---- few rows, quantised where they are multiplied -----------------------------------
// A workgroup takes 32 rows x 32 CT channels x up to 24 chunks of 64 k.  It asks for its f32
// rows and its weights at once, quantises the rows into LDS as the largest magnitude is known, and its eight
// wavefronts multiply: CT of them side by side, the others on further parts of K, whose sums
// meet in LDS.  What bounds it: a launch and one trip to memory (16 rows of 1536 -> 8960 6.4 us, of which an empty
// launch is 2.3; a compute unit takes in 290 KB of rows and weights).
typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef int v16i32 __attribute__((ext_vector_type(16)));
constexpr int kRowsThreads = 512, kRowsChunks = 24;
constexpr int kMaxParts = 256; // workgroups of the launch of partial maxima, four to a lane of its readers

// max(absmax / 127, 1e-10) from the partial maxima, in every wavefront by itself
__device__ __forceinline__ float scale_of_parts(const float *part, int parts) {
  const int lane = threadIdx.x & 63;
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < kMaxParts / 64; ++i)
    m = fmaxf(m, part[min(lane + 64 * i, parts - 1)]);
  const float r127 = 1.0f / 127.0f;
  return fmaxf(wave_max(m) * r127, 1e-10f);
}

// Four quantised values as bytes.  v * inv is at most 127 and some last bits of it, so 1.5 * 2^23 added
// to it leaves the nearest whole number, ties to even, in the low byte; what is not finite
// shows in bit 29 of the sum and takes the definition's way.
__device__ __forceinline__ unsigned quantise4(float4 v, float inv) {
#pragma clang fp contract(off) // the product is rounded by itself
  const float t[4] = {v.x * inv, v.y * inv, v.z * inv, v.w * inv};
  unsigned y[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    y[e] = __float_as_uint(t[e] + 12582912.0f);
  if (__builtin_expect((y[0] | y[1] | y[2] | y[3]) & 0x20000000u, 0)) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      y[e] = (unsigned)(int)fminf(fmaxf(rintf(t[e]), -128.0f), 127.0f);
  }
  const unsigned a = __builtin_amdgcn_perm(y[1], y[0], 0x0c0c0400u), b = __builtin_amdgcn_perm(y[3], y[2], 0x0c0c0400u);
  return a | b << 16;
}

// stage 2: workgroup `row` writes row `row` of the plane (zeros past M
// and K) and its step, the activation scale (1 for padding rows).  VEC: rows are read 16 bytes at a time
template <bool VEC>
__global__ void __launch_bounds__(256)
w8a8_rows_to_plane_kernel(const float *__restrict__ x, int M, int K, int Kp,
                          const float *__restrict__ part, int parts,
                          int8_t *__restrict__ plane, float *__restrict__ steps) {
  const int row = blockIdx.x;
  const float *xr = x + (int64_t)min(row, M - 1) * K;
  constexpr int kFirst = 2; // runs of four values a thread asks for ahead of the scale
  auto load = [&](int k0) {
    float4 v;
    if constexpr (VEC) {
      v = *reinterpret_cast<const float4 *>(xr + min(k0, K - 4));
    } else {
      float *p = &v.x;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        p[e] = xr[min(k0 + e, K - 1)];
    }
    return v;
  };
  float4 v[kFirst];
#pragma unroll
  for (int i = 0; i < kFirst; ++i)
    v[i] = load((threadIdx.x + 256 * i) * 4);
  const float s = scale_of_parts(part, parts);
  const float inv = 1.0f / s;
  if (threadIdx.x == 0)
    steps[row] = row < M ? s : 1.0f;
  auto put = [&](int k0, float4 q) {
    unsigned word = quantise4(q, inv);
    const int keep = row < M ? min(max(K - k0, 0), 4) : 0;
    if (keep < 4)
      word &= (1u << (8 * keep)) - 1u;
    *reinterpret_cast<unsigned *>(plane + plane_at(row, k0, 0, 1, Kp)) = word;
  };
#pragma unroll
  for (int i = 0; i < kFirst; ++i)
    if ((threadIdx.x + 256 * i) * 4 < Kp)
      put((threadIdx.x + 256 * i) * 4, v[i]);
#pragma unroll 4
  for (int k0 = (threadIdx.x + 256 * kFirst) * 4; k0 < Kp; k0 += 256 * 4)
    put(k0, load(k0));
}

struct RowsOut {
  const float *wscale;
  float *C;
  int32_t *sums;    // dense [M, N] or null
  int32_t *partial; // K in slices: [slice][M][columns of all tiles]
};

// OWN: the workgroup's rows are all of x, and so is their maximum.
template <int CT, bool OWN>
__global__ void __launch_bounds__(kRowsThreads)
w8a8_rows_kernel(const float *x, const int4 *W, const float *part, int parts, int M, int K, int N, int groups,
                 int chunks, int per_slice, int ncols, int slices, RowsOut out) {
  constexpr int kKs = 8 / CT, kPer = kRowsChunks / kKs; // parts of K, and chunks of one
  constexpr int kTile = 32 * CT, kTurn = kTile + 4;
  constexpr int kPlanes = kRowsChunks * kPlaneBlock, kSums = kKs * 32 * kTurn * 4;
  __shared__ __attribute__((aligned(16))) unsigned char lds[kPlanes > kSums ? kPlanes : kSums];
  __shared__ float red[8];
  if ((int)blockIdx.x >= ncols * slices) // padded, so that a column's row tiles share an XCD
    return;
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, up = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ctile = blockIdx.x % ncols, slice = blockIdx.x / ncols, m0 = blockIdx.y * 32;
  const int cb = slice * per_slice, nch = min(per_slice, chunks - cb); // >= 1

  // sixteen threads to a row; values beyond K repeat the last ones, and weights are zero there
  const int r = tid >> 4, j = tid & 15;
  const float *row = x + (int64_t)min(m0 + r, M - 1) * K;
  float4 v[kRowsChunks];
#pragma unroll
  for (int i = 0; i < kRowsChunks; ++i)
    v[i] = *reinterpret_cast<const float4 *>(row + min((cb + min(i, nch - 1)) * kTileK + j * 4, K - 4));
  const int c0 = wave / CT * kPer;
  const v4i32 *wp = reinterpret_cast<const v4i32 *>(W) +
                    ((size_t)min((ctile * CT + wave % CT) * 2 + ((lane >> 4) & 1), groups - 1) * chunks + cb) * 64 +
                    up * 16 + (lane & 15);
  v4i32 w[kPer][2];
#pragma unroll
  for (int c = 0; c < kPer; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      w[c][h] = wp[(size_t)min(c0 + c, nch - 1) * 64 + h * 32];
  const int row_out = tid / (kTile / 4), n = ctile * kTile + tid % (kTile / 4) * 4;
  float ws[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    ws[e] = out.wscale[min(n + e, N - 1)];
  __builtin_amdgcn_sched_barrier(0); // all of them before the first value is looked at

  float s;
  if constexpr (OWN) {
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < kRowsChunks; ++i)
      m = fmaxf(fmaxf(m, fmaxf(fabsf(v[i].x), fabsf(v[i].y))), fmaxf(fabsf(v[i].z), fabsf(v[i].w)));
    m = wave_max(m);
    if (lane == 0)
      red[wave] = m;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i)
      m = fmaxf(m, red[i]);
    const float r127 = 1.0f / 127.0f;
    s = fmaxf(m * r127, 1e-10f);
  } else {
    s = scale_of_parts(part, parts);
  }
  const float inv = 1.0f / s;
  // pieces of 16 bytes permuted by the row's number: fragment reads meet every bank once
  unsigned char *dst = lds + r * kTileK + ((j >> 2) ^ (r >> 2 & 3)) * 16 + (j & 3) * 4;
#pragma unroll
  for (int i = 0; i < kRowsChunks; ++i)
    *reinterpret_cast<unsigned *>(dst + i * kPlaneBlock) = quantise4(v[i], inv);
  __syncthreads();

  v16i32 acc{};
#pragma unroll
  for (int c = 0; c < kPer; ++c)
    if (c0 + c < nch) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const v4i32 f = *reinterpret_cast<const v4i32 *>(lds + (c0 + c) * kPlaneBlock + col * kTileK +
                                                         ((2 * h + up) ^ (col >> 2 & 3)) * 16);
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[c][h], f, acc, 0, 0, 0);
      }
    }
  __syncthreads();
  // a lane holds channels 8 q + 4 up + 0..3 of row `col`
  int *tile = reinterpret_cast<int *>(lds);
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<v4i32 *>(tile + (wave / CT * 32 + col) * kTurn + wave % CT * 32 + 8 * q + 4 * up) =
        v4i32{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  __syncthreads();
  const bool vec = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(out.C) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(out.sums) & 15) == 0;
#pragma unroll
  for (int i = 0; i < CT / 2; ++i) {
    const int rr = row_out + i * (kRowsThreads / (kTile / 4)), m = m0 + rr;
    v4i32 t{};
#pragma unroll
    for (int k = 0; k < kKs; ++k)
      t += *reinterpret_cast<const v4i32 *>(tile + (k * 32 + rr) * kTurn + tid % (kTile / 4) * 4);
    if (m >= M)
      continue;
    if (out.partial) {
      *reinterpret_cast<v4i32 *>(out.partial + ((size_t)slice * M + m) * ((size_t)ncols * kTile) + n) = t;
    } else if (vec) {
      if (n < N) {
        *reinterpret_cast<float4 *>(out.C + (size_t)m * N + n) =
            make_float4((float)t[0] * (s * ws[0]), (float)t[1] * (s * ws[1]), (float)t[2] * (s * ws[2]),
                        (float)t[3] * (s * ws[3]));
        if (out.sums)
          *reinterpret_cast<v4i32 *>(out.sums + (size_t)m * N + n) = t;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) {
          out.C[(size_t)m * N + n + e] = (float)t[e] * (s * ws[e]);
          if (out.sums)
            out.sums[(size_t)m * N + n + e] = t[e];
        }
    }
  }
}

// the slices of w8a8_rows_kernel, added as integers
__global__ void __launch_bounds__(256)
w8a8_add_slices_kernel(const int32_t *partial, const float *part, int parts, int M, int N, int columns, int slices,
                       RowsOut out) {
  const int n4 = (N + 3) / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int m = min((int)(i / n4), M - 1), n = (int)(i % n4) * 4;
  const v4i32 *p = reinterpret_cast<const v4i32 *>(partial + (size_t)m * columns + n);
  const size_t stride = (size_t)M * columns / 4;
  float ws[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    ws[e] = out.wscale[min(n + e, N - 1)];
  v4i32 t{};
  for (int sl = 0; sl < slices; sl += 6) {
    v4i32 q[6];
#pragma unroll
    for (int u = 0; u < 6; ++u)
      q[u] = p[(size_t)min(sl + u, slices - 1) * stride];
#pragma unroll
    for (int u = 0; u < 6; ++u)
      if (sl + u < slices)
        t += q[u];
  }
  const float s = scale_of_parts(part, parts);
  if (i >= (int64_t)M * n4)
    return;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n + e < N) {
      out.C[(size_t)m * N + n + e] = (float)t[e] * (s * ws[e]);
      if (out.sums)
        out.sums[(size_t)m * N + n + e] = t[e];
    }
}

BH_TILE_FAMILY(RowsFamily, "w8a8_rows_kernel"); // channel tiles side by side; whether the rows are all there are
struct RowsPlan {
  int ct = 0; // 0: another way
  int slices, per_slice, ncols, row_tiles;
};
// Workgroups of w8a8_rows_kernel have a compute unit each: while one round takes them, on tiles of 64
// channels where those still do.  us a call, before and so (as a plane -> in two rounds):
//   1536 -> 1536   8 rows 18.4 and 6.2   64 11.2 and 8.4    512 12.5 and 10.6  (700: 14.4 -> 18.5)
//   1536 -> 8960  16      32.3 and 6.4   96 11.9 and 10.3                      (128: 13.3 -> 16.7)
//   8960 -> 1536  16      171 and 10.9   64 19.1 and 13.8    96 22.3 and 15.8  (128: 20.0 -> 23.2)
// A row or two of few values are quantised by one workgroup in as much time: one row of 1536 values
// 5.3 and 6.2, two 7.7 and 6.2; one of 8960, three launches here, 15.5 and 10.4.
RowsPlan plan_rows(int64_t M, int64_t K, int64_t N) {
  RowsPlan p;
  const int64_t chunks = ceil_div(K, kTileK), rows = ceil_div(M, 32), least = ceil_div(chunks, kRowsChunks);
  if ((K & 3) != 0 || K > (1 << 17) || rows > 256 || N > (1 << 20) ||
      (M <= 16 && M * K <= (least > 1 ? 5120 : 2048)))
    return p;
  p.per_slice = (int)ceil_div(chunks, least);
  p.slices = (int)ceil_div(chunks, p.per_slice);
  p.row_tiles = (int)rows;
  for (int ct : {2, 4}) {
    p.ncols = (int)ceil_div(N, 32 * ct);
    if ((int64_t)p.ncols * p.slices * rows <= 256) {
      p.ct = ct;
      break;
    }
  }
  return p;
}

// partial maxima of n values; how many
int launch_absmax(const float *x, int64_t n, float *part, hipStream_t st) {
  const int parts = (int)std::min<int64_t>(kMaxParts, ceil_div(n, 4096)); // 16 values per thread at least
  hipLaunchKernelGGL(w8a8_absmax_parts_kernel, dim3(parts), dim3(256), 0, st, x, n, part);
  return parts;
}

// *done stays false where the other way is to be taken: nothing has been launched then
int launch_rows(const float *A, const int4 *W, const RowsOut &to, int64_t M, int64_t K, int64_t N, float *part,
                bool *done, hipStream_t st) {
  const RowsPlan p = plan_rows(M, K, N);
  if (!p.ct || (reinterpret_cast<uintptr_t>(A) & 15) != 0)
    return BUDDY_HIP_OK;
  RowsOut out = to;
  const int columns = p.ncols * 32 * p.ct;
  if (p.slices > 1) {
    char *ws = nullptr;
    if (int rc = gemm_slices_workspace(st, sizeof(int32_t) * (size_t)p.slices * M * columns, &ws))
      return rc;
    if (!ws) // under capture, and none of this size
      return BUDDY_HIP_OK;
    out.partial = reinterpret_cast<int32_t *>(ws);
  }
  const bool own = p.slices == 1 && p.row_tiles == 1;
  int parts = 1;
  if (!own)
    parts = launch_absmax(A, M * K, part, st);
  // a multiple of 8 keeps a column's row tiles on one XCD, which must have compute units for all of them:
  // 672 rows of 1536 -> 1536 padded to 16 columns were two rounds on four XCDs, 19.6 us
  const int64_t cols = (int64_t)p.ncols * p.slices, padded = round_up(cols, 8);
  const dim3 grid((unsigned)(padded * p.row_tiles <= 256 ? padded : cols), (unsigned)p.row_tiles);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kRowsThreads), 0, st, A, W, part, parts, (int)M, (int)K, (int)N,
                       (int)ceil_div(N, kTileN), (int)ceil_div(K, kTileK), p.per_slice, p.ncols, p.slices, out);
  };
  auto launch_ct = [&](auto ct) {
    constexpr int kCt = decltype(ct)::value;
    if (own) {
      BH_NOTE_VARIANT(RowsFamily, kCt, 1);
      launch(w8a8_rows_kernel<kCt, true>);
    } else {
      BH_NOTE_VARIANT(RowsFamily, kCt, 0);
      launch(w8a8_rows_kernel<kCt, false>);
    }
  };
  if (p.ct == 2)
    launch_ct(std::integral_constant<int, 2>{});
  else
    launch_ct(std::integral_constant<int, 4>{});
  if (p.slices > 1)
    hipLaunchKernelGGL(w8a8_add_slices_kernel, dim3((unsigned)ceil_div(M * ceil_div(N, 4), 256)), dim3(256), 0, st,
                       out.partial, part, parts, (int)M, (int)N, columns, p.slices, out);
  BH_CHECK_HIP(hipGetLastError());
  *done = true;
  return BUDDY_HIP_OK;
}

} // namespace
} // namespace bh

extern "C" {

size_t buddy_hip_w8a8_workspace_bytes(int64_t M, int64_t K) {
  if (M <= 0 || K <= 0)
    return 0;
  if (M <= 16)
    return (size_t)(M * bh::round_up(K, 64)) + 64;
  // the plane with its row steps, the partial maxima, the scale
  const bh::GemmStagingLayout l = bh::gemm_staging_layout(M, K);
  return l.bytes_digits(1) + sizeof(float) * (1024 + 16);
}

int buddy_hip_w8a8_matmul(const float *A, const int8_t *packed, const float *wscale,
                          float *C, int32_t *acc_out, int64_t M, int64_t K,
                          int64_t N, void *workspace, size_t workspace_bytes,
                          buddy_hip_stream stream) try {
  BH_REQUIRE(A && packed && wscale && C && workspace, "w8a8_matmul: null pointer");
  BH_REQUIRE(M >= 1 && M < (1 << 24), "w8a8_matmul: M=%lld outside 1..2^24", (long long)M);
  BH_REQUIRE(K > 0 && N > 0 && K < (1 << 30) && N < (1 << 30), "w8a8_matmul: bad shape");
  BH_REQUIRE(workspace_bytes >= buddy_hip_w8a8_workspace_bytes(M, K),
             "w8a8_matmul: workspace of %zu bytes needed, %zu given",
             buddy_hip_w8a8_workspace_bytes(M, K), workspace_bytes);
  BH_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0 &&
                 (reinterpret_cast<uintptr_t>(packed) & 15) == 0,
             "w8a8_matmul: workspace and weights must be 16-byte aligned");
  hipStream_t st = bh::as_stream(stream);
  BH_REQUIRE(M <= 16 || K <= (1 << 17), "w8a8_matmul: K=%lld above 131072 with more than 16 rows", (long long)K);
  bool done = false;
  // (the partial maxima take less than the rows do as bytes)
  if (int rc = bh::launch_rows(A, reinterpret_cast<const int4 *>(packed), {wscale, C, acc_out, nullptr}, M, K, N,
                               static_cast<float *>(workspace), &done, st))
    return rc;
  if (done)
    return BUDDY_HIP_OK;
  if (M > 16) {
    const bh::GemmStagingLayout l = bh::gemm_staging_layout(M, K);
    int8_t *plane = static_cast<int8_t *>(workspace);
    float *steps = reinterpret_cast<float *>(plane + (size_t)l.rows_padded * l.cols_padded);
    float *part = steps + l.rows_padded;
    const int parts = bh::launch_absmax(A, M * K, part, st);
    const bool vec = (K & 3) == 0 && (reinterpret_cast<uintptr_t>(A) & 15) == 0;
    hipLaunchKernelGGL(vec ? bh::w8a8_rows_to_plane_kernel<true> : bh::w8a8_rows_to_plane_kernel<false>,
                       dim3(l.rows_padded), dim3(256), 0, st, A, (int)M, (int)K, l.cols_padded, part, parts, plane,
                       steps);
    BH_CHECK_HIP(hipGetLastError());
    return bh::launch_gemm_w8a8_plane(plane, packed, wscale, C, acc_out, M, K, N, st);
  }
  const int Kp = (int)bh::round_up(K, 64);
  int8_t *xq = static_cast<int8_t *>(workspace);
  float *scale = reinterpret_cast<float *>(xq + (size_t)M * Kp);
  // the scale slot must be 4-byte aligned: M*Kp is a multiple of 64
  hipLaunchKernelGGL(bh::w8a8_quantize_kernel, dim3(1), dim3(1024), 0, st, A, M * K,
                     (int)M, (int)K, Kp, xq, scale);
  const int groups = (int)bh::ceil_div(N, 16), chunks = Kp / 64;
  const int4 *W = reinterpret_cast<const int4 *>(packed);
#define BH_W8A8(MT)                                                            \
  hipLaunchKernelGGL(bh::w8a8_gemv_kernel<MT>, dim3(groups), dim3(256), 0, st, W, \
                     xq, scale, wscale, C, acc_out, (int)M, (int)N, groups,    \
                     chunks, Kp)
  if (M == 1)
    BH_W8A8(1);
  else if (M <= 4)
    BH_W8A8(4);
  else
    BH_W8A8(16);
#undef BH_W8A8
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
} BH_CATCH_INT("buddy_hip_w8a8_matmul")
}
