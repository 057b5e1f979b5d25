// gemv_w8a32_batch.hip -- the two products of a feed-forward block for 5..16 rows, with every load of a
// workgroup on its way at once.
//
// The same arithmetic as gemv_w8a32_i8.hip: per row and 64 k a power-of-two step, three balanced
// int8 digits, exact int32 sums on v_mfma_i32_16x16x64_i8, added up in f32.  There a wavefront turns
// one 64 k after the other into digits, each a chain of LDS trips and exchanges that little else
// runs beside.  Here it asks for the rows and the weights of its whole slice of K, makes all the
// digits while the weights are on their way, and multiplies.
//
//   batch_pair_kernel   SiLU(x' . W0) * (x' . W1), K of up to 24 chunks of 64: eight wavefronts cut K
//                       between them and share P channel groups of both matrices; their sums meet
//                       in LDS.
//   batch_slice_kernel  x . W for long K and few channels: a workgroup has 128 channels and C chunks of
//                       K, whose rows it turns into digits once for all of them; its sums go to a
//                       workspace and batch_add_kernel adds the slices in order.
//
// Which products: the pair where a wavefront's slice fits its registers whole, hidden of 961 to 1536, and
// up to 16384 channels; the slices from inter = 4033 on for up to 2048 channels.  Others (4096 -> 14336 ->
// 4096, both products) go one 64 k after the other.  Blocks of 1024 to 1536 inputs and 256 to 16384
// channels, 5 to 16 rows, replayed from a graph: 1.0 to 1.46 times as fast as one 64 k after the other (1024
// x 256 and 1024 0.95 to 0.97 at 16 rows, of 9 us), and 1.0 to 1.35 of 256, 512, 1600 and 2048 inputs, whose
// down alone is cut.
//
// What bounds them: the launch, one trip to memory and the weights' way from HBM.  12 rows of
// 1536 -> 2 x 8960 10.2 us (one 64 k after the other 14.5), 8960 -> 1536 5.0 and 3.7 for the kernel that adds
// (11.4); both together in a stream 25.8 -> 19.1, at 5 rows 23.5 -> 16.9, at 16 26.7 -> 19.7.
#include "digits_dev.h"
#include "gemv_w8a32.h"

namespace bh {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * kWave;
constexpr int kPlane = 16 * kTileK; // bytes of a digit plane of 16 rows x 64 k
constexpr int kPairChunks = 3;      // chunks of a wavefront's slice, at most
constexpr int kSliceChunks = 64;    // chunks from which on K goes to several workgroups

template <int CTRL> __device__ __forceinline__ unsigned dpp_u(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
// the largest magnitude over a row of 16 lanes, each with four values, as bits: a NaN or an infinity
// wins over every finite number
__device__ __forceinline__ unsigned row16_magnitude(const f32x4 &x) {
  constexpr unsigned kAbs = 0x7fffffffu;
  unsigned m = max(max(__float_as_uint(x[0]) & kAbs, __float_as_uint(x[1]) & kAbs),
                   max(__float_as_uint(x[2]) & kAbs, __float_as_uint(x[3]) & kAbs));
  m = max(m, dpp_u<0xB1>(m));
  m = max(m, dpp_u<0x4E>(m));
  m = max(m, dpp_u<0x141>(m));
  return max(m, dpp_u<0x140>(m));
}
// the smallest power of two s, not below 2^-126, with magnitude / s < 2^22, NaN where the magnitude is
// not finite, and 1 / s
__device__ __forceinline__ void step_of(unsigned magnitude, float &step, float &inv) {
  const int e2 = max((int)(magnitude >> 23) - 127 + 1 - 22, -126);
  step = magnitude < 0x7f800000u ? __uint_as_float((unsigned)(e2 + 127) << 23) : __uint_as_float(0x7fc00000u);
  inv = __uint_as_float((unsigned)(127 - e2) << 23);
}
// Four values of row `row`, k 4 k4 .. + 3 of a chunk, as digits into the chunk's planes.  The 16-byte
// pieces of a row lie permuted by its number, so that the operand reads of 16 rows meet every bank once.
__device__ __forceinline__ int piece_at(int row, int piece) { return row * kTileK + (piece ^ (row >> 2)) * 16; }
__device__ __forceinline__ void put_digits(const f32x4 &x, float inv, unsigned char *planes, int row, int k4) {
  const float v[4] = {x[0], x[1], x[2], x[3]};
  unsigned word[3];
  digits_of(v, inv, 3, word);
  unsigned *dst = reinterpret_cast<unsigned *>(planes + piece_at(row, k4 >> 2) + (k4 & 3) * 4);
  dst[0] = word[0];
  dst[kPlane / 4] = word[1];
  dst[2 * (kPlane / 4)] = word[2];
}
// acc += step * (a tile times the planes): a lane's four channels of row lane % 16
__device__ __forceinline__ void add_tile(f32x4 &acc, const v4i &w, const v4i (&d)[3], float step) {
  const v4i zero = v4i{0, 0, 0, 0};
  const v4i r0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, d[0], zero, 0, 0, 0);
  const v4i r1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, d[1], zero, 0, 0, 0);
  const v4i r2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, d[2], zero, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int u = r0[i] + (r1[i] << 8); // |r0|, |r1| <= 2^20: exact
    acc[i] = fmaf((float)r2[i], step * 65536.0f, fmaf((float)u, step, acc[i]));
  }
}

struct PairArgs {
  const float *s0, *s1;
  float *C;
  int64_t ldc;
  float norm_eps, norm_inv_k;
  int N;
};

// Q: groups of four rows.  A group of 16 lanes has 64 k of a row.
template <int P, int Q>
__global__ void __launch_bounds__(kThreads)
batch_pair_kernel(const float *A, const int4 *W0, const int4 *W1, const float *norm_w, int lda, int K, int rows,
                  int groups, int chunks, int per, PairArgs a) {
  constexpr int C = kPairChunks, kTile = 16 * 17; // floats of a tile's sums in LDS, [channel][row]
  constexpr int kPlanes = kWaves * C * 3 * kPlane, kMeet = kWaves * 2 * P * kTile * 4;
  __shared__ __attribute__((aligned(16))) unsigned char lds[kPlanes > kMeet ? kPlanes : kMeet];
  __shared__ float step_s[kWaves][C][16], ss_s[kWaves][16];
  const int tid = threadIdx.x, lane = tid & 63, kg = lane >> 4, c16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g0 = blockIdx.x * P, c0 = wave * per, n = min(per, chunks - c0); // chunks of this slice, may be none

  f32x4 x[C][Q], nw[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int k = min((c0 + c) * kTileK + c16 * 4, K - 4);
#pragma unroll
    for (int q = 0; q < Q; ++q)
      x[c][q] = *reinterpret_cast<const f32x4 *>(A + (int64_t)min(4 * q + kg, rows - 1) * lda + k);
    nw[c] = norm_w ? *reinterpret_cast<const f32x4 *>(norm_w + k) : f32x4{1.f, 1.f, 1.f, 1.f};
  }
  v4i w[2][P][C];
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int g = 0; g < P; ++g) {
      const size_t at = ((size_t)min(g0 + g, groups - 1) * chunks + min(c0 + c, chunks - 1)) * 64 + lane;
      w[0][g][c] = __builtin_nontemporal_load(reinterpret_cast<const v4i *>(W0) + at);
      w[1][g][c] = __builtin_nontemporal_load(reinterpret_cast<const v4i *>(W1) + at);
    }
  // the results this thread finishes: channel (tid % 16) of group tid / 256 + 2 i, row tid / 16 % 16
  constexpr int kItems = (P + 1) / 2;
  float e0[kItems], e1[kItems];
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int ch = min((g0 + tid / 256 + 2 * i) * kTileN + (tid & 15), a.N - 1);
    e0[i] = a.s0[ch];
    e1[i] = a.s1[ch];
  }
  __builtin_amdgcn_sched_barrier(0); // all of them before the first value is looked at

  unsigned char *planes = lds + wave * (C * 3 * kPlane);
  float ss[Q] = {};
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const bool in = c < n && (c0 + c) * kTileK + c16 * 4 < K; // K is a multiple of four
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      f32x4 v = x[c][q];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = in ? v[e] : 0.f;
        ss[q] = fmaf(v[e], v[e], ss[q]);
        v[e] *= nw[c][e];
      }
      float step, inv;
      step_of(row16_magnitude(v), step, inv);
      put_digits(v, inv, planes + c * (3 * kPlane), 4 * q + kg, c16);
      if (c16 == 0)
        step_s[wave][c][4 * q + kg] = step;
    }
  }
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    ss[q] = row16_sum(ss[q]);
    if (c16 == 0)
      ss_s[wave][4 * q + kg] = ss[q];
  }
  // (a wavefront's own part of LDS: its operations complete in order)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  f32x4 acc[2][P];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int g = 0; g < P; ++g)
      acc[m][g] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int row = 4 * Q == 16 ? c16 : c16 & (4 * Q - 1); // columns beyond the rows repeat them
#pragma unroll
  for (int c = 0; c < C; ++c)
    if (c < n) {
      v4i d[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
        d[p] = *reinterpret_cast<const v4i *>(planes + (c * 3 + p) * kPlane + piece_at(row, kg));
      const float step = step_s[wave][c][row];
#pragma unroll
      for (int g = 0; g < P; ++g) {
        add_tile(acc[0][g], w[0][g][c], d, step);
        add_tile(acc[1][g], w[1][g][c], d, step);
      }
    }
  __syncthreads(); // the planes have been read
  float *meet = reinterpret_cast<float *>(lds);
#pragma unroll
  for (int g = 0; g < P; ++g)
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        meet[((wave * P + g) * 2 + m) * kTile + (kg * 4 + i) * 17 + c16] = acc[m][g][i];
  __syncthreads();
  const int r = tid >> 4 & 15;
  if (r >= rows)
    return;
  float rs = 1.0f;
  if (norm_w) {
    float tot = 0.f;
#pragma unroll
    for (int u = 0; u < kWaves; ++u)
      tot += ss_s[u][r];
    rs = 1.0f / sqrtf(tot * a.norm_inv_k + a.norm_eps);
  }
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int g = tid / 256 + 2 * i, ch = (g0 + g) * kTileN + (tid & 15);
    if (g >= P || ch >= a.N)
      continue;
    float v[2] = {0.f, 0.f};
#pragma unroll
    for (int u = 0; u < kWaves; ++u)
#pragma unroll
      for (int m = 0; m < 2; ++m)
        v[m] += meet[((u * P + g) * 2 + m) * kTile + (tid & 15) * 17 + r];
    const float gate = v[0] * rs * e0[i], up = v[1] * rs * e1[i];
    a.C[(int64_t)r * a.ldc + ch] = gate * (1.0f / (1.0f + expf(-gate))) * up;
  }
}

// 16 rows x 128 channels x C chunks: a thread has every 32nd run of four values of a row, so that a
// group of 16 lanes has 64 k of it; a wavefront has a channel group.
template <int C>
__global__ void __launch_bounds__(kThreads)
batch_slice_kernel(const float *A, const int4 *W, int lda, int K, int rows, int groups, int chunks, float *sums) {
  constexpr int kLoads = C / 2;
  static_assert(C % 2 == 0, "half a wavefront has two chunks of a row");
  __shared__ __attribute__((aligned(16))) unsigned char planes[C * 3 * kPlane];
  __shared__ float step_s[C][16];
  const int tid = threadIdx.x, lane = tid & 63, kg = lane >> 4, c16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c0 = blockIdx.y * C, n = min(C, chunks - c0), group = blockIdx.x * kWaves + wave;
  const int row = tid >> 5, j = tid & 31;
  f32x4 x[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i)
    x[i] = *reinterpret_cast<const f32x4 *>(A + (int64_t)min(row, rows - 1) * lda +
                                            min(c0 * kTileK + (j + 32 * i) * 4, K - 4));
  v4i w[C];
#pragma unroll
  for (int c = 0; c < C; ++c)
    w[c] = __builtin_nontemporal_load(reinterpret_cast<const v4i *>(W) +
                                      ((size_t)min(group, groups - 1) * chunks + min(c0 + c, chunks - 1)) * 64 + lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int c = 2 * i + (j >> 4);
    const bool in = (c0 + c) * kTileK + c16 * 4 < K;
    f32x4 v = x[i];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = in ? v[e] : 0.f;
    float step, inv;
    step_of(row16_magnitude(v), step, inv);
    put_digits(v, inv, planes + c * (3 * kPlane), row, c16);
    if (c16 == 0)
      step_s[c][row] = step;
  }
  __syncthreads();
  if (group >= groups)
    return;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < C; ++c)
    if (c < n) {
      v4i d[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
        d[p] = *reinterpret_cast<const v4i *>(planes + (c * 3 + p) * kPlane + piece_at(c16, kg));
      add_tile(acc, w[c], d, step_s[c][c16]);
    }
  if (c16 < rows)
    *reinterpret_cast<f32x4 *>(sums + ((size_t)blockIdx.y * rows + c16) * (groups * kTileN) + group * kTileN + kg * 4) =
        acc;
}

struct AddArgs {
  const float *scale, *bias;
  float *C;
  int64_t ldc;
  int N, accumulate;
};
__global__ void __launch_bounds__(64) batch_add_kernel(const float *sums, int slices, int rows, int groups, AddArgs a) {
  const int q = blockIdx.x * 64 + threadIdx.x, m = blockIdx.y, n = q * 4;
  if (n >= a.N)
    return;
  const float *p = sums + (size_t)m * groups * kTileN + n;
  const size_t stride = (size_t)rows * groups * kTileN;
  float *c = a.C + (int64_t)m * a.ldc + n;
  float scale[4], add[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const bool in = n + e < a.N;
    scale[e] = in ? a.scale[n + e] : 0.f;
    add[e] = !in ? 0.f : a.accumulate ? c[e] : a.bias ? a.bias[n + e] : 0.f;
  }
  f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < slices; s += 8) {
    f32x4 t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      t[u] = *reinterpret_cast<const f32x4 *>(p + (size_t)min(s + u, slices - 1) * stride);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s + u < slices)
        v += t[u];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n + e < a.N)
      c[e] = add[e] + v[e] * scale[e];
}

BH_TILE_FAMILY(PairFamily, "batch_pair_kernel");   // channel groups, groups of four rows
BH_TILE_FAMILY(SliceFamily, "batch_slice_kernel"); // chunks of a slice

template <int P, int Q> int launch_pair(const GemvArgs &g, int groups, int chunks, hipStream_t stream) {
  BH_NOTE_VARIANT(PairFamily, P, Q);
  PairArgs a;
  a.s0 = g.s0;
  a.s1 = g.s1;
  a.C = g.C;
  a.ldc = g.ldc;
  a.norm_eps = g.norm_eps;
  a.norm_inv_k = g.norm_inv_k;
  a.N = (int)g.N;
  hipLaunchKernelGGL((batch_pair_kernel<P, Q>), dim3((unsigned)ceil_div(groups, P)), dim3(kThreads), 0, stream, g.A,
                     reinterpret_cast<const int4 *>(g.W0), reinterpret_cast<const int4 *>(g.W1), g.norm_w, (int)g.lda,
                     (int)g.K, g.M, groups, chunks, (int)ceil_div(chunks, kWaves), a);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}
template <int P> int launch_pair_rows(const GemvArgs &g, int groups, int chunks, hipStream_t stream) {
  return g.M <= 8 ? launch_pair<P, 2>(g, groups, chunks, stream) : launch_pair<P, 4>(g, groups, chunks, stream);
}

template <int C>
int launch_slice(const GemvArgs &g, int groups, int chunks, int slices, float *sums, hipStream_t stream) {
  BH_NOTE_VARIANT(SliceFamily, C);
  hipLaunchKernelGGL((batch_slice_kernel<C>), dim3((unsigned)ceil_div(groups, kWaves), (unsigned)slices),
                     dim3(kThreads), 0, stream, g.A, reinterpret_cast<const int4 *>(g.W0), (int)g.lda, (int)g.K, g.M,
                     groups, chunks, sums);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

} // namespace

size_t gemv_batch_sums_bytes(int64_t M, int64_t K) {
  // at most a workgroup of 128 channels to a compute unit
  if (M < 5 || M > 16 || ceil_div(K, kTileK) < kSliceChunks)
    return 0;
  return sizeof(float) * (size_t)M * 256 * kWaves * kTileN;
}

int launch_gemv_batch(const GemvArgs &g, bool *done, hipStream_t stream) {
  *done = false;
  if (g.lda >= 1 << 30) // a row's stride is an int here
    return BUDDY_HIP_OK;
  const int groups = (int)ceil_div(g.N, kTileN), chunks = (int)ceil_div(g.K, kTileK);
  if (g.epilogue == kEpiSiluMul) {
    // a wavefront's slice fits its registers whole, and the launch is one round of the chip: as many
    // groups to a workgroup as that takes (8960 channels, 12 rows, the block: one group in three rounds 21.6
    // us, two with two workgroups to a compute unit in 128 registers 24.1, three 19.2, four 20.2)
    if (chunks < 2 * kWaves || chunks > kWaves * kPairChunks || groups > 4 * 256)
      return BUDDY_HIP_OK;
    *done = true;
    switch ((int)ceil_div(groups, 256)) {
    case 1:
      return launch_pair_rows<1>(g, groups, chunks, stream);
    case 2:
      return launch_pair_rows<2>(g, groups, chunks, stream);
    case 3:
      return launch_pair_rows<3>(g, groups, chunks, stream);
    default:
      return launch_pair_rows<4>(g, groups, chunks, stream);
    }
  }
  // long K and few channels, where the launch that adds slices is the smaller part
  if (groups > 128 || chunks < kSliceChunks || g.norm_w)
    return BUDDY_HIP_OK;
  const int columns = (int)ceil_div(groups, kWaves);
  int c = 0;
  for (int t : {4, 8, 16})
    if (!c && columns * ceil_div(chunks, t) <= 256)
      c = t;
  if (!c)
    return BUDDY_HIP_OK;
  const int slices = (int)ceil_div(chunks, c);
  if (sizeof(float) * (size_t)slices * g.M * groups * kTileN > g.sums_bytes)
    return BUDDY_HIP_OK;
  float *sums = g.sums;
  if (int rc = c == 4 ? launch_slice<4>(g, groups, chunks, slices, sums, stream)
                      : c == 8 ? launch_slice<8>(g, groups, chunks, slices, sums, stream)
                               : launch_slice<16>(g, groups, chunks, slices, sums, stream))
    return rc;
  *done = true;
  AddArgs a;
  a.scale = g.s0;
  a.bias = g.epilogue == kEpiStore ? g.bias : nullptr;
  a.C = g.C;
  a.ldc = g.ldc;
  a.N = (int)g.N;
  a.accumulate = g.epilogue == kEpiAccum;
  hipLaunchKernelGGL(batch_add_kernel, dim3((unsigned)ceil_div(g.N, 256), g.M), dim3(64), 0, stream, sums, slices, g.M,
                     groups, a);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

} // namespace bh
