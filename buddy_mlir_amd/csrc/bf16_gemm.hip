// bf16_gemm.hip -- many activation rows times resident bfloat16 matrices on the
// matrix cores: the matrix products of a prompt, plain and per expert.
//
// Weights go from memory to registers as they lie, each of the four wavefronts of a
// workgroup its own channels; the activation rows are the B operand and are shared
// through LDS.  Both are requested three steps ahead.  Up to 16 rows, and for some more
// bfloat16 ones (launch_shape), a tile of 16 channels x 32 k is the A operand as it lies, and
// f32 activations are multiplied by v_mfma_f32_16x16x4_f32; above that see
// rows_gemm_wide_kernel.
#include "bf16_linear.h"
#include "bf16_dev.h"
#include "digits_dev.h"

#include <algorithm>
#include <type_traits>

namespace bh {
namespace {

constexpr int kGemmThreads = 256;
constexpr int kWideK = 64; // k per step of the tiles of 32 rows and more
constexpr int kStages = 4;
constexpr int kRowBytes = 128;           // of one row per step
constexpr int kLdsRow = kRowBytes + 16;  // padded: rows start 4 banks apart

struct GemmDev {
  const void *A;
  void *C;
  int lda, ldc;
  int rows, K, groups; // groups of one matrix
  int ring_base, ring_mask;
  int silu_channels;
  GatedAct act;
  float limit;
  const int *counts, *lists;
  int experts, list_cap, list_div;
  int64_t expert_tiles;
};
// The same with K cut into slices (kOutF32, not grouped).  A type and an instantiation of its
// own: with these fields in every launch's arguments the launches that cut nothing took 0.3 us
// longer (1536 -> 1536, 8 bfloat16 rows: 6.9 and 7.2).
struct SlicedDev : GemmDev {
  int slice_steps;      // of a slice of k
  int64_t slice_stride; // from one slice's sums to the next in C
};
template <bool SLICED> using DevOf = std::conditional_t<SLICED, SlicedDev, GemmDev>;

template <typename T> struct ActTraits;
template <> struct ActTraits<bf16_bits> {
  static constexpr int kElems = 64, kTiles = 2; // per step: elements of a row, weight tiles
};
template <> struct ActTraits<float> {
  static constexpr int kElems = 32, kTiles = 1;
};

// the first `keep` elements of a 16-byte run, the others as zeros
template <typename T> __device__ __forceinline__ uint4 keep_run(uint4 v, int keep) {
  unsigned d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (sizeof(T) == 4)
      d[j] = j < keep ? d[j] : 0u;
    else
      d[j] = 2 * j + 1 < keep ? d[j] : 2 * j < keep ? d[j] & 0xffffu : 0u;
  }
  return uint4{d[0], d[1], d[2], d[3]};
}

template <typename T>
__device__ __forceinline__ void store4(T *p, f32x4 v);
template <> __device__ __forceinline__ void store4<float>(float *p, f32x4 v) {
  *reinterpret_cast<f32x4 *>(p) = v;
}
template <> __device__ __forceinline__ void store4<bf16_bits>(bf16_bits *p, f32x4 v) {
  *reinterpret_cast<uint2 *>(p) = uint2{pack_bf(v[0], v[1]), pack_bf(v[2], v[3])};
}

// Workgroups go to the eight dies in turn, each with an L2 of its own.  A die takes a run
// of tiles, in panels of kPanel column blocks by all row blocks: the workgroups that it
// runs at the same time share rows and channels.  Of experts' tiles the die takes a run of
// row blocks too, so that an expert's weights come to one or two L2s and not to all eight.
constexpr int kDies = 8, kPanel = 4;
__device__ __forceinline__ void place_tile(int gx, int gy, int &bx, int &by) {
  const int total = gx * gy, id = blockIdx.y * gx + blockIdx.x;
  const int die = id % kDies, q = total / kDies, r = total % kDies;
  const int t = die * q + min(die, r) + id / kDies;
  const int panel = t / (kPanel * gy), rest = t - panel * kPanel * gy;
  const int width = min(kPanel, gx - panel * kPanel);
  by = rest / width;
  bx = panel * kPanel + rest - by * width;
}

// row blocks of all experts together
__device__ __forceinline__ int count_blocks(const int *counts, int experts, int rows, int lane) {
  int n = 0;
  for (int i = lane; i < experts; i += 64)
    n += (counts[i] + rows - 1) / rows;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1)
    n += __shfl_xor(n, o, 64);
  return __builtin_amdgcn_readfirstlane(n);
}
// the expert that a row block counted over all experts belongs to; `block` becomes the one
// within it
__device__ __forceinline__ int find_expert(const int *counts, int experts, int rows, int lane,
                                           int &block) {
  for (int base = 0; base < experts; base += 64) {
    const int i = base + lane;
    const int nb = i < experts ? (counts[i] + rows - 1) / rows : 0;
    int incl = nb;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o)
        incl += v;
    }
    const unsigned long long past = __ballot(incl > block);
    if (past) {
      const int l = __builtin_ctzll(past);
      block -= __builtin_amdgcn_readlane(incl - nb, l);
      return __builtin_amdgcn_readfirstlane(base + l);
    }
    block -= __builtin_amdgcn_readlane(incl, 63);
  }
  return -1;
}

template <typename T, int GT, int OUT, bool GROUPED, bool SLICED>
__global__ void __launch_bounds__(kGemmThreads)
rows_gemm_kernel(const uint4 *__restrict__ W, int ktiles, int steps, int columns, int row_blocks,
                 DevOf<SLICED> a) {
  using Tr = ActTraits<T>;
  constexpr bool kPair = OUT == kOutExpertAct;
  constexpr int kGroups = kPair ? GT / 2 : GT; // channel groups of the result per wavefront
  constexpr int kRows = 16;
  constexpr int kRuns = kRows * 8;                               // 16-byte runs per step
  constexpr int kLoads = (kRuns + kGemmThreads - 1) / kGemmThreads;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2][kRows * kLdsRow];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  int bx, by;
  if constexpr (GROUPED) {
    const int id = blockIdx.y * columns + blockIdx.x;
    by = id / columns; // counts the row blocks of all experts
    bx = id - by * columns;
  } else {
    place_tile(columns, row_blocks, bx, by);
  }
  int row0 = by * kRows, rows = a.rows;
  const int *list = nullptr;
  if constexpr (GROUPED) {
    const int e = find_expert(a.counts, a.experts, kRows, lane, by);
    if (e < 0)
      return; // more workgroups than row blocks
    row0 = by * kRows;
    rows = a.counts[e];
    list = a.lists + (int64_t)e * a.list_cap;
    W += (int64_t)e * a.expert_tiles * 64;
  }

  // this workgroup's slice of k
  int K = a.K, first = 0;
  if constexpr (SLICED) {
    first = blockIdx.z * a.slice_steps;
    steps = min(a.slice_steps, steps - first);
    K -= first * Tr::kElems;
    a.C = static_cast<float *>(a.C) + blockIdx.z * a.slice_stride;
  }

  // the runs this thread moves: fixed rows, k advancing by the step
  const T *src[kLoads];
  int run_k[kLoads];
  int lds_at[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int c = i * kGemmThreads + tid;
    const int r = c >> 3, q = c & 7;
    run_k[i] = q * (16 / (int)sizeof(T));
    lds_at[i] = r * kLdsRow + q * 16;
    // a row past the end repeats the last one: its column of the result is not stored
    const int lr = min(row0 + r, rows - 1);
    int pr;
    if constexpr (GROUPED)
      pr = list[lr] / a.list_div;
    else
      pr = (a.ring_base + lr) & a.ring_mask;
    src[i] = static_cast<const T *>(a.A) + (int64_t)pr * a.lda + first * Tr::kElems;
  }

  const int ch0 = (bx * 4 + wave) * kGroups; // first channel group of this wavefront
  const uint4 *wp[GT];
#pragma unroll
  for (int g = 0; g < GT; ++g) {
    const int mat = kPair ? g / kGroups : 0, gg = min(ch0 + (kPair ? g % kGroups : g), a.groups - 1);
    wp[g] = W + ((int64_t)(mat * a.groups + gg) * ktiles + first * Tr::kTiles) * 64 + lane;
  }

  uint4 wr[kStages][GT * Tr::kTiles], ar[kStages][kLoads];
  constexpr int kRunElems = 16 / (int)sizeof(T);
  const int last_run = (K - 1) / kRunElems * kRunElems;
  const bool ragged = K % Tr::kElems != 0; // the last step reaches past K
  auto fetch = [&](int s, uint4 (&w)[GT * Tr::kTiles], uint4 (&x)[kLoads]) {
    const int t = min(s, steps - 1) * Tr::kTiles;
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      x[i] = *reinterpret_cast<const uint4 *>(src[i] + min(t * kBfTileK + run_k[i], last_run));
#pragma unroll
    for (int g = 0; g < GT; ++g)
#pragma unroll
      for (int u = 0; u < Tr::kTiles; ++u)
        w[g * Tr::kTiles + u] = wp[g][(int64_t)(t + u) * 64];
  };
#pragma unroll
  for (int s = 0; s < kStages - 1; ++s)
    fetch(s, wr[s], ar[s]);

  f32x4 acc[GT];
#pragma unroll
  for (int g = 0; g < GT; ++g)
    acc[g] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int frag_at = (lane & 15) * kLdsRow + (lane >> 4) * 8 * (int)sizeof(T);
  auto step = [&](int s, uint4 (&w)[GT * Tr::kTiles], uint4 (&x)[kLoads], uint4 (&w_next)[GT * Tr::kTiles],
                  uint4 (&x_next)[kLoads], unsigned char *buf) {
    if (ragged && s == steps - 1) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        x[i] = keep_run<T>(x[i], K - s * Tr::kElems - run_k[i]);
    }
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      if (kRuns % kGemmThreads == 0 || i * kGemmThreads + tid < kRuns)
        *reinterpret_cast<uint4 *>(buf + lds_at[i]) = x[i];
    fetch(s + kStages - 1, w_next, x_next);
    __syncthreads(); // the other buffer was last read before the previous barrier
#pragma unroll
    for (int t = 0; t < Tr::kTiles; ++t) {
      Frag<T> b;
      b.load(reinterpret_cast<const T *>(buf + frag_at + t * kBfTileK * (int)sizeof(T)));
#pragma unroll
      for (int g = 0; g < GT; ++g) {
        Frag<T> wf;
        if constexpr (sizeof(T) == 2)
          wf.v = w[g * Tr::kTiles + t];
        else
          wf = widen(w[g * Tr::kTiles + t]);
        acc[g] = mfma32(wf, b, acc[g]);
      }
    }
  };
  static_assert(kStages == 4, "the stages below are written out");
  int s = 0;
  for (; s + kStages <= steps; s += kStages) {
    step(s, wr[0], ar[0], wr[3], ar[3], lds[0]);
    step(s + 1, wr[1], ar[1], wr[0], ar[0], lds[1]);
    step(s + 2, wr[2], ar[2], wr[1], ar[1], lds[0]);
    step(s + 3, wr[3], ar[3], wr[2], ar[2], lds[1]);
  }
  if (s < steps)
    step(s, wr[0], ar[0], wr[3], ar[3], lds[0]);
  if (s + 1 < steps)
    step(s + 1, wr[1], ar[1], wr[0], ar[0], lds[1]);
  if (s + 2 < steps)
    step(s + 2, wr[2], ar[2], wr[1], ar[1], lds[0]);

  // a lane holds channels (lane / 16) * 4 + 0..3 of row lane % 16 of every tile
  const int lr = row0 + (lane & 15);
  if (lr >= rows)
    return;
  int orow = lr;
  if constexpr (GROUPED)
    orow = list[lr];
#pragma unroll
  for (int g = 0; g < kGroups; ++g) {
    if (ch0 + g >= a.groups)
      continue;
    const int ch = (ch0 + g) * 16 + (lane >> 4) * 4;
    f32x4 v = acc[g];
    if constexpr (OUT == kOutExpertAct) {
      const f32x4 up = acc[g + kGroups];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] = gated_act(a.act, v[j], up[j], a.limit);
      store4<T>(static_cast<T *>(a.C) + (int64_t)orow * a.ldc + ch, v);
    } else if constexpr (OUT == kOutF32) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (ch + j < a.silu_channels)
          v[j] = silu_f(v[j]);
      store4<float>(static_cast<float *>(a.C) + (int64_t)orow * a.ldc + ch, v);
    } else if constexpr (OUT == kOutAct) {
      store4<T>(static_cast<T *>(a.C) + (int64_t)orow * a.ldc + ch, v);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        store_act<T>(static_cast<T *>(a.C) + (int64_t)(ch + j) * a.ldc + orow, v[j]);
    }
  }
}

// ---- tiles of 32 rows and more -----------------------------------------------------
// The same product on v_mfma_f32_32x32x16_bf16.  A wavefront that has its SIMD to itself
// issues 16 x 16 x 32 at 22 cycles apiece (1.2 PFLOP/s of the chip), 32 x 32 x 16 at its
// 32 (1.9), with half the operand reads per product.  The A operand is 32 channels x 16 k:
// the lanes take it from the tiles of two channel groups, 512 contiguous bytes of each.
//
// f32 activations are cut into three bfloat16 terms of 8 bits each as they enter LDS,
// which is every bit of them; the weights are bfloat16 as they are.  All products are
// exact, the sums f32: three matrix instructions at sixteen times the rate of the f32
// ones.
//
// What bounds it: on tiles of 128 bfloat16 rows, two to a compute unit, a chip full of them
// multiplies at 1.0 PFLOP/s however long K is (large plain products reach 1.15), which is what
// the power allows: the clock falls with what the matrix cores draw.  A round of 24 steps is
// 43 us of that and 15 of its beginning and its activation and stores.  With the rows through
// registers, one such tile to a compute unit and its loads between its products: gate | up of 16
// experts, 2048 x 4 rows of 1536 -> 2 x 1792, 148 us, with rows by DMA 120; 777 x 1536 -> 2 x 8960
// 68 and 58.  With the activation and the stores in cheaper forms (gated_act_bf16, the turn below)
// 110 and 54.
// (Rows past the registers for the tiles of 32 and 64 rows too: 8960 -> 1536 at 777 rows 47 us
// whole, 56 so; 1536 -> 1536 of 400 rows 8.1 and 8.5.)  Against 16 x 16 tiles (us, rows x K x channels):
//   bfloat16  2048 x 4096 x 4096   82.0 -> 75.2    f32   523 -> 216
//             2048 x 1536 x 7168   72.4 -> 66.7          341 -> 154
//              777 x 8960 x 1536   60.4 -> 41.3          307 -> 115
//              777 x 1536 x 1536   13.8 -> 10.7           57 ->  23
// The f32 sums are also nearer to 64 bits (4.2e-7 against 7.0e-7 at K = 1536).

// four consecutive f32 values as three runs of bfloat16; the terms behind an infinity are
// zero, those of a NaN are NaN
__device__ __forceinline__ void split3(uint4 v, uint2 (&out)[3]) {
  const unsigned u[4] = {v.x, v.y, v.z, v.w};
  unsigned t[3][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float x = __uint_as_float(u[j]);
    const unsigned hi = u[j] & 0xffff0000u;
    const float r = __builtin_isinf(x) ? 0.f : x - __uint_as_float(hi);
    const unsigned mid = __float_as_uint(r) & 0xffff0000u;
    t[0][j] = u[j];
    t[1][j] = __float_as_uint(r);
    t[2][j] = __float_as_uint(r - __uint_as_float(mid));
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) // the upper halves of two words
    out[p] = uint2{__builtin_amdgcn_perm(t[p][1], t[p][0], 0x07060302u),
                   __builtin_amdgcn_perm(t[p][3], t[p][2], 0x07060302u)};
}

// one row times one channel in f32, until the sum is NaN; w: the channel's runs of 8 k, 16
// runs apart
__device__ __forceinline__ float f32_sum(const float *x, const uint4 *w, int K) {
  float sum = 0.f;
#pragma unroll 1
  for (int k = 0; k < K && sum == sum; k += 8) {
    const uint4 q = w[k / 8 * 16];
    const unsigned d[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (k + e < K)
        sum = fmaf(x[k + e], e & 1 ? bf_hi(d[e / 2]) : bf_lo(d[e / 2]), sum);
  }
  return sum;
}

__device__ __forceinline__ f32x16 mfma_bf16_wide(uint4 a, uint4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Tiles of 128 bfloat16 rows run two to a compute unit.
template <typename T, int RT> constexpr bool kBrings = sizeof(T) == 2 && RT == 4;

template <typename T, int RT, int GT, int OUT, bool GROUPED, bool SLICED>
__global__ void __launch_bounds__(kGemmThreads, (kBrings<T, RT> ? 2 : 1))
rows_gemm_wide_kernel(const uint4 *W, int ktiles, int steps, int columns, int row_blocks,
                      DevOf<SLICED> a) {
  constexpr bool kPair = OUT == kOutExpertAct;
  constexpr int kTilesOut = kPair ? GT / 2 : GT; // 32-channel tiles of the result per wavefront
  constexpr int kTerms = sizeof(T) == 4 ? 3 : 1;
  constexpr int kRows = 32 * RT;
  constexpr int kRunElems = 16 / (int)sizeof(T);
  constexpr int kRowRuns = kWideK / kRunElems;
  constexpr int kLoads = kRows * kRowRuns / kGemmThreads;
  constexpr int kPlane = kRows * kLdsRow, kBuf = kTerms * kPlane;
  static_assert(kRows * kRowRuns % kGemmThreads == 0, "every thread moves the same number of runs");
  constexpr int kBrought = kRows * kRowBytes; // of a step's rows, where they come past the registers
  // the way out: 32 rows of a wavefront's channels at a time are turned in LDS, so that a store writes whole row
  // segments (as the registers lie, pieces of 8 or 16 bytes of 32 rows: 777 x 1536 -> 2 x 8960 55.4 us and so 53.1,
  // experts' gate | up 114 and 109, their down 77 and 69)
  constexpr bool kTurns = OUT != kOutActTrans;
  constexpr int kOutSize = OUT == kOutF32 ? 4 : (int)sizeof(T);
  constexpr int kSegment = 32 * kTilesOut * kOutSize, kTurnRow = kSegment + 16;
  constexpr int kTurn = kTurns ? 4 * 32 * kTurnRow : 0, kStage = kBrings<T, RT> ? 4 * kBrought : 3 * kBuf;
  __shared__ __attribute__((aligned(16))) unsigned char lds[kStage > kTurn ? kStage : kTurn];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  int bx, by;
  if constexpr (!GROUPED)
    place_tile(columns, row_blocks, bx, by);
  int row0, rows = a.rows;
  const int *list = nullptr;
  if constexpr (GROUPED) {
    const int blocks = count_blocks(a.counts, a.experts, kRows, lane);
    if ((int)(blockIdx.y * columns + blockIdx.x) >= blocks * columns)
      return; // more workgroups than tiles
    place_tile(columns, blocks, bx, by);
    const int e = find_expert(a.counts, a.experts, kRows, lane, by);
    if (e < 0)
      return;
    rows = a.counts[e];
    list = a.lists + (int64_t)e * a.list_cap;
    W += (int64_t)e * a.expert_tiles * 64;
  }
  row0 = by * kRows;
  // this workgroup's slice of k
  int K = a.K, first = 0;
  if constexpr (SLICED) {
    first = blockIdx.z * a.slice_steps;
    steps = min(a.slice_steps, steps - first);
    K -= first * kWideK;
    a.C = static_cast<float *>(a.C) + blockIdx.z * a.slice_stride;
  }

  const int ch0 = (bx * 4 + wave) * kTilesOut * 2; // first channel group of this wavefront
  const uint4 *wp[GT];
#pragma unroll
  for (int g = 0; g < GT; ++g) {
    const int mat = kPair ? g / kTilesOut : 0;
    const int gg = min(ch0 + 2 * (kPair ? g % kTilesOut : g) + ((lane >> 4) & 1), a.groups - 1);
    wp[g] = W + ((int64_t)(mat * a.groups + gg) * ktiles + first * 2) * 64 + (lane >> 5) * 16 + (lane & 15);
  }

  f32x16 acc[GT][RT];
#pragma unroll
  for (int g = 0; g < GT; ++g)
#pragma unroll
    for (int r = 0; r < RT; ++r)
      acc[g][r] = f32x16{};

  if constexpr (kBrings<T, RT>) {
    // Rows come to LDS past the registers, three steps ahead, weights a quarter of a step (16 k) at
    // a time, seven of them ahead: 256 registers a wavefront.  LDS holds rows of 128 bytes whose
    // eight 16-byte pieces are permuted by the row's number (piece p of row r where p ^ (r / 2 % 8)
    // would be), so that the fragments of sixteen rows in a line meet every bank once.
    // A step issues GT loads of weights in each quarter and RT into LDS, one ahead of those of each of
    // its four quarters.  What K has beyond whole steps follows at the end, on its own.
    constexpr int kAhead = 7, kSlots = 8;
    const int whole = min(steps, K / kWideK);
    const int f = ((wave & 1) * 4 + (lane >> 4)) & 7;
    const char *src[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int lr = min(row0 + (i * 4 + wave) * 8 + (lane >> 3), rows - 1);
      int pr;
      if constexpr (GROUPED)
        pr = list[lr] / a.list_div;
      else
        pr = (a.ring_base + lr) & a.ring_mask;
      src[i] = static_cast<const char *>(a.A) + ((int64_t)pr * a.lda + first * kWideK) * 2 + ((lane & 7) ^ f) * 16;
    }
    const unsigned lds0 = (unsigned)__builtin_amdgcn_readfirstlane(
        (int)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds);
    auto bring = [&](int s, int buf, int i) {
      load_1k_to_lds(src[i] + (int64_t)min(s, whole - 1) * kRowBytes, lds0 + buf * kBrought + (i * 4 + wave) * 1024);
    };
    uint4 wr[kSlots][GT];
    auto fetch = [&](int q, uint4 (&w)[GT]) { // quarter q of all
#pragma unroll
      for (int g = 0; g < GT; ++g)
        w[g] = wp[g][(int64_t)min(q, 4 * whole - 1) * 32];
    };
    int frag_at[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      frag_at[u] = (lane & 31) * kRowBytes + ((2 * u + (lane >> 5)) ^ ((lane >> 1) & 7)) * 16;
    uint4 frag[2][RT];
    auto load_frag = [&](int buf, int u, uint4 (&x)[RT]) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
        x[r] = *reinterpret_cast<const uint4 *>(lds + buf * kBrought + r * 32 * kRowBytes + frag_at[u]);
    };
    auto multiply = [&](const uint4 (&w)[GT], const uint4 (&x)[RT]) {
#pragma unroll
      for (int g = 0; g < GT; ++g)
#pragma unroll
        for (int r = 0; r < RT; ++r)
          acc[g][r] = mfma_bf16_wide(w[g], x[r], acc[g][r]);
    };
    if (whole > 0) {
#pragma unroll
      for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int i = 0; i < RT; ++i)
          bring(s, s, i);
#pragma unroll
      for (int q = 0; q < kAhead; ++q)
        fetch(q, wr[q]);
      landed<RT + kAhead * GT>(); // steps 0 and 1
      __syncthreads();
      load_frag(0, 0, frag[0]);
      // step s0 + slot: from buffer `slot`; step s + 3 goes into the one before it
      auto step = [&](int s0, auto slot) {
        constexpr int sl = slot;
        const int s = s0 + sl;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          load_frag(u < 3 ? sl : (sl + 1) & 3, (u + 1) & 3, frag[(u + 1) & 1]);
          bring(s + 3, (sl + 3) & 3, u);
          fetch(4 * s + u + kAhead, wr[(4 * sl + u + kAhead) % kSlots]);
          __builtin_amdgcn_sched_barrier(0);
          multiply(wr[(4 * sl + u) % kSlots], frag[u & 1]);
          __builtin_amdgcn_sched_barrier(0);
        }
        landed<GT + 4 * (1 + GT)>(); // step s + 2, whose last load is in quarter 3 of step s - 1
        __syncthreads();
      };
      using std::integral_constant;
      int s = 0;
      for (; s + 4 <= whole; s += 4) {
        step(s, integral_constant<int, 0>{});
        step(s, integral_constant<int, 1>{});
        step(s, integral_constant<int, 2>{});
        step(s, integral_constant<int, 3>{});
      }
      if (s < whole) {
        step(s, integral_constant<int, 0>{});
        if (s + 1 < whole) {
          step(s, integral_constant<int, 1>{});
          if (s + 2 < whole)
            step(s, integral_constant<int, 2>{});
        }
      }
      landed<0>(); // steps asked for beyond the last
      __syncthreads();
    }
    if (whole < steps) { // the rest of K
      const int r0 = tid / kRowRuns, q = tid % kRowRuns, k = whole * kWideK + q * kRunElems;
      const int last_run = (K - 1) / kRunElems * kRunElems;
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        const int r = r0 + i * (kGemmThreads / kRowRuns), lr = min(row0 + r, rows - 1);
        int pr;
        if constexpr (GROUPED)
          pr = list[lr] / a.list_div;
        else
          pr = (a.ring_base + lr) & a.ring_mask;
        const T *p = static_cast<const T *>(a.A) + (int64_t)pr * a.lda + first * kWideK;
        const uint4 x = keep_run<T>(*reinterpret_cast<const uint4 *>(p + min(k, last_run)), K - k);
        *reinterpret_cast<uint4 *>(lds + r * kRowBytes + (q ^ (r >> 1 & 7)) * 16) = x;
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        uint4 w[GT];
#pragma unroll
        for (int g = 0; g < GT; ++g)
          w[g] = wp[g][(int64_t)(4 * whole + u) * 32];
        load_frag(0, u, frag[0]);
        multiply(w, frag[0]);
      }
    }
  } else {
    // the runs this thread moves: fixed rows, k advancing by the step
    const T *src[kLoads];
    int lds_at[kLoads];
    const int run_k = tid % kRowRuns * kRunElems;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int r = (i * kGemmThreads + tid) / kRowRuns;
      lds_at[i] = r * kLdsRow + run_k * 2;
      // a row past the end repeats the last one: its column of the result is not stored
      const int lr = min(row0 + r, rows - 1);
      int pr;
      if constexpr (GROUPED)
        pr = list[lr] / a.list_div;
      else
        pr = (a.ring_base + lr) & a.ring_mask;
      src[i] = static_cast<const T *>(a.A) + (int64_t)pr * a.lda + first * kWideK;
    }

    uint4 wr[4][GT * 4], xr[4][kLoads];
    const int last_run = (K - 1) / kRunElems * kRunElems;
    const bool ragged = K % kWideK != 0; // the last step reaches past K
    auto fetch_w = [&](int s, uint4 (&w)[GT * 4]) {
      const int t = min(s, steps - 1) * 2;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int g = 0; g < GT; ++g)
          w[g * 4 + u] = wp[g][(int64_t)(t + u / 2) * 64 + (u & 1) * 32];
    };
    auto fetch_x = [&](int s, uint4 (&x)[kLoads]) {
      const int k = min(min(s, steps - 1) * kWideK + run_k, last_run);
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        x[i] = *reinterpret_cast<const uint4 *>(src[i] + k);
    };
    auto put_x = [&](int s, uint4 (&x)[kLoads], unsigned char *buf) {
      if (ragged && s == steps - 1) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i)
          x[i] = keep_run<T>(x[i], K - s * kWideK - run_k);
      }
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        if constexpr (kTerms == 1) {
          *reinterpret_cast<uint4 *>(buf + lds_at[i]) = x[i];
        } else {
          uint2 t[3];
          split3(x[i], t);
#pragma unroll
          for (int p = 0; p < 3; ++p)
            *reinterpret_cast<uint2 *>(buf + p * kPlane + lds_at[i]) = t[p];
        }
      }
    };

    const int frag_at = (lane & 31) * kLdsRow + (lane >> 5) * 16;
    uint4 frag[2][kTerms][RT];
    auto load_frag = [&](const unsigned char *buf, int u, uint4 (&f)[kTerms][RT]) {
#pragma unroll
      for (int p = 0; p < kTerms; ++p)
#pragma unroll
        for (int r = 0; r < RT; ++r)
          f[p][r] = *reinterpret_cast<const uint4 *>(buf + p * kPlane + frag_at + r * 32 * kLdsRow + u * 32);
    };

    // Step s multiplies buffer s % 3, whose first fragments were read during step s - 1, and
    // fills buffer (s + 2) % 3, last read before the previous barrier.
    unsigned char *cur = lds, *next = lds + kBuf, *fill = lds + 2 * kBuf;
    fetch_x(0, xr[0]);
    fetch_x(1, xr[1]);
    fetch_w(0, wr[0]);
    fetch_x(2, xr[2]);
    fetch_w(1, wr[1]);
    fetch_x(3, xr[3]);
    fetch_w(2, wr[2]);
    put_x(0, xr[0], cur);
    put_x(1, xr[1], next);
    fetch_x(4, xr[0]);
    __syncthreads();
    load_frag(cur, 0, frag[0]);
    auto step = [&](int s, uint4 (&w)[GT * 4], uint4 (&w_new)[GT * 4], uint4 (&x)[kLoads],
                    uint4 (&x_new)[kLoads]) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        // the next fragments are asked for ahead of the products that cover their way, and
        // stay there: left to itself the scheduler moves them to their use
        load_frag(u < 3 ? cur : next, (u + 1) & 3, frag[(u + 1) & 1]);
        // the step's loads in two parts (evenly between its products 91.4 us against 90.4 for an
        // experts' way back: several workgroups of a compute unit hide each other's)
        if (u == 0)
          fetch_w(s + 3, w_new);
        if (u == 2)
          fetch_x(s + 5, x_new);
        if (u == 1)
          put_x(s + 2, x, fill);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = kTerms - 1; p >= 0; --p)
#pragma unroll
          for (int g = 0; g < GT; ++g)
#pragma unroll
            for (int r = 0; r < RT; ++r)
              acc[g][r] = mfma_bf16_wide(w[g * 4 + u], frag[u & 1][p][r], acc[g][r]);
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      unsigned char *t = cur;
      cur = next;
      next = fill;
      fill = t;
    };
    int s = 0;
    for (; s + 4 <= steps; s += 4) {
      step(s, wr[0], wr[3], xr[2], xr[1]);
      step(s + 1, wr[1], wr[0], xr[3], xr[2]);
      step(s + 2, wr[2], wr[1], xr[0], xr[3]);
      step(s + 3, wr[3], wr[2], xr[1], xr[0]);
    }
    if (s < steps)
      step(s, wr[0], wr[3], xr[2], xr[1]);
    if (s + 1 < steps)
      step(s + 1, wr[1], wr[0], xr[3], xr[2]);
    if (s + 2 < steps)
      step(s + 2, wr[2], wr[1], xr[0], xr[3]);
  }

  __syncthreads(); // LDS is free
  // a lane holds channels 8 j + (lane / 32) * 4 + 0..3, j = 0..3, of row lane % 32 of every tile
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int lr = row0 + r * 32 + (lane & 31);
    if (kTerms > 1 && lr < rows) {
      // An infinite weight times a term that is zero is NaN where the f32 product is
      // infinite: what came out as NaN is added up again without terms.
      float most = acc[0][r][0]; // NaN if one of them is
#pragma unroll
      for (int n = 1; n < GT * 16; ++n)
        most = __builtin_elementwise_maximum(most, acc[n / 16][r][n % 16]);
      if (most != most) {
        int pr;
        if constexpr (GROUPED)
          pr = list[lr] / a.list_div;
        else
          pr = (a.ring_base + lr) & a.ring_mask;
        const float *x = static_cast<const float *>(a.A) + (int64_t)pr * a.lda + first * kWideK;
#pragma unroll 1
        for (int n = 0; n < GT * 16; ++n) {
          float v = 0.f;
#pragma unroll
          for (int i = 0; i < GT * 16; ++i)
            v = i == n ? acc[i / 16][r][i % 16] : v;
          const int tile = n / 16, of = 8 * (n % 16 / 4) + (lane >> 5) * 4 + n % 4; // of 32 channels
          const int group = ch0 + 2 * (kPair ? tile % kTilesOut : tile) + of / 16;
          if (v == v || group >= a.groups)
            continue;
          const int64_t w_at = (int64_t)((kPair ? tile / kTilesOut : 0) * a.groups + group) * ktiles + first * 2;
          const uint4 *w = W + w_at * 64 + of % 16;
          v = f32_sum(x, w, SLICED ? min(K, steps * kWideK) : K);
#pragma unroll
          for (int i = 0; i < GT * 16; ++i)
            acc[i / 16][r][i % 16] = i == n ? v : acc[i / 16][r][i % 16];
        }
      }
    }
    if constexpr (kTurns) {
      unsigned char *turn = lds + wave * (32 * kTurnRow);
#pragma unroll
      for (int g = 0; g < kTilesOut; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int ch = 32 * g + 8 * j + (lane >> 5) * 4;
          f32x4 v;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v[i] = acc[g][r][4 * j + i];
            if constexpr (OUT == kOutExpertAct) {
              const float up = acc[g + kTilesOut][r][4 * j + i];
              v[i] = sizeof(T) == 2 ? gated_act_bf16(a.act, v[i], up, a.limit) : gated_act(a.act, v[i], up, a.limit);
            } else if constexpr (OUT == kOutF32) {
              if (ch0 * 16 + ch + i < a.silu_channels)
                v[i] = silu_f(v[i]);
            }
          }
          unsigned char *to = turn + (lane & 31) * kTurnRow + ch * kOutSize;
          if constexpr (kOutSize == 4)
            *reinterpret_cast<f32x4 *>(to) = v;
          else
            *reinterpret_cast<uint2 *>(to) = uint2{pack_bf(v[0], v[1]), pack_bf(v[2], v[3])};
        }
      lds_turn();
      constexpr int kPieces = kSegment / 16; // of a row
#pragma unroll
      for (int i = 0; i < kPieces / 2; ++i) {
        const int id = i * 64 + lane, row = id / kPieces, ch = id % kPieces * (16 / kOutSize);
        const int out = row0 + r * 32 + row;
        const uint4 x = *reinterpret_cast<const uint4 *>(turn + row * kTurnRow + ch * kOutSize);
        if (out >= rows || ch0 * 16 + ch >= a.groups * 16)
          continue;
        int orow = out;
        if constexpr (GROUPED)
          orow = list[out];
        unsigned char *to = static_cast<unsigned char *>(a.C) + ((int64_t)orow * a.ldc + ch0 * 16 + ch) * kOutSize;
        *reinterpret_cast<uint4 *>(to) = x;
      }
      lds_turn();
    } else if (lr < rows) {
#pragma unroll
      for (int g = 0; g < kTilesOut; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int ch = (ch0 + 2 * g) * 16 + 8 * j + (lane >> 5) * 4;
          if (ch >= a.groups * 16)
            continue;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            store_act<T>(static_cast<T *>(a.C) + (int64_t)(ch + i) * a.ldc + lr, acc[g][r][4 * j + i]);
        }
    }
  }
}

template <int ROWS, int CHANNELS, bool GROUPED, bool SLICED, typename F>
int launch_tiles(F kernel, int elems, const RowsGemm &a, hipStream_t stream) {
  DevOf<SLICED> d{};
  d.A = a.A;
  d.C = a.C;
  d.lda = a.lda;
  d.ldc = a.ldc;
  d.rows = a.rows;
  d.K = a.W.K;
  d.groups = a.W.groups();
  d.ring_base = a.ring_base;
  d.ring_mask = a.ring_mask;
  d.silu_channels = a.silu_channels;
  d.act = a.act;
  d.limit = a.limit;
  d.counts = a.counts;
  d.lists = a.lists;
  d.experts = a.experts;
  d.list_cap = a.list_cap;
  d.list_div = a.list_div;
  d.expert_tiles = a.expert_tiles;
  const int steps = (int)ceil_div(a.W.K, elems);
  unsigned slices = 1;
  if constexpr (SLICED) { // slices of equal steps but the last, none of them empty
    d.slice_steps = (int)ceil_div(ceil_div(a.W.K, kWideK), a.slices) * (kWideK / elems);
    d.slice_stride = a.slice_stride;
    slices = (unsigned)ceil_div(steps, d.slice_steps);
  }
  const int64_t blocks = GROUPED ? std::min<int64_t>(ceil_div(a.list_total, ROWS) + a.experts,
                                                     a.list_total)
                                 : ceil_div(a.rows, ROWS);
  const int64_t columns = ceil_div(d.groups * 16, CHANNELS);
  BH_REQUIRE(blocks * columns < (int64_t)1 << 31, "rows_gemm: %lld row blocks", (long long)blocks);
  // The second dimension of a grid ends at 65535 (2.1 million rows in tiles of 32): then all
  // in the first.  (Always so, launches of 4 us took 0.2 longer.)
  const dim3 grid = blocks <= 65535 ? dim3((unsigned)columns, (unsigned)blocks, slices)
                                    : dim3((unsigned)(blocks * columns), 1, slices);
  hipLaunchKernelGGL(kernel, grid, dim3(kGemmThreads), 0, stream, a.W.tiles,
                     a.W.ktiles, steps, (int)columns, (int)blocks, d);
  BH_CHECK_HIP(hipGetLastError());
  return BUDDY_HIP_OK;
}

BH_TILE_FAMILY(RowsFamily, "rows_gemm_kernel");
BH_TILE_FAMILY(WideFamily, "rows_gemm_wide_kernel");
// ... and those of them whose K was cut
BH_TILE_FAMILY(RowsSlicesFamily, "rows_gemm_kernel slices");
BH_TILE_FAMILY(WideSlicesFamily, "rows_gemm_wide_kernel slices");

// 16 rows, GT channel groups per wavefront (pairs count twice).  CUT: K may be in slices.
template <typename T, int GT, int OUT, bool GROUPED, bool CUT>
int launch_flat(const RowsGemm &a, hipStream_t stream) {
  BH_NOTE_VARIANT(RowsFamily, sizeof(T) == 4, GT, OUT, GROUPED);
  auto run = [&](auto sliced) {
    constexpr bool S = sliced;
    return launch_tiles<16, 64 * (OUT == kOutExpertAct ? GT / 2 : GT), GROUPED, S>(
        rows_gemm_kernel<T, GT, OUT, GROUPED, S>, ActTraits<T>::kElems, a, stream);
  };
  if constexpr (CUT)
    if (a.slices > 1) {
      BH_NOTE_VARIANT(RowsSlicesFamily, sizeof(T) == 4, GT);
      return run(std::true_type{});
    }
  return run(std::false_type{});
}
// RT tiles of 32 rows, GT tiles of 32 channels per wavefront
template <typename T, int RT, int GT, int OUT, bool GROUPED, bool CUT>
int launch_wide(const RowsGemm &a, hipStream_t stream) {
  BH_NOTE_VARIANT(WideFamily, sizeof(T) == 4, RT, GT, OUT, GROUPED);
  auto run = [&](auto sliced) {
    constexpr bool S = sliced;
    return launch_tiles<32 * RT, 128 * (OUT == kOutExpertAct ? GT / 2 : GT), GROUPED, S>(
        rows_gemm_wide_kernel<T, RT, GT, OUT, GROUPED, S>, kWideK, a, stream);
  };
  if constexpr (CUT)
    if (a.slices > 1) {
      BH_NOTE_VARIANT(WideSlicesFamily, sizeof(T) == 4, RT, GT);
      return run(std::true_type{});
    }
  return run(std::false_type{});
}

// Up to 16 rows the product is bound by the weights: 16-row tiles, wide ones where they
// still fill the 256 compute units.  Above that the tile with the lowest estimate: tiles
// per compute unit x steps of 64 k x what a step of such a tile takes (us, measured with
// K of 1536 to 8960 on full and on partly filled chips; those of 128 rows fitted again to
// nine matrices at 24 to 2048 rows, of which the picks are 0.6 % off the best tile on average),
// plus what a tile takes to begin and to store.  Tiles of 16 rows x 64 channels stay the best of few rows, whose
// launches are bound by how many compute units ask for the weights (bfloat16, us against
// 32 or 64 x 128): 8960 -> 1536 at 24 rows 21.2 vs 28.4, at 150 22.7 vs 31.3, at 220 36.0
// vs 31.5; 1536 -> 1536 at 64 rows 5.6 vs 6.9; 1536 -> 17920 at 64 rows 18.4 vs 12.4.  In
// f32, whose three terms make the products the longer part, they gain nothing.
// What slices cost besides their bytes, in the norm that adds them: with half of that, products of
// 256 to 1024 inputs were cut whose prompts then took 1 to 2 % longer (Lirulix of width 256, 64 bfloat16
// tokens: 221.6 us whole, 226.5 cut).
constexpr double kSliceUs = 1.0;
// Tiles of 128 bfloat16 rows go two to a compute unit: rounds of 512, of which a last one of up to 256 has
// them alone.  Of 360 products of 256 to 14336 inputs and channels and 96 to 4096 rows the picks are 0.05 %
// off the best tile on average and at most 4 (with rounds of 256 at 0.68 us a step, as gate | up and
// experts have them, 0.3 and 20: 600 rows of 4096 -> 14336, 280 tiles, 113 us and 94 on tiles of 64 rows).
inline double shared_us(int64_t tiles, int64_t steps) {
  const double alone = 0.65 * (double)steps, both = 1.45 * (double)steps;
  const int64_t left = tiles % 512;
  return (double)(tiles / 512) * both + (left == 0 ? 0.0 : left <= 256 ? alone : both) + 6.0;
}
template <typename T, int OUT, bool GROUPED>
int launch_shape(const RowsGemm &a, hipStream_t stream, int *slices) {
  const int64_t rows = GROUPED ? ceil_div(a.list_total, a.experts) : a.rows;
  const int64_t all_blocks = GROUPED ? std::min<int64_t>(a.experts, a.list_total) : 1;
  constexpr bool kPair = OUT == kOutExpertAct;
  constexpr int P = kPair ? 2 : 1; // groups come in pairs
  constexpr bool CUT = OUT == kOutF32 && !GROUPED;
  auto workgroups = [&](int rt, int ch) {
    return ceil_div(a.W.N, ch) * ceil_div(rows, rt) * all_blocks;
  };
  if (rows <= 16) {
    RowsGemm b = a;
    b.slices = 1;
    return workgroups(16, 128) >= 256 ? launch_flat<T, 2 * P, OUT, GROUPED, false>(b, stream)
                                      : launch_flat<T, P, OUT, GROUPED, false>(b, stream);
  }
  // With slices of k that the caller adds: the tile and the number of slices together, which
  // cost the bytes of their sums.  8960 -> 1536: 777 bfloat16 rows 50 us whole and 38 in three slices,
  // 300 f32 rows 72 and 36 in four; Lirulix prompts of 17 to 450 tokens at width 1536 1.07 to 1.2
  // times as fast in bfloat16, 1.1 to 1.46 in f32.
  const int64_t steps = ceil_div(a.W.K, kWideK);
  int cut = 1; // slices of the estimate that was the lowest of a tile
  struct Cost {
    double us;
    int slices;
    bool operator<=(const Cost &o) const { return us <= o.us; }
    bool operator<(const Cost &o) const { return us < o.us; }
  };
  auto cost_by = [&](int rt, int ch, auto time) {
    Cost best{1e30, 1};
    for (int s = 1; s <= a.slices; ++s) {
      const int64_t per = ceil_div(steps, s);
      if (ceil_div(steps, per) != s)
        continue; // the last slice would be empty
      const double us = time(workgroups(rt, ch / P) * s, per) +
                        (s - 1) * 8e-6 / 4.8 * (double)rows * a.W.N + (s > 1 ? kSliceUs : 0.0);
      if (us < best.us)
        best = {us, s};
    }
    return best;
  };
  auto cost = [&](int rt, int ch, double step_us, double fixed_us) {
    return cost_by(rt, ch, [=](int64_t tiles, int64_t per) {
      return (double)(ceil_div(tiles, 256) * per) * step_us + fixed_us;
    });
  };
  auto with = [&](const Cost &c) {
    cut = c.slices;
    RowsGemm b = a;
    b.slices = cut;
    return b;
  };
  auto done = [&](int rc) {
    if (slices)
      *slices = cut;
    return rc;
  };
  if constexpr (sizeof(T) == 4) {
    const Cost wide = cost(32, 256, 0.80, 4.5);
    if constexpr (!kPair) {
      const Cost low = cost(32, 128, 0.46, 4.0);
      if (low <= wide)
        return done(launch_wide<T, 1, 1, OUT, GROUPED, CUT>(with(low), stream));
    }
    return done(launch_wide<T, 1, 2, OUT, GROUPED, CUT>(with(wide), stream));
  } else {
    // few rows: 16-row tiles of 64 channels, while they are few rounds of the chip
    const Cost tall = kPair || GROUPED ? cost(128, 256, 0.68, 7.0) : cost_by(128, 256, shared_us),
               flat = cost(16, 64 * P, 0.13 * P, 2.5);
    Cost half, low;
    if constexpr (kPair) {
      // fewer workgroups than half the chip draw the weights from memory too slowly
      auto thin = [&](int rt) { return workgroups(rt, 128) < 128 ? 6.0 : 0.0; };
      half = cost(64, 256, 0.60, 5.0);
      half.us += thin(64);
      low = cost(32, 256, 0.40, 4.0);
      low.us += thin(32);
    } else {
      half = cost(64, 128, 0.29, 4.5);
      low = cost(32, 128, 0.21, 4.0);
    }
    if (flat <= std::min({tall, half, low}))
      return done(launch_flat<T, P, OUT, GROUPED, CUT>(with(flat), stream));
    if (tall <= std::min(half, low))
      return done(launch_wide<T, 4, 2, OUT, GROUPED, CUT>(with(tall), stream));
    constexpr int GT = kPair ? 2 : 1;
    return done(half <= low ? launch_wide<T, 2, GT, OUT, GROUPED, CUT>(with(half), stream)
                            : launch_wide<T, 1, GT, OUT, GROUPED, CUT>(with(low), stream));
  }
}

template <typename T> int launch_typed(const RowsGemm &a, hipStream_t stream, int *slices) {
  const bool grouped = a.counts != nullptr;
  switch (a.out) {
  case kOutF32:
    return grouped ? launch_shape<T, kOutF32, true>(a, stream, slices)
                   : launch_shape<T, kOutF32, false>(a, stream, slices);
  case kOutAct:
    BH_REQUIRE(!grouped, "rows_gemm: form not compiled for expert lists");
    return launch_shape<T, kOutAct, false>(a, stream, slices);
  case kOutActTrans:
    BH_REQUIRE(!grouped, "rows_gemm: form not compiled for expert lists");
    return launch_shape<T, kOutActTrans, false>(a, stream, slices);
  case kOutExpertAct:
    return grouped ? launch_shape<T, kOutExpertAct, true>(a, stream, slices)
                   : launch_shape<T, kOutExpertAct, false>(a, stream, slices);
  }
  return fail(BUDDY_HIP_ERR_ARG, "rows_gemm: output form %d", (int)a.out);
}

} // namespace

int launch_rows_gemm(const RowsGemm &a, hipStream_t stream, int *slices) {
  const Bf16Matrix &W = a.W;
  BH_REQUIRE(W.tiles && W.K > 0 && W.N > 0 && W.N % 16 == 0 && W.ktiles == bf16_ktiles(W.K) &&
                 a.A && a.C && a.rows >= 0,
             "rows_gemm: bad argument");
  // rows are read 16 bytes at a time up to the run that holds element K - 1
  BH_REQUIRE(a.lda % 8 == 0 && a.lda >= round_up(W.K, 8) && ((uintptr_t)a.A & 15) == 0,
             "rows_gemm: activation rows must be 16-byte aligned (lda %d, K %d)", a.lda, W.K);
  BH_REQUIRE(((uintptr_t)a.C & 15) == 0 &&
                 (a.out == kOutActTrans ? a.ldc >= a.rows
                                         : (a.ldc % (a.out == kOutF32 ? 4 : 8) == 0 && a.ldc >= W.N)),
             "rows_gemm: result rows (ldc %d, N %d)", a.ldc, W.N);
  BH_REQUIRE(!a.counts || (a.lists && a.experts > 0 && a.list_cap > 0 && a.list_div > 0),
             "rows_gemm: expert lists");
  BH_REQUIRE(a.slices >= 1 && (a.slices == 1 || (slices && a.out == kOutF32 && !a.silu_channels && !a.counts &&
                                                 a.slice_stride >= (int64_t)a.rows * a.ldc && a.slice_stride % 4 == 0)),
             "rows_gemm: slices of k");
  if (slices)
    *slices = 1;
  if (a.counts ? a.list_total == 0 : a.rows == 0)
    return BUDDY_HIP_OK;
  return a.f32 ? launch_typed<float>(a, stream, slices) : launch_typed<bf16_bits>(a, stream, slices);
}

} // namespace bh

extern "C" {

int buddy_hip_gemm_bf16(const void *A, int64_t lda, int dtype, const void *tiles, float *C,
                        int64_t ldc, int64_t M, int64_t K, int64_t N, buddy_hip_stream stream) try {
  BH_REQUIRE(A && tiles && C && M > 0 && K > 0 && N > 0 && M < (1 << 30) && K < (1 << 30) &&
                 N < (1 << 30) && lda < (1 << 30) && ldc < (1 << 30) &&
                 (dtype == BUDDY_HIP_MODEL_BF16 || dtype == BUDDY_HIP_MODEL_F32),
             "gemm_bf16: bad argument");
  bh::RowsGemm g;
  g.W.tiles = static_cast<const uint4 *>(tiles);
  g.W.K = (int)K;
  g.W.N = (int)bh::round_up(N, 16);
  g.W.ktiles = bh::bf16_ktiles(K);
  g.A = A;
  g.lda = (int)lda;
  g.f32 = dtype == BUDDY_HIP_MODEL_F32;
  g.rows = (int)M;
  g.C = C;
  g.ldc = (int)ldc;
  return bh::launch_rows_gemm(g, bh::as_stream(stream));
} BH_CATCH_INT("buddy_hip_gemm_bf16")
}
