// attn_terms.h -- keys, values, queries and weights of a prompt's attention as float16 terms.
//
// A row of 128 values is brought to a largest magnitude of 2^14 .. 2^15 by a power of two of its own; an f32
// value is then the sum of two float16 ones, rounded to nearest, 2^-23 of it off at most (a row's small values 2^-40
// of its largest one).  Of the four products of two such sums the one of two second terms, 2^-22 at most, is left
// out; the others are exact, all summed in f32.
//
// The rows of values whose keys share a sum must not be scaled too differently: a weight is held times its row's
// scale, and the sum of the weights as those are (tile_weights).  Scales end at 2^50 and 2^-25, rows that
// ask for more are computed again in f32 (value_scale).  A weight held is then at most 2^15, in the sum 2^65, and
// 2^-43 of a row's largest weight is 2^-126 at least, as a weight held and as the factor between two parts of a row.
//
// 32 keys are a tile:  S^T[key, row] = K . Q^T and O^T[d, row] += V^T . P^T on v_mfma_f32_32x32x16_f16, a lane
// with row lane % 32.  The registers of S^T are the operand P^T as they lie: a lane has keys
// 8 j + 4 (lane / 32) + 0..3, and V^T is stored with its keys in that order.
#pragma once

#include "attn_fold.h"
#include "bf16_dev.h"
#include "gemm.h"

namespace bh {

constexpr int kTileKeys = 32;
constexpr int kTermBytes = kTileKeys * kPromptD * 2; // one term of a tile's keys or values
// what a tile's keys are multiplied by at the end, [32] each: of a score; log2 of a value's; its inverse
struct TileScales {
  float key[kTileKeys], value[kTileKeys], undo[kTileKeys];
};
// A tile as launch_attn_terms reads it: keys, values, [term][step][lane][16 bytes] each, then its scales.
constexpr int kTermTile = 4 * kTermBytes + 512; // (PromptTerms has them)
static_assert(sizeof(TileScales) <= 512, "a tile's scales");
inline size_t attn_terms_bytes(int kv_heads, int max_len) {
  return (size_t)kv_heads * ceil_div(max_len, kTileKeys) * kTermTile + 512; // scales are read by whole KiB
}
// Attention of a session's prompt tokens ahead of which there is nothing, on terms that the rotation of its
// q | k | v left (finished rows in a.out); up to kTermsMostKeys tokens.
constexpr int kTermsMostKeys = 8192;
struct AttnPrefillArgs;
int launch_attn_terms(const AttnPrefillArgs &a, const PromptTerms &terms, hipStream_t stream);

#if defined(__HIPCC__)
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
constexpr float kSeedM = -1.0e30f;                   // tosa.py:4383
constexpr float kBelow = 8.0f, kMost = 15.0f;        // log2 of a row's largest weight as it is set, and at most

__device__ __forceinline__ f32x16 mma_f16(uint4 a, uint4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
// two values as two words of two float16 terms; what is not finite has a NaN among its terms
__device__ __forceinline__ void split2(float x, float y, unsigned &t0, unsigned &t1) {
  const f16x2 h = __builtin_convertvector((f32x2{x, y}), f16x2);
  t0 = __builtin_bit_cast(unsigned, h);
  t1 = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{x - (float)h[0], y - (float)h[1]}), f16x2));
}
__device__ __forceinline__ void split8(const float (&x)[8], uint4 (&t)[2]) {
  unsigned w[2][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    split2(x[2 * i], x[2 * i + 1], w[0][i], w[1][i]);
#pragma unroll
  for (int p = 0; p < 2; ++p)
    t[p] = uint4{w[p][0], w[p][1], w[p][2], w[p][3]};
}
// The power of two that brings a magnitude (as bits) to 2^14 .. 2^15, between 2^-114 and 2^126, as the
// exponent that a float has it with.  (An infinity stays one.)
__device__ __forceinline__ unsigned scale_exponent(unsigned magnitude) { return min(268u - (magnitude >> 23), 253u); }
__device__ __forceinline__ float pow2(unsigned exponent) { return __uint_as_float(exponent << 23); }
// maxima and sums over rows of 8 and 16 lanes
__device__ __forceinline__ unsigned row8_max_u32(unsigned v) {
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true));
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true));
  return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true));
}
__device__ __forceinline__ unsigned row16_max_u32(unsigned v) {
  v = row8_max_u32(v);
  return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, true));
}
__device__ __forceinline__ int row8_sum_i32(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, true);
  return v + __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);
}
__device__ __forceinline__ int row16_sum_i32(int v) {
  v = row8_sum_i32(v);
  return v + __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true);
}
__device__ __forceinline__ unsigned magnitude8(const float (&x)[8]) {
  unsigned m = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    m = max(m, __float_as_uint(x[e]) & 0x7fffffffu);
  return m;
}
// A row of 128 values in sixteen groups of eight keeps its accuracy, that of every group, while its largest
// group is not far above the others.  How far a group's magnitude is below the row's in powers of two, 24 at
// most and none for a group of zeros, comes to more than kStray for all sixteen where one group is 2^12 above
// the other fifteen, or eight are 2^22 above the other eight.
constexpr int kStray = 180;
__device__ __forceinline__ int below(unsigned group, unsigned row) {
  const int e = (int)(group >> 23);
  return e ? min((int)(row >> 23) - e, 24) : 0;
}

// The scale of a key's row, sixteen lanes with eight values each: its exponent, and what goes into
// TileScales::key.  Of a stray row that is NaN: the rows that see the key are computed again.
__device__ __forceinline__ unsigned key_scale(const float (&x)[8], float &undo) {
  const unsigned group = magnitude8(x), most = row16_max_u32(group), e = scale_exponent(most);
  undo = row16_sum_i32(below(group, most)) > kStray ? __uint_as_float(0x7fc00000u) : pow2(254 - e);
  return e;
}
// The same of a value's row.  A value that has no terms, or leaves none to the others, must not reach rows that
// do not see its key, whose weight there is zero, nor other channels: it becomes zero, and the
// row's log2, NaN, makes NaN of the rows that do see the key, which are computed again.  cleared(i): value i of this
// lane became zero.  So are rows that see one all below 2^-36 and not zero, or of 2^40 and more; a row of zeros, for
// whose key there is a weight like any other's, has the scale of one of 2^-36.
constexpr unsigned kLeastValue = 127 - 36, kMostValue = 127 + 39; // exponents of a row's largest magnitude
template <class F>
__device__ __forceinline__ unsigned value_scale(float (&x)[8], float &log2_of, F &&cleared) {
  bool bad = false;
  unsigned most;
  for (;;) {
    const unsigned group = magnitude8(x);
    most = row16_max_u32(group);
    const bool stray = most >= 0x7f800000u || row16_sum_i32(below(group, most)) > kStray;
    if (__builtin_expect(!__any(stray), 1))
      break;
    bad |= stray;
    const unsigned from = most >= 0x7f800000u ? 0x7f800000u : most - min(most, 11u << 23);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (stray && (__float_as_uint(x[i]) & 0x7fffffffu) >= from) {
        x[i] = 0.f;
        cleared(i);
      }
  }
  const unsigned of = most >> 23, e = scale_exponent(max(of, kLeastValue) << 23);
  bad |= (most != 0 && of < kLeastValue) || of > kMostValue;
  log2_of = bad ? __uint_as_float(0x7fc00000u) : 127.0f - (float)e;
  return e;
}

// Row `pos` of a KV head's keys and values, sixteen lanes with values 4 i + 0..3 and 64 + 4 i + 0..3 each, into
// the tile it belongs to.
__device__ __forceinline__ unsigned char *terms_tile(const PromptTerms &t, int kvh, int pos) {
  return t.tiles + ((size_t)kvh * t.per_head + pos / kTileKeys) * kTermTile;
}
__device__ __forceinline__ void put_key_terms(const PromptTerms &t, int kvh, int pos, int i, const float (&lo)[4],
                                              const float (&hi)[4]) {
  float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, undo;
  const unsigned e = key_scale(x, undo);
  unsigned char *tile = terms_tile(t, kvh, pos);
  const int key = pos % kTileKeys;
  if (i == 0)
    reinterpret_cast<TileScales *>(tile + 4 * kTermBytes)->key[key] = undo;
#pragma unroll
  for (int j = 0; j < 8; ++j)
    x[j] *= pow2(e);
  uint4 term[2];
  split8(x, term);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int d = 64 * h + 4 * i;
    unsigned char *at = tile + d / 16 * 1024 + (d / 8 % 2 * 32 + key) * 16 + d % 8 * 2;
#pragma unroll
    for (int p = 0; p < 2; ++p)
      *reinterpret_cast<uint2 *>(at + p * kTermBytes) = h ? uint2{term[p].z, term[p].w} : uint2{term[p].x, term[p].y};
  }
}
// Where channel c of key `key` is among term p of a tile's values: key 16 s + 8 x + 4 half + r is value r + 4 x of
// the eight that lane 32 half + channel has in step s.
__device__ __forceinline__ unsigned char *value_term_at(unsigned char *tile, int key, int c, int p) {
  return tile + (2 + p) * kTermBytes + (c / 32 * 2 + key / 16) * 1024 + (key / 4 % 2 * 32 + c % 32) * 16 +
         (key / 8 % 2 * 4 + key % 4) * 2;
}
// the scales of a value's row to its tile, its terms to the caller
__device__ __forceinline__ void value_terms(const PromptTerms &t, int kvh, int pos, int i, const float (&lo)[4],
                                            const float (&hi)[4], uint4 (&term)[2]) {
  float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, log2_of;
  const unsigned e = value_scale(x, log2_of, [](int) {});
  if (i == 0) {
    TileScales *sc = reinterpret_cast<TileScales *>(terms_tile(t, kvh, pos) + 4 * kTermBytes);
    sc->value[pos % kTileKeys] = log2_of;
    sc->undo[pos % kTileKeys] = pow2(e);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j)
    x[j] *= pow2(e);
  split8(x, term);
}
__device__ __forceinline__ void put_value_terms(const PromptTerms &t, int kvh, int pos, int i, const float (&lo)[4],
                                                const float (&hi)[4]) {
  uint4 term[2];
  value_terms(t, kvh, pos, i, lo, hi, term);
  unsigned char *tile = terms_tile(t, kvh, pos);
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const unsigned w[4] = {term[p].x, term[p].y, term[p].z, term[p].w};
#pragma unroll
    for (int j = 0; j < 8; ++j)
      *reinterpret_cast<unsigned short *>(value_term_at(tile, pos % kTileKeys, 64 * (j / 4) + 4 * i + j % 4, p)) =
          (unsigned short)(j & 1 ? w[j / 2] >> 16 : w[j / 2]);
  }
}

// A row's weights from its scores, which a lane has of sixteen keys as S^T leaves them.  m: a running
// bound on log2 of the weights times their values' scales, a whole number; l: this lane's share of the sum of the
// weights; o: the sums so far, which move with m.  gap: the row's position minus the tile's first key, looked at
// where `edge`.
struct RowState {
  float m, l, q_scale; // q_scale: of a score
  f32x16 o[4];
};
__device__ __forceinline__ void tile_weights(float (&w)[16], const TileScales &sc, int up, bool edge, int gap,
                                             RowState &r, uint4 (&pf)[2][2]) {
  auto four = [&](const float (&of)[kTileKeys], int j) {
    return *reinterpret_cast<const f32x4 *>(of + 8 * j + 4 * up);
  };
  f32x4 by[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const f32x4 k4 = four(sc.key, j);
    by[j] = four(sc.value, j);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      w[4 * j + e] *= k4[e];
  }
  auto hide = [&](float (&p)[16]) { // keys behind the row
#pragma unroll
    for (int i = 0; i < 16; ++i)
      p[i] = 8 * (i >> 2) + 4 * up + (i & 3) <= gap ? p[i] : -INFINITY;
  };
  // above m, which is whole: one rounding
  float p[16];
  auto above = [&](float m) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      p[i] = fmaf(w[i], r.q_scale, by[i >> 2][i & 3] - m);
    if (edge)
      hide(p);
  };
  auto largest = [&]() {
    float mt = p[0];
#pragma unroll
    for (int i = 1; i < 16; ++i)
      mt = fmaxf(mt, p[i]);
    return mt;
  };
  above(r.m);
  // m moves, and the sums are rescaled, only when a weight exceeds 2^kMost
  if (__any(largest() > kMost)) {
    above(0.f);
    float x, y;
    lane_pair<32>(largest(), x, y);
    const float m = fmaxf(ceilf(fmaxf(x, y)) - kBelow, r.m), alpha = __builtin_amdgcn_exp2f(r.m - m);
    r.m = m;
    r.l *= alpha;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      r.o[i] *= alpha;
    above(m);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    by[j] = four(sc.undo, j);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    p[i] = __builtin_amdgcn_exp2f(p[i]);
    r.l = fmaf(p[i], by[i >> 2][i & 3], r.l);
  }
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const float p8[8] = {p[8 * ks],     p[8 * ks + 1], p[8 * ks + 2], p[8 * ks + 3],
                         p[8 * ks + 4], p[8 * ks + 5], p[8 * ks + 6], p[8 * ks + 7]};
    split8(p8, pf[ks]);
  }
}
#endif

} // namespace bh
