// attn_prompt.hip -- causal GQA attention of a session's prompt tokens over its KV cache.
//
// The same operation as attn_prefill.hip (flash_attention_for_cpu_prefill_op,
// frontend/Python/ops/tosa.py:4326-4810) with a workspace and on the float16 matrix
// cores, on two float16 terms a value (attn_terms.h): three
// instructions at sixteen times the rate of the f32 matrix instructions (with three bfloat16 terms, which need
// no scales, six: 6 us a tile for 3).  The error against 64 bits of this kernel's results, of the f32 kernel's and of
// three bfloat16 terms', normal values, 12 heads: 1931 tokens 2.5e-7, 2.3e-7 and 2.7e-7, 150 behind 1900 2.9e-7,
// 3.5e-7 and 3.1e-7, with scores twelve times as large 8.5e-7, 8.3e-7 and 1.2e-6; 28-layer prompts of 150 to 1931
// tokens, eleven of them, 5.9e-6 on average with the first two.
//
// What bounds it: per tile of 256 rows x 32 keys a SIMD has 3072 cycles of matrix
// instructions and some 3600 of vector instructions (softmax, conversions), which overlap in part:
// 3 us a tile.  What a launch costs beside its tiles: 6 us until the first one is in terms, as much as two
// tiles to end a block and begin the next (queries and results go through LDS so that a load or store is of whole
// lines: as operands lie, it was 10 us), and the partial results' way out of the L2s behind it, 33 MB.
// 150 tokens behind 1900 of 12 query heads and 2 KV heads 26.6 -> 22 us; 1931 tokens 91 -> 53, and 47 where keys and
// values come as terms (a prompt alone, whose rotation writes them: 6.5 -> 9.8 us).
// us per layer, this kernel and the fold behind it against
// attn_prefill.hip and the conversion behind that (attn_prompt_pays says which is taken):
//   150 behind 1900 30 vs 64
#include "attn.h"
#include "attn_terms.h"
#include "digits_dev.h"

#include <algorithm>
#include <cmath>

namespace bh {
namespace {

constexpr int kThreads = 2 * kPromptRows; // a wavefront has 32 rows
constexpr int kKeys = kTileKeys;
constexpr int kHalf = 2 * kTermBytes;     // keys, then values
constexpr int kBuf = 2 * kHalf;
// two buffers of terms and 4 KiB of each wavefront for what it converts; three that take tiles of terms as they
// come, scales behind them; and 4 KiB of each to turn rows in
constexpr int kTermBuf = kBuf + 1024;
constexpr int lds_bytes(bool terms) {
  return (terms ? 3 * kTermBuf : 2 * kBuf + kThreads / 64 * 4096) + kThreads / 64 * 4096;
}

struct PromptArgs {
  const float *q, *k, *v;
  float *out;
  int64_t q_stride, q_hstride, o_stride, o_hstride, kv_stride;
  int kv_heads, group, q_len, k_len, q_offset, nblk;
  int ahead;        // units ahead of a block's first tile
  int per_head;     // units of a KV head: its tiles and those
  int share, extra; // units of a workgroup, `ahead` + 1 at least; the first `extra` ones take one more
  float scale;      // of the scores, times log2 e
  float *acc, *ml;
  PromptBlock *blocks;
  const unsigned char *terms; // [KV heads][per_head tiles]
  int terms_per_head;
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
// the block that unit t of a KV head belongs to (t becomes the unit within it), or
// nblk with t the number of units beyond the last block
__device__ __forceinline__ int find_block(const PromptArgs &a, int lane, int &t) {
  for (int base = 0; base < a.nblk; base += 64) {
    const int n = base + lane < a.nblk ? tiles_of(a, base + lane) + a.ahead : 0;
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

// Workgroup i takes an equal share of all (KV head, row block, key tile) triples in that
// order, wherever it begins and ends; of a long prompt with two units more ahead of each block's first, for to
// end a block and begin the next takes as long as two tiles (1931 tokens, without them: workgroups end 42 to
// 64 us after the launch began, with them 40 to 52).  Blocks it holds whole leave as finished rows, the
// others as partial results.  Its eight wavefronts have 32 rows each and share the tiles,
// of which each turns an eighth into terms a tile ahead.
// LDS: [buffer][keys | values][term][step][lane][16 bytes], operands as they are
// read; the keys' slots are permuted within a step so that writing them by rows meets
// every bank once.
// TERMS: keys and values lie as terms already, and come tile by tile two ahead.
template <bool TERMS>
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
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  __shared__ __attribute__((aligned(16))) TileScales scales_s[TERMS ? 1 : 2];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, up = lane >> 5;

  // this workgroup's units [t0, t1) of all
  const int self = blockIdx.x;
  auto begins = [&](int i) { return i * a.share + min(i, a.extra); };
  const int t0 = begins(self), t1 = begins(self + 1);

  struct Place {
    int h, b, j, n; // KV head, row block, tile within it, tiles of the block
    int t;          // unit
  };
  Place at;
  {
    at.h = t0 / a.per_head;
    int r = t0 - at.h * a.per_head;
    at.b = find_block(a, lane, r);
    at.j = max(r - a.ahead, 0);
    at.n = tiles_of(a, at.b);
    at.t = t0 + max(a.ahead - r, 0);
  }
  auto next_of = [&](Place p) {
    ++p.t;
    if (++p.j == p.n) {
      p.t += a.ahead;
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
  const int first = at.t; // the workgroup's first tile

  // ---- a tile on its way ------------------------------------------------------------
  // Each wavefront brings what it converts itself into 4 KiB of LDS of its own, a tile
  // ahead and past the registers (there are none left), by the four instructions below:
  // rows 4 wave .. + 3 of the keys and of the values.  The compiler does not see these loads; bring_wait() waits for
  // them, and nothing else reads that memory.
  const int g8 = tid & 15;
  unsigned char *raw = lds + 2 * kBuf + wave * 4096;
  unsigned char *turn = lds + lds_bytes(TERMS) - (kThreads / 64 - wave) * 4096;
  auto buffer = [&](int i) { return lds + i * (TERMS ? kTermBuf : kBuf); };
  auto scales_of = [&](int i) -> TileScales & {
    if constexpr (TERMS)
      return *reinterpret_cast<TileScales *>(buffer(i) + kBuf);
    else
      return scales_s[i];
  };
  // a tile of terms: 4 KiB of it to a wavefront, and its scales to the first
  auto bring_terms = [&](const Place &p, int i) {
    const unsigned char *tile = a.terms + ((size_t)p.h * a.terms_per_head + p.j) * kTermTile;
    const unsigned to = (unsigned)__builtin_amdgcn_readfirstlane(
        (int)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)buffer(i));
#pragma unroll
    for (int n = 0; n < 4; ++n)
      load_1k_to_lds(tile + (wave * 4 + n) * 1024, lane * 16, to + (wave * 4 + n) * 1024);
    if (wave == 0)
      load_1k_to_lds(tile + kBuf, lane * 16, to + kBuf);
  };
  auto bring = [&](const Place &p) {
    const float *k = a.k + (int64_t)p.h * a.kv_stride * kPromptD, *v = a.v + (int64_t)p.h * a.kv_stride * kPromptD;
    const int k0 = p.j * kKeys;
    const unsigned to = (unsigned)__builtin_amdgcn_readfirstlane(
        (int)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)raw);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = min(k0 + 4 * wave + 2 * (i & 1) + up, a.k_len - 1);
      const float *src = (i < 2 ? k : v) + (int64_t)key * kPromptD + col * 4;
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(to + i * 1024)
                   : "memory", "m0");
    }
  };
  auto bring_wait = []() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  // What this wavefront brought as the tile's terms.  Sixteen lanes have a key's row, eight channels each,
  // of keys and of values; a lane turns channels lane and lane + 64 of the four values, which are keys
  // 16 ks + 8 x + 4 half + 0..3.  Everything is read at once.
  auto row_of = [&](const unsigned char *at, float (&x)[8]) {
    const float4 x0 = *reinterpret_cast<const float4 *>(at + (lane >> 4) * 512 + g8 * 32);
    const float4 x1 = *reinterpret_cast<const float4 *>(at + (lane >> 4) * 512 + g8 * 32 + 16);
    x[0] = x0.x; x[1] = x0.y; x[2] = x0.z; x[3] = x0.w;
    x[4] = x1.x; x[5] = x1.y; x[6] = x1.z; x[7] = x1.w;
  };
  auto columns_of = [&](float (&y)[2][4]) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        y[j][r] = *reinterpret_cast<const float *>(raw + 2048 + r * 512 + (lane + 64 * j) * 4);
  };
  auto put_tile = [&](unsigned char *buf, TileScales &sc) {
    float k[8], v[8], y[2][4];
    row_of(raw, k);
    row_of(raw + 2048, v);
    columns_of(y);
    const int key = tid >> 4;
    {
      float undo;
      const unsigned e = key_scale(k, undo);
      if (g8 == 0)
        sc.key[key] = undo;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        k[i] *= pow2(e);
      uint4 term[2];
      split8(k, term);
#pragma unroll
      for (int p = 0; p < 2; ++p)
        *reinterpret_cast<uint4 *>(buf + ((p * 8 + (g8 >> 1)) * 64 + (g8 & 1) * 32 + (key ^ g8)) * 16) = term[p];
    }
    float log2_of;
    bool again = false;
    const unsigned e = value_scale(v, log2_of, [&](int i) {
      *reinterpret_cast<float *>(raw + 2048 + (lane >> 4) * 512 + g8 * 32 + i * 4) = 0.f;
      again = true;
    });
    if (__any(again)) {
      lds_turn();
      columns_of(y);
    }
    if (g8 == 0) {
      sc.value[key] = log2_of;
      sc.undo[key] = pow2(e);
    }
    float by[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      by[r] = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)(e << 23), 16 * r));
    const int ks = wave >> 2, x8 = (wave >> 1) & 1, half = wave & 1;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c = lane + 64 * j;
      unsigned t[2][2];
      split2(y[j][0] * by[0], y[j][1] * by[1], t[0][0], t[1][0]);
      split2(y[j][2] * by[2], y[j][3] * by[3], t[0][1], t[1][1]);
#pragma unroll
      for (int p = 0; p < 2; ++p)
        *reinterpret_cast<uint2 *>(buf + kHalf + (((p * 4 + (c >> 5)) * 2 + ks) * 64 + half * 32 + (c & 31)) * 16 +
                                   x8 * 8) = uint2{t[p][0], t[p][1]};
    }
  };

  uint4 qf[8][2];
  RowState rs;
  int qpos = 0, pos_first = 0, pos_last = 0; // of this lane's row; of the wavefront's rows
  // A block's queries come in as eight lanes to a row, 32 channels at a time (as a lane's own operand they
  // are pieces of 32 rows to a load, and the address unit sets the pace: 4 us), and are turned in
  // another 4 KiB of the wavefront's.
  // this lane, as something to work addresses out from where they are used: kept from block to block they
  // would take registers there are not
  auto unkept = [&]() {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  const float per_group = 1.0f / (float)a.group;
  struct Base {
    int tok, rem, last; // of a block's first row: token, row within it; the last row from that token on
  };
  auto base_of = [&](int b) {
    const int tok = b * kPromptRows / a.group;
    return Base{tok, b * kPromptRows - tok * a.group, (a.q_len - tok) * a.group - 1};
  };
  auto place_of = [&](const Base &base, int r, int &tok) { // row r of the wavefront: its token, and head of the group
    const int rem = min(base.rem + wave * 32 + r, base.last);
    const int t = (int)(((float)rem + 0.5f) * per_group);
    tok = base.tok + t;
    return rem - t * a.group;
  };
  auto ask_queries = [&](const Place &p, float4 (&asked)[16]) {
    const int lane = unkept();
    const Base base = base_of(p.b);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      int tok;
      const int hh = place_of(base, 8 * j + (lane >> 3), tok);
      const float *src = a.q + (int64_t)tok * a.q_stride + (int64_t)(p.h * a.group + hh) * a.q_hstride + (lane & 7) * 4;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        asked[4 * c + j] = *reinterpret_cast<const float4 *>(src + c * 32);
    }
  };
  auto begin_block = [&](int b, float4 (&asked)[16]) {
    const int lane = unkept(), col = lane & 31, up = lane >> 5;
    int tok;
    place_of(base_of(b), col, tok);
    qpos = a.q_offset + tok;
    pos_first = __builtin_amdgcn_readfirstlane(qpos);
    pos_last = __builtin_amdgcn_readlane(qpos, 31);
    float of_row[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) { // row 8 j + lane / 8: eight lanes with two groups of eight values each
      unsigned group[2], most;
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const float4 u = asked[8 * g + j], v = asked[8 * g + 4 + j];
        const float y[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
        group[g] = magnitude8(y);
      }
      most = row8_max_u32(max(group[0], group[1]));
      const int sum = row8_sum_i32(below(group[0], most) + below(group[1], most));
      const unsigned e = scale_exponent(most);
      of_row[j] = sum > kStray ? __uint_as_float(0x7fc00000u) : pow2(254 - e) * a.scale;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float4 &u = asked[4 * c + j];
        u = make_float4(u.x * pow2(e), u.y * pow2(e), u.z * pow2(e), u.w * pow2(e));
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      // 32 channels of all rows as terms, [term][row][64 bytes]; pieces of 16 bytes permuted by the row's number
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4 u = asked[4 * c + j];
        const int r = 8 * j + (lane >> 3);
        uint2 t[2];
        split2(u.x, u.y, t[0].x, t[1].x);
        split2(u.z, u.w, t[0].y, t[1].y);
#pragma unroll
        for (int p = 0; p < 2; ++p)
          *reinterpret_cast<uint2 *>(turn + p * 2048 + r * 64 + (((lane & 7) >> 1) ^ (r >> 1 & 3)) * 16 +
                                     (lane & 1) * 8) = t[p];
      }
      lds_turn();
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          qf[2 * c + i][p] = *reinterpret_cast<const uint4 *>(turn + p * 2048 + col * 64 +
                                                              ((2 * i + up) ^ (col >> 1 & 3)) * 16);
      lds_turn();
      __builtin_amdgcn_sched_barrier(0);
    }
    if ((lane & 7) == 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<float *>(turn + (8 * j + (lane >> 3)) * 4) = of_row[j];
    }
    lds_turn();
    rs.q_scale = *reinterpret_cast<const float *>(turn + col * 4);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      rs.o[i] = f32x16{};
    rs.m = kSeedM;
    rs.l = 0.f;
  };

  float w[16];    // scores of this lane's row, then their weights
  uint4 pf[2][2]; // the weights as terms
  auto scores = [&](const unsigned char *buf) {
    f32x16 s0{}, s1{}; // the small products by themselves
    // the slot of this lane's key in step s is (col ^ up) ^ 2 s: worked out at each tile,
    // not kept in registers that there are not
    int at_key = TERMS ? lane * 16 : up * 512 + (col ^ up) * 16;
    asm volatile("" : "+v"(at_key));
    // fragments are asked for two steps ahead of their products, and stay there: left to itself the
    // scheduler moves them to their use, and every one is waited out
    uint4 kf[3][2];
    auto ask = [&](int s) {
#pragma unroll
      for (int p = 0; p < 2; ++p)
        kf[s % 3][p] =
            *reinterpret_cast<const uint4 *>(buf + (TERMS ? at_key : at_key ^ (32 * s)) + (p * 8 + s) * 1024);
    };
    ask(0);
    ask(1);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      if (s + 2 < 8)
        ask(s + 2);
      __builtin_amdgcn_sched_barrier(0);
      s1 = mma_f16(kf[s % 3][0], qf[s][1], s1);
      s0 = mma_f16(kf[s % 3][0], qf[s][0], s0);
      s1 = mma_f16(kf[s % 3][1], qf[s][0], s1);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
      w[i] = s0[i] + s1[i];
  };
  auto add_values = [&](const unsigned char *buf) {
    uint4 vf[2][2][2];
    auto ask = [&](int i) { // 16 keys, two of the four blocks of 32 channels
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          vf[i & 1][p][e] = *reinterpret_cast<const uint4 *>(
              buf + (((p * 4 + 2 * (i & 1) + e) * 2 + (i >> 1)) * 64 + lane) * 16);
    };
    ask(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i < 3)
        ask(i + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 3; ++c) // small ones first
#pragma unroll
        for (int e = 0; e < 2; ++e)
          rs.o[2 * (i & 1) + e] = mma_f16(vf[i & 1][c == 0][e], pf[i >> 1][c == 1], rs.o[2 * (i & 1) + e]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  auto end_block = [&](const Place &p, int first_tile, bool from_start, bool whole) {
    float x, y;
    lane_pair<32>(rs.l, x, y);
    const float sum = x + y;
    const int lane = unkept(), col = lane & 31, up = lane >> 5;
    const int r0 = wave * 32, left = a.q_len * a.group - p.b * kPromptRows - r0; // rows of the wavefront that there are
    // the first part of this workgroup's share in slot 2 i, one behind it in 2 i + 1
    const size_t slot = (2 * (size_t)self + (first_tile > first ? 1 : 0)) * kPromptRows + r0;
    if (!whole && up == 0 && col < left)
      *reinterpret_cast<float2 *>(a.ml + (slot + col) * 2) = make_float2(rs.m, sum);
    // turned so that a store writes 128 bytes of each of eight rows (as they lie, 32 of each of 32: twice
    // as long)
    const float f = whole ? inverse_of(sum) : 1.0f;
    const Base base = base_of(p.b);
    float *dst[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 8 * i + (lane >> 3);
      int tok;
      const int hh = place_of(base, r, tok);
      dst[i] = (whole ? a.out + (int64_t)tok * a.o_stride + (int64_t)(p.h * a.group + hh) * a.o_hstride
                      : a.acc + (slot + r) * kPromptD) +
               (lane & 7) * 4;
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) { // pieces of 16 bytes permuted by the row's number
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<float4 *>(turn + col * 128 + ((2 * j + up) ^ (col & 7)) * 16) =
            float4{rs.o[dt][4 * j] * f, rs.o[dt][4 * j + 1] * f, rs.o[dt][4 * j + 2] * f, rs.o[dt][4 * j + 3] * f};
      lds_turn();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4 x = *reinterpret_cast<const float4 *>(turn + (8 * i + (lane >> 3)) * 128 +
                                                           ((lane & 7) ^ (lane >> 3)) * 16);
        if (8 * i + (lane >> 3) < left)
          *reinterpret_cast<float4 *>(dst[i] + dt * 32) = x;
      }
      lds_turn();
    }
    if (tid == 0 && from_start) {
      // whoever has the block's first tile says where its parts are
      PromptBlock d{0, 0, 0, 0};
      if (!whole) {
        const int last = first_tile + p.n - 1, longer = a.extra * (a.share + 1);
        const int i = last < longer ? last / (a.share + 1) : a.extra + (last - longer) / a.share;
        d.first = 2 * self + (first_tile > first ? 1 : 0);
        d.owner = self;
        d.parts = i - self + 1;
      }
      a.blocks[p.h * a.nblk + p.b] = d;
    }
  };

  Place nx = next_of(at);
  float4 asked[16];
  if constexpr (TERMS) {
    bring_terms(at, 0);
    if (nx.t < t1)
      bring_terms(nx, 1);
    ask_queries(at, asked); // which begin_block waits for, and with them for those
  } else {
    bring(at);
    ask_queries(at, asked);
    __syncthreads();
    bring_wait();
    put_tile(buffer(0), scales_of(0));
    if (nx.t < t1)
      bring(nx);
  }
  int cur = 0;
  bool arrived = false; // the tile on its way
  for (;;) { // a block, or the part of it held here, at a time
    begin_block(at.b, asked);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      asked[i] = float4{}; // what was in them need not be kept
    const int seg0 = at.t; // its first tile
    const bool from_start = at.j == 0;
    bool more, ends;
    for (;;) {
      __syncthreads();
      more = nx.t < t1;
      const Place nn = next_of(nx);
      const int next = TERMS ? (cur == 2 ? 0 : cur + 1) : cur ^ 1;
      unsigned char *buf = buffer(cur);
      if constexpr (TERMS) {
        if (nn.t < t1) // into the buffer read in the step before
          bring_terms(nn, next == 2 ? 0 : next + 1);
      }
      auto stage = [&]() {
        if (!more)
          return;
        if (!arrived)
          bring_wait();
        put_tile(buffer(next), scales_of(next));
        if (nn.t < t1)
          bring(nn);
      };
      // the two wavefronts of a SIMD in opposite order: one's conversion beside the other's
      // products
      if (!TERMS && wave < 4)
        stage();
      if (at.j * kKeys <= pos_last) {
        scores(buf);
        const int k0 = at.j * kKeys;
        tile_weights(w, scales_of(cur), up, k0 + kKeys - 1 > pos_first, qpos - k0, rs, pf);
        add_values(buf + kHalf);
      }
      if constexpr (TERMS) { // the next tile, behind which this step has asked for one more at most
        if (nn.t >= t1)
          landed<0>();
        else if (wave == 0)
          landed<5>();
        else
          landed<4>();
      } else if (wave >= 4) {
        stage();
      }
      arrived = false;
      ends = at.j + 1 == at.n;
      if (ends || !more)
        break;
      at = nx;
      nx = nn;
      cur = next;
    }
    if (more)
      ask_queries(nx, asked); // ahead of the stores, which a load behind them would wait for
    end_block(at, seg0, from_start, ends && from_start);
    if (!more)
      break;
    at = nx;
    nx = next_of(nx);
    cur = TERMS ? (cur == 2 ? 0 : cur + 1) : cur ^ 1;
    // begin_block waits for the queries, which were asked for behind that tile, and not for the stores
    arrived = true;
  }
}

} // namespace

// The (KV head, row block, key tile) triples of a launch and who takes them.
namespace {
BH_TILE_FAMILY(PromptFamily, "attn_prompt_kernel");
struct PromptShare {
  int64_t rows, tiles; // rows of a KV head; tiles of all
  int64_t units;       // what is shared out
  int nblk, workgroups, ahead;
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
  // each at least a tile, and of few no more than the longest share asks for: partial results go with them
  s.ahead = s.tiles >= 4 * kPromptWorkgroups ? 2 : 0;
  s.workgroups = s.ahead ? kPromptWorkgroups : (int)ceil_div(s.tiles, ceil_div(s.tiles, kPromptWorkgroups));
  s.units = s.tiles + s.ahead * (int64_t)s.nblk * kv_heads;
  return s;
}
} // namespace

// An estimate of both ways in microseconds, fitted to 1748 prompts of 12 layers (eight shapes of 1
// to 64 heads, 4 to 1000 tokens behind 0 to 1200, in three modes) when this kernel took 5.1 us a tile, for 3 now, and
// the fold one workgroup a token.  The line still lies where the two were equal then: prompts a little on the
// other way's side of it may be faster this way by now.  `converts`: behind the other way the
// rows take a launch of their own to become the output product's input, which the fold is here
// (not up to 16 tokens as f32, nor up to 128 as digits, which that product makes itself).  us a
// layer with its products, the other way and this one as it was, where the line lies:
//   12 heads, 2 KV heads, digits: 4 behind 400 40.9, 42.3, behind 700 47.0, 43.9, 32 behind 256
//     53.3, 54.9, behind 700 60.7, 58.0, 256 behind 400 70.1, 70.1, 500 alone 74.9, 75.6, behind
//     128 79.5, 86.7, behind 400 93.0, 90.3, 730 alone 99.8, 102.0, 920 115.9, 113.7
//   64 and 8, digits: 32 behind 256 63.6, 77.2, 128 behind 700 107.7, 107.0, 256 behind 128 111,
//     115, behind 256 123, 118, 500 alone 165, 160
//   one head, every bit: 64 behind 64 54.7, 56.5, behind 128 57.4, 56.8, 256 behind 64 65.6, 64.6
// More than 32 tokens behind 400 and more go this way in doubt, up to 6 us, and more than 640 up to
// 2.5: it asks for each key once for all heads of a KV head, and what is not finite stays with the
// rows that see it.
// `on_terms`: a prompt alone that has attn_terms.hip as the other way, whose workgroups read every key of their 32 rows for
// themselves: us a layer, that way and this one, 12 heads, 2 KV heads, 400 tokens 126 and 133, 800 195 and 206, 1000
// 226 and 235, 1500 320 and 323, 1931 405 and 401; 32 and 8, 400 tokens 156 and 165, 600 202 and 210, 800 256 and
// 252, 1000 301 and 291, 1931 570 and 532.  One line for both: 890 tokens, of more than 22 heads fewer.
bool attn_prompt_pays(int q_len, int q_offset, int heads, int kv_heads, bool converts, bool on_terms) {
  if (on_terms)
    return q_len > 890 || (int64_t)q_len * heads > 20000;
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

int launch_attn_prompt(const AttnPrefillArgs &in, const PromptTerms &terms, void *workspace, PromptFold &fold,
                       hipStream_t stream) {
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
  BH_REQUIRE(share.units < (1u << 30), "attn_prompt: %lld tiles of keys", (long long)share.units);
  a.nblk = share.nblk;
  a.acc = static_cast<float *>(workspace);
  const size_t slots = 2 * (size_t)share.workgroups;
  a.ml = a.acc + slots * kPromptRows * kPromptD;
  a.blocks = reinterpret_cast<PromptBlock *>(a.ml + slots * kPromptRows * 2);
  a.ahead = share.ahead;
  a.per_head = (int)(share.units / in.kv_heads);
  a.share = (int)(share.units / share.workgroups);
  a.extra = (int)(share.units % share.workgroups);
  BH_NOTE_VARIANT(PromptFamily, kPromptRows);
  a.terms = terms.tiles;
  a.terms_per_head = terms.per_head;
  BH_REQUIRE(!terms.tiles || (a.q_offset == 0 && ceil_div(in.k_len, kKeys) <= terms.per_head),
             "attn_prompt: %d tiles of terms for %d keys", terms.per_head, in.k_len);
  static DynLdsOnce dyn_lds[2];
  auto launch = [&](auto kernel, bool on_terms) -> int {
    BH_CHECK_HIP(ensure_dyn_lds(dyn_lds[on_terms], reinterpret_cast<const void *>(kernel), lds_bytes(on_terms)));
    hipLaunchKernelGGL(kernel, dim3((unsigned)share.workgroups), dim3(kThreads), lds_bytes(on_terms), stream, a.k, a.v,
                       a.kv_stride, a.share, a.extra, a.per_head, a.nblk, a.group, a.q_len, a.k_len, a.q_offset, a);
    return BUDDY_HIP_OK;
  };
  if (int rc = terms.tiles ? launch(attn_prompt_kernel<true>, true) : launch(attn_prompt_kernel<false>, false))
    return rc;
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
