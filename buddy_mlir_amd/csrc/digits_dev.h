// digits_dev.h -- fixed-point digits of f32 values, and loads from memory past the registers into LDS,
// as the kernels on the int8 and bfloat16 matrix cores take them.
#pragma once

#include "common.h"

namespace bh {

// Four values as the words of their balanced digits: word j of four bytes, digit j of each.
// v * inv + 1.5 * 2^23 is rounded to a whole number X, ties to even, in one instruction, and its
// bits are those of the constant plus X (|X| <= 2^22).  X plus 128 in every digit but the last has the
// digits' bytes, each with its top bit turned, in place: no carries to take from digit to digit.
// (Digit by digit with shifts and masks this was 27 instructions a value and is 5.)
// Of values that are not finite anything may come out, for their step is NaN.
__device__ __forceinline__ void digits_of(const float (&v)[4], float inv, int D, unsigned (&word)[3]) {
  const unsigned bias = D == 3 ? 0x8080u : 0x80u;
  unsigned y[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    y[e] = __float_as_uint(fmaf(v[e], inv, 12582912.0f)) + (bias - 0x4B400000u);
  // bytes 0 and 1 of two values each, then of four
  const unsigned a = __builtin_amdgcn_perm(y[1], y[0], 0x05010400u), b = __builtin_amdgcn_perm(y[3], y[2], 0x05010400u);
  word[0] = __builtin_amdgcn_perm(b, a, 0x05040100u) ^ 0x80808080u;
  word[1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
  word[2] = 0;
  if (D == 3) {
    word[1] ^= 0x80808080u;
    const unsigned c = __builtin_amdgcn_perm(y[1], y[0], 0x0c0c0602u), d = __builtin_amdgcn_perm(y[3], y[2], 0x0c0c0602u);
    word[2] = __builtin_amdgcn_perm(d, c, 0x05040100u);
  }
}

// 1 KiB from memory past the registers into LDS: a lane's 16 bytes, at an address of its own or
// `lane_offset` behind a scalar one, to `to` + 16 lane.  Not the compiler's load: landed<N> waits until
// at most N loads are under way that were issued behind the ones asked about.  No load moves across
// one of these statements, which may write any memory as far as the compiler knows.
__device__ __forceinline__ void load_1k_to_lds(const void *from, unsigned to) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(to) : "memory", "m0");
}
__device__ __forceinline__ void load_1k_to_lds(const void *base, unsigned lane_offset, unsigned to) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_offset), "s"(base),
               "s"(to)
               : "memory", "m0");
}
template <int N> __device__ __forceinline__ void landed() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

} // namespace bh
