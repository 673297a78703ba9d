// Requantisation to int8 behind a product, for kernels that know a chain of one clamp and one shift (what the planner leaves of a
// cvm_right_shift once its rounding term is in the bias): which chains those are, for the host, and the instructions, for the device.
#ifndef CVM_REQUANT_H_
#define CVM_REQUANT_H_

#include "hip_common.h"

namespace cvmhip {

// One clamp and one shift?  (lo <= hi; an empty chain is a clamp to all values and no shift)
inline bool clamp_shift_of(const DevChain& c, int* lo, int* hi, int* shift) {
  *lo = INT32_MIN;
  *hi = INT32_MAX;
  *shift = 0;
  if (c.count == 0) return true;
  const DevStage& q = c.st[0];
  if (c.count > 1 || q.mul != 1 || q.add != 0 || (q.s1 != 0 && q.s2 != 0) || q.lo > q.hi) return false;
  *lo = q.lo;
  *hi = q.hi;
  *shift = q.s1 + q.s2;
  return true;
}
// Are its results int8 whatever it is given?  (shift_to_bytes saturates where other forms of a layer take the low byte.)
inline bool clamp_shift_narrow(int lo, int hi, int shift) { return lo >> shift >= -128 && hi >> shift <= 127; }

#if defined(__HIPCC__)
typedef int requant_v4i __attribute__((ext_vector_type(4)));

// A vector instruction may read a product's registers 19 wait states behind one of sixteen passes (32 x 32 x 32) and 11 behind one of eight
// (16 x 16 x 64).  The compiler sees to that for instructions it knows; the clamp below is inline assembly to it, and so the wait is part of the
// values' way there: asm volatile(WAIT_16_PASSES : "+v"(acc) ...), all of them in one statement.
#define WAIT_16_PASSES "s_nop 15\n\ts_nop 3"
#define WAIT_8_PASSES "s_nop 15"

// lo <= hi, uniform
__device__ __forceinline__ int clamp_uniform(int v, int lo, int hi) {
  int r;
  asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(lo), "v"(hi));
  return r;
}

// low bytes of four values -> one dword
__device__ __forceinline__ uint32_t low_bytes(int32_t a, int32_t b, int32_t c, int32_t d) {
  const uint32_t lo2 = __builtin_amdgcn_perm((uint32_t)b, (uint32_t)a, 0x0c0c0400u);
  const uint32_t hi2 = __builtin_amdgcn_perm((uint32_t)d, (uint32_t)c, 0x0c0c0400u);
  return __builtin_amdgcn_perm(hi2, lo2, 0x05040100u);
}
// four values that are int8 once shifted -> one dword: three instructions where a shift each and low_bytes are seven
__device__ __forceinline__ uint32_t shift_to_bytes(int32_t a, int32_t b, int32_t c, int32_t d, int shift) {
  uint32_t lo2, hi2;   // (the builtin's 16 bits would be masked once more)
  asm("v_ashr_pk_i8_i32 %0, %1, %2, %3" : "=v"(lo2) : "v"(a), "v"(b), "s"(shift));
  asm("v_ashr_pk_i8_i32 %0, %1, %2, %3" : "=v"(hi2) : "v"(c), "v"(d), "s"(shift));
  return __builtin_amdgcn_perm(hi2, lo2, 0x05040100u);
}

// The sixteen results of a lane of a 32 x 32 product, four channels to a dword -> 16 consecutive channels of its pixel: in the lower half of
// the wavefront channels 0 .. 15 of the 32, in the upper 16 .. 31.  (The halves trade registers: all lanes take part, also those that store nothing.)
__device__ __forceinline__ requant_v4i sixteen_channels(const uint32_t (&d)[4]) {
  typedef unsigned v2u __attribute__((ext_vector_type(2)));
  const v2u s0 = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false), s1 = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
  return requant_v4i{(int)s0.x, (int)s0.y, (int)s1.x, (int)s1.y};
}
#endif

}  // namespace cvmhip
#endif
