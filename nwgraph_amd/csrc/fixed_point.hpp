// fixed_point.hpp -- exact row sums: float <-> 64-bit fixed point in units of 2^-60, used by the
// binned sweep (binned.hip) and the item sweep (items.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nwg {

// Row sums are exact 64-bit fixed-point sums in units of 2^-60.  A float contribution
// c in [0, 1] is converted with float operations that are all exact: s = c * 2^28,
// h = floor(s) (h <= 2^28; (float)h is exact), r = s - h (the fraction bits of s), and
// l = floor(r * 2^32); the fixed-point value h * 2^32 + l is c * 2^60 truncated to an
// integer, which is exact for c >= 2^-37 (every significand bit at or above 2^-60).  As a
// row sum z <= 1 stays below 2^60 units, integer adds never overflow and the sum does not
// depend on the order or the split of the entries.  (z <= sum of all x <= 1: x starts
// summing to 1 and a sweep maps a vector of sum <= 1 to one of sum <= 1.)  No FP64
// arithmetic is used.
__device__ __forceinline__ unsigned long long quantize(float c) {
  const float sc = c * 268435456.f;  // c * 2^28
  const uint32_t h = (uint32_t)sc;
  const float r = __builtin_amdgcn_fractf(sc);  // sc - floor(sc) = sc - h, exact
  const uint32_t l = (uint32_t)(r * 4294967296.f);  // floor(r * 2^32) < 2^32
  return ((unsigned long long)h << 32) | l;
}
// Whether quantize cuts bits of some value off: the smallest magnitude but 0 among the values noted is
// below 2^-37 (signed: 2^-37 / 2^t).  Kept as twice the bits less 2, of which 0 gives the largest
// number: one or two integer operations a value.
struct CutNote {
  uint32_t least = ~0u;
  __device__ __forceinline__ void note(float v) { least = min(least, (__float_as_uint(v) << 1) - 2u); }
  __device__ __forceinline__ bool cuts(int t = 0) const {
    return least < (__float_as_uint(__builtin_ldexpf(1.f, -37 - t)) << 1) - 2u;
  }
};
// A sum of m such values is short by less than m units of 2^-60 (of 2^(-60 - t) when scaled by 2^t),
// which is above 2^-26 of a result x only below m * 2^-34: there a float sum would be the more precise,
// and the sweeps add the row up once more in double.
__device__ __forceinline__ bool sum_is_coarse(float x, uint32_t m, int t = 0) {
  return fabsf(x) < __builtin_ldexpf((float)m, -34 - t);
}
// v * 2^-60 rounded to the nearest float (ties to even).  Below 2^53 (sums under 2^-7, nearly
// every row) v is exact as a double, so one rounding to float and an exact scale by 2^-60 give
// it; above, integer operations do.
__device__ __forceinline__ float dequantize(unsigned long long v) {
  const uint32_t hi = (uint32_t)(v >> 32);
  if (hi < (1u << 21)) return (float)__builtin_fma((double)hi, 4294967296.0, (double)(uint32_t)v) * 0x1p-60f;
  const int lz = __clzll((long long)v);
  const unsigned long long nv = v << lz;  // bit 63 set
  uint32_t mant = (uint32_t)(nv >> 40);   // 24 significant bits
  const unsigned long long rest = nv & ((1ull << 40) - 1), half = 1ull << 39;
  if (rest > half || (rest == half && (mant & 1u))) ++mant;
  int ex = 63 - lz - 60 - 23;  // value = mant * 2^ex
  if (mant == (1u << 24)) {
    mant >>= 1;
    ++ex;
  }
  return __builtin_ldexpf((float)mant, ex);  // exact: mant < 2^24, result a normal float
}

// Weighted sweep: an entry's value w * v may be negative (the adjoint) and of any magnitude.
// The solve picks a power of two 2^t that maps every product and every partial row sum into
// [-1/2, 1/2] (a bound it proves from the weights and its right-hand side), and the scaled
// value is summed in two's complement fixed point in units of 2^-60: exact integer adds,
// independent of order and split, no overflow (|sum| < 2^59 units).
__device__ __forceinline__ unsigned long long quantize_signed(float v, int t) {
  const float sc = __builtin_ldexpf(v, t);  // a power-of-two scale: exact (tiny values may flush)
  const unsigned long long q = quantize(fabsf(sc));
  return sc < 0.f ? 0ull - q : q;
}
__device__ __forceinline__ float dequantize_signed(unsigned long long v, int t) {
  const bool neg = (long long)v < 0;
  const float f = __builtin_ldexpf(dequantize(neg ? 0ull - v : v), -t);
  return neg ? -f : f;
}

}  // namespace nwg
