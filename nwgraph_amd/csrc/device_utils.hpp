// device_utils.hpp -- wave64 / workgroup collectives used by the kernels.
// All reductions use a fixed combination tree, so results are run-to-run
// deterministic for a fixed launch shape.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "items.hpp"

namespace nwg {

// Native 4 x 32-bit vector (one 16-byte load or store); the nontemporal builtins take it.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

// Butterfly sum over the low `width` lanes of each width-aligned group (width <= 64).
template <int Width, class T>
__device__ __forceinline__ T group_sum(T v) {
#pragma unroll
  for (int o = Width / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, Width);
  return v;
}

template <class T>
__device__ __forceinline__ T wave_sum(T v) {
  return group_sum<64>(v);
}

// Integer scans and sums over the wave with DPP moves (row shifts, then the last lanes of rows broadcast
// to the rows after them): a VALU operation per step where a shuffle goes through LDS.  The same
// integers, as addition is exact.  Item sweeps on MI355X: RMAT-12 129 to 123 us for 20 sweeps, RMAT-16 199 to 184.
template <int Ctrl, int Rows>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, Ctrl, Rows, 0xf, false);
}
template <int Ctrl, int Rows>
__device__ __forceinline__ unsigned long long dpp_or_zero(unsigned long long v) {
  return ((unsigned long long)dpp_or_zero<Ctrl, Rows>((uint32_t)(v >> 32)) << 32) |
         dpp_or_zero<Ctrl, Rows>((uint32_t)v);
}
template <int Ctrl, int Rows>
__device__ __forceinline__ double dpp_or_zero(double v) {
  return __longlong_as_double((long long)dpp_or_zero<Ctrl, Rows>((unsigned long long)__double_as_longlong(v)));
}
template <class T>
__device__ __forceinline__ T wave_scan_dpp(T v) {
  v += dpp_or_zero<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
  v += dpp_or_zero<0x112, 0xf>(v);
  v += dpp_or_zero<0x114, 0xf>(v);
  v += dpp_or_zero<0x118, 0xf>(v);
  v += dpp_or_zero<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_or_zero<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v) {
  v = wave_scan_dpp(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, 63);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), 63);
  return ((unsigned long long)hi << 32) | lo;
}

// Doubles too, in one fixed order (weighted item sweep of 12,007 rows and 140 K edges: 5.94 to 5.68 us).
__device__ __forceinline__ double wave_sum(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(wave_scan_dpp(v));
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, 63);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), 63);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Sum over a workgroup of NT threads (NT multiple of 64); result valid in thread 0.
template <int NT, class T>
__device__ __forceinline__ T block_sum(T v, T* lds /* NT/64 entries */) {
  v = wave_sum(v);
  const int w = threadIdx.x / 64;
  if (lane_id() == 0) lds[w] = v;
  __syncthreads();
  T r = T(0);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) r += lds[i];
  }
  __syncthreads();
  return r;
}

// Inclusive prefix sum across the wave.
template <class T>
__device__ __forceinline__ T wave_inclusive_scan(T v) {
  const uint32_t l = lane_id();
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    T y = __shfl_up(v, o, 64);
    if (l >= (uint32_t)o) v += y;
  }
  return v;
}

__device__ __forceinline__ unsigned long long wave_inclusive_scan(unsigned long long v) { return wave_scan_dpp(v); }
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) { return wave_scan_dpp(v); }

// Exclusive prefix sum across a workgroup of NT threads; *total gets the block sum.
template <int NT, class T>
__device__ __forceinline__ T block_exclusive_scan(T v, T* lds /* NT/64 + 1 entries */, T* total) {
  constexpr int NW = NT / 64;
  const int w = threadIdx.x / 64;
  T inc = wave_inclusive_scan(v);
  if (lane_id() == 63) lds[w] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    T run = T(0);
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      T t = lds[i];
      lds[i] = run;
      run += t;
    }
    lds[NW] = run;
  }
  __syncthreads();
  T r = inc - v + lds[w];
  *total = lds[NW];
  __syncthreads();
  return r;
}

// One workgroup leaves a segment's L1 changes and the solve's scales for the host (items.hpp, WMail):
// err[first .. k), and last for sweep k, whose own store it may just have made.
__device__ __forceinline__ void wmail_post(const WMail& m, const double* err, uint32_t k, double last) {
  if (!m.words) return;
  if (threadIdx.x < 2) m.words[threadIdx.x] = m.scale[threadIdx.x];
  for (uint32_t q = m.first + threadIdx.x; q < k; q += blockDim.x) m.words[2 + q] = __double_as_longlong(err[q]);
  if (threadIdx.x == 0) m.words[2 + k] = __double_as_longlong(last);
}

// Fixed-point accumulation of the L1 change: integer atomics make the sum
// independent of block completion order (resolution 2^-58, range [0, 32)).
constexpr double kErrScale = 288230376151711744.0;  // 2^58
__device__ __forceinline__ unsigned long long err_to_fixed(double e) {
  if (!(e >= 0.0)) e = 31.0;  // NaN or negative cannot occur; saturate defensively
  if (e > 31.0) e = 31.0;
  return (unsigned long long)__double2ull_rn(e * kErrScale);
}
__host__ __device__ inline double fixed_to_err(unsigned long long q) { return (double)q / kErrScale; }

}  // namespace nwg
