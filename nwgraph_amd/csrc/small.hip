// small.hip -- whole PageRank solves of small graphs: one workgroup, one launch, every sweep in LDS.
//
// The sweep is the item sweep's (items.hip): exact 64-bit fixed-point row sums as differences of a
// running prefix over the edges, Jacobi order (include/nwgraph/algorithms/page_rank.hpp:121-147).  A
// launch per sweep costs 5.4 us however little it does; two barriers of one workgroup cost a
// fraction of one.  What is left is LDS work, E gathers of 8 bytes per lane, and the chain of scan, update
// and change.
//
// Lane t keeps its E consecutive edges for the whole solve: their sources (two to a register) and one
// bit each that says whether the edge is its row's last.  Rows are spread over the lanes, R each, with
// score, degree and base in registers.  A sweep:
//   1  E gathers of the sources' quantized contributions, added up as they come; the lane's running sum
//      at every row's last edge goes to LDS, and the scan of the lanes' sums over the wave
//   2  (barrier) row sums as differences of two prefixes (the lane's, the lanes' before it, the waves'
//      before it), the update, the new quantized contributions, the L1 change
//   3  (barrier) stop or go on
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_utils.hpp"
#include "fixed_point.hpp"
#include "nwg_internal.hpp"
#include "small.hpp"

namespace nwg {

namespace {

constexpr uint32_t kR = 4;      // rows per lane
constexpr uint32_t kNone = 0xFFFFFFFFu;

template <uint32_t NT, uint32_t E>
__global__ __launch_bounds__(NT) void small_solve_kernel(SmallParams P, uint64_t k0, uint64_t k1) {
  static_assert(E % 8 == 0 && E <= 24, "an edge window spans at most two words of row ends");
  constexpr uint32_t kWaves = NT / 64, kRows = kR * NT, kWords = NT * E / 32;
  __shared__ unsigned long long q[kRows + 1];  // contributions; the last one is 0, for lanes past the edges
  __shared__ unsigned long long pre[kRows];    // by rank of the non-empty rows: the lane's running sum at the row's last edge
  __shared__ unsigned long long lpre[NT];      // the lanes' sums before a lane in its wave
  __shared__ unsigned long long wtot[kWaves], werr[kWaves];
  __shared__ uint32_t bits[kWords + 1], word_pre[kWords + 1], wcnt[kWaves];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t g = blockIdx.x;
  const uint32_t r0 = P.voff ? P.voff[g] : 0u;
  const uint32_t n = P.voff ? P.voff[g + 1] - r0 : P.n;
  if (!n) {
    for (uint64_t k = k0 + tid; k < k1; k += NT) P.acc[k * P.ngraphs + g] = 0ull;
    return;
  }
  const bool done = k0 > 0 && fixed_to_err(P.acc[(k0 - 1) * P.ngraphs + g]) < P.threshold;
  const uint32_t eb = P.rp[r0], nnz = P.rp[r0 + n] - eb;
  // the rows, and where they end
  const float init = (float)(1.0 / n);  // page_rank.hpp:93
  float x[kR], b[kR];
  uint32_t lanes[kR];  // of the row's last edge, and of the edge before its first one
  uint32_t dg[kR], end[kR], rk[kR];  // end: the row's last edge
  for (uint32_t w = tid; w <= kWords; w += NT) bits[w] = 0u;
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < kR; ++r) {
    const uint32_t i = tid + r * NT;
    x[r] = 0.f;
    b[r] = 0.f;
    dg[r] = 0u;
    end[r] = kNone;
    lanes[r] = 0u;
    if (i < n) {
      const uint32_t a = P.rp[r0 + i] - eb, e = P.rp[r0 + i + 1] - eb;
      dg[r] = P.deg[r0 + i];
      b[r] = P.basev ? P.basev[r0 + i] : P.base;
      x[r] = k0 ? P.x[r0 + i] : init;
      q[i] = quantize(x[r] / (float)dg[r]);
      if (e > a) {
        end[r] = e - 1;
        lanes[r] = (e - 1) / E | (a ? (a - 1) / E : 0u) << 16;
        atomicOr(&bits[(e - 1) >> 5], 1u << ((e - 1) & 31u));
      }
    }
  }
  if (tid == 0) q[kRows] = 0ull;
  // the lane's edges
  const uint32_t p0 = tid * E;
  uint32_t ids[E / 2];
#pragma unroll
  for (uint32_t t = 0; t < E; t += 2) {
    const uint32_t u = p0 + t < nnz ? P.col[eb + p0 + t] - r0 : kRows;
    const uint32_t v = p0 + t + 1 < nnz ? P.col[eb + p0 + t + 1] - r0 : kRows;
    ids[t / 2] = u * 8 | (v * 8 << 16);  // byte offsets in q
  }
  __syncthreads();
  // row ends before each word
  uint32_t run = 0;
  for (uint32_t w0 = 0; w0 <= kWords; w0 += NT) {
    const uint32_t w = w0 + tid;
    const uint32_t c = w <= kWords ? (uint32_t)__popc(bits[w]) : 0u;
    const uint32_t inc = wave_inclusive_scan(c);
    if (lane == 63) wcnt[wave] = inc;
    __syncthreads();
    uint32_t before = run;
    for (uint32_t v = 0; v < kWaves; ++v) {
      before += v < wave ? wcnt[v] : 0u;
      run += wcnt[v];
    }
    if (w <= kWords) word_pre[w] = before + inc - c;
    __syncthreads();
  }
  auto rank_of = [&](uint32_t p) {  // row ends before edge p
    return word_pre[p >> 5] + (uint32_t)__popc(bits[p >> 5] & ((1u << (p & 31u)) - 1u));
  };
#pragma unroll
  for (uint32_t r = 0; r < kR; ++r) rk[r] = end[r] == kNone ? kNone : rank_of(end[r]);
  const uint32_t first = rank_of(p0);  // p0 <= 32 kWords - E
  const uint64_t window = ((uint64_t)bits[(p0 >> 5) + 1] << 32) | bits[p0 >> 5];
  const uint32_t ends = (uint32_t)(window >> (p0 & 31u)) & ((1u << E) - 1u);

  uint64_t k = k0;
  if (!done) {
    while (k < k1) {
      unsigned long long s = 0ull;
      uint32_t at = first;
#pragma unroll
      for (uint32_t t = 0; t < E; ++t) {
        const uint32_t o = t % 2 ? ids[t / 2] >> 16 : ids[t / 2] & 0xFFFFu;
        s += *reinterpret_cast<const unsigned long long*>(reinterpret_cast<const char*>(q) + o);
        if (ends >> t & 1u) pre[at++] = s;
      }
      const unsigned long long inc = wave_inclusive_scan(s);
      lpre[tid] = inc - s;
      if (lane == 63) wtot[wave] = inc;
      __syncthreads();
      unsigned long long err = 0ull;
#pragma unroll
      for (uint32_t r = 0; r < kR; ++r) {
        const uint32_t i = tid + r * NT;
        if (i < n) {
          float z = 0.f;
          if (rk[r] != kNone) {
            const uint32_t t1 = lanes[r] & 0xFFFFu, t0 = lanes[r] >> 16;
            unsigned long long d = pre[rk[r]] + lpre[t1];
            if (rk[r]) d -= pre[rk[r] - 1] + lpre[t0];
            for (uint32_t w = t0 >> 6; w < t1 >> 6; ++w) d += wtot[w];
            z = dequantize(d);
          }
          const float xn = __builtin_fmaf(P.damp, z, b[r]);  // page_rank.hpp:133-135
          err += quantize(fabsf(xn - x[r]));  // in units of 2^-60
          x[r] = xn;
          q[i] = quantize(xn / (float)dg[r]);
        }
      }
      err = wave_sum(err);
      if (lane == 0) werr[wave] = err;
      __syncthreads();
      unsigned long long total = 0ull;
#pragma unroll
      for (uint32_t w = 0; w < kWaves; ++w) total += werr[w];
      total = (total + 2) >> 2;  // 2^-58, as every solve's changes
      if (tid == 0) {
        P.acc[k * P.ngraphs + g] = total;
        if (P.mail) P.mail[k] = total;
      }
      ++k;
      if (fixed_to_err(total) < P.threshold) break;  // page_rank.hpp:144
    }
  }
  for (k += tid; k < k1; k += NT) {
    P.acc[k * P.ngraphs + g] = 0ull;
    if (P.mail) P.mail[k] = 0ull;
  }
  const bool write = P.out && !(P.tele && !teleport_ok(*P.tele));
#pragma unroll
  for (uint32_t r = 0; r < kR; ++r) {
    const uint32_t i = tid + r * NT;
    if (i < n) {
      P.x[r0 + i] = x[r];
      if (write) P.out[P.order ? P.order[r0 + i] : r0 + i] = x[r];
    }
  }
}

template <uint32_t NT, uint32_t E>
bool fits(uint64_t n, uint64_t nnz) {
  return n <= kR * NT && nnz <= NT * E;
}

}  // namespace

// Measured on MI355X (R-MAT, 20 sweeps, us for a whole resident solve, here / one launch per sweep): 257 vertices
// 52 / 109, 1000 with 7 K edges 57 / 114, 1024 with 13 K 82 / 123, 1500 with 20 K 95 / 120, 2048 with 24 K 119 / 115;
// many graphs share the launches of the other side, but not its lanes: 63 of 256 to 1024 vertices
// 107 / 167, 96 of 256 to 2048 (up to 22 K edges) 146 / 201.
bool small_fits(uint64_t n, uint64_t nnz, bool many) {
  return many ? fits<1024, 24>(n, nnz) : fits<1024, 16>(n, nnz);
}

void small_enqueue(hipStream_t s, const SmallParams& P, uint64_t n, uint64_t nnz, uint64_t k0, uint64_t k1) {
  NWG_REQUIRE(small_fits(n, nnz, true) && k1 - k0 <= kSmallSweeps, "graph too large for one workgroup");
  if (fits<256, 16>(n, nnz)) small_solve_kernel<256, 16><<<P.ngraphs, 256, 0, s>>>(P, k0, k1);
  else if (fits<1024, 8>(n, nnz)) small_solve_kernel<1024, 8><<<P.ngraphs, 1024, 0, s>>>(P, k0, k1);
  else if (fits<1024, 16>(n, nnz)) small_solve_kernel<1024, 16><<<P.ngraphs, 1024, 0, s>>>(P, k0, k1);
  else small_solve_kernel<1024, 24><<<P.ngraphs, 1024, 0, s>>>(P, k0, k1);
  NWG_LAUNCH_CHECK();
}

}  // namespace nwg
