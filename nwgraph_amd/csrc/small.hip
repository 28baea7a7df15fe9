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
struct Shape {
  static_assert(E % 4 == 0 && E <= 24, "an edge window spans at most two words of row ends");
  static constexpr uint32_t kWaves = NT / 64, kRows = kR * NT, kWords = NT * E / 32;
  struct Shared {
    unsigned long long pre[kRows];  // by rank of the non-empty rows: the lane's sum up to their last edge
    unsigned long long lpre[NT];    // the lanes' sums before a lane in its wave
    unsigned long long wtot[kWaves];
    uint32_t bits[kWords + 1], word_pre[kWords + 1], wcnt[kWaves];
  };
  // what a lane keeps of the structure
  struct Lane {
    uint32_t rk[kR];     // its rows' ranks among the non-empty ones, or kNone
    uint32_t lanes[kR];  // lane of the row's last edge, and << 16 of the edge before its first one
    uint32_t first;      // rank of the row its first edge belongs to
    uint32_t ends;       // bit t: edge t is its row's last
  };

  // from the row pointers (rp[0 .. n], edges counted from rp[0])
  static __device__ __forceinline__ void setup(Shared& S, Lane& L, const uint32_t* __restrict__ rp, uint32_t n) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, eb = rp[0];
    uint32_t end[kR];
    for (uint32_t w = tid; w <= kWords; w += NT) S.bits[w] = 0u;
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < kR; ++r) {
      const uint32_t i = tid + r * NT;
      end[r] = kNone;
      L.lanes[r] = 0u;
      if (i < n) {
        const uint32_t a = rp[i] - eb, e = rp[i + 1] - eb;
        if (e > a) {
          end[r] = e - 1;
          L.lanes[r] = (e - 1) / E | (a ? (a - 1) / E : 0u) << 16;
          atomicOr(&S.bits[(e - 1) >> 5], 1u << ((e - 1) & 31u));
        }
      }
    }
    __syncthreads();
    // row ends before each word
    uint32_t run = 0;
    for (uint32_t w0 = 0; w0 <= kWords; w0 += NT) {
      const uint32_t w = w0 + tid;
      const uint32_t c = w <= kWords ? (uint32_t)__popc(S.bits[w]) : 0u;
      const uint32_t inc = wave_inclusive_scan(c);
      if (lane == 63) S.wcnt[wave] = inc;
      __syncthreads();
      uint32_t before = run;
      for (uint32_t v = 0; v < kWaves; ++v) {
        before += v < wave ? S.wcnt[v] : 0u;
        run += S.wcnt[v];
      }
      if (w <= kWords) S.word_pre[w] = before + inc - c;
      __syncthreads();
    }
    auto rank_of = [&](uint32_t p) {  // row ends before edge p
      return S.word_pre[p >> 5] + (uint32_t)__popc(S.bits[p >> 5] & ((1u << (p & 31u)) - 1u));
    };
#pragma unroll
    for (uint32_t r = 0; r < kR; ++r) L.rk[r] = end[r] == kNone ? kNone : rank_of(end[r]);
    const uint32_t p0 = tid * E;  // <= 32 kWords - E
    L.first = rank_of(p0);
    const uint64_t window = ((uint64_t)S.bits[(p0 >> 5) + 1] << 32) | S.bits[p0 >> 5];
    L.ends = (uint32_t)(window >> (p0 & 31u)) & ((1u << E) - 1u);
  }

  // the sources of the lane's edges as byte offsets in an array of `size` bytes per vertex, two to a
  // register; kRows for lanes past the edges
  static __device__ __forceinline__ void sources(uint32_t (&ids)[E / 2], const uint32_t* __restrict__ col, uint32_t r0,
                                                 uint32_t nnz, uint32_t size) {
    const uint32_t p0 = threadIdx.x * E;
#pragma unroll
    for (uint32_t t = 0; t < E; t += 2) {
      const uint32_t u = p0 + t < nnz ? col[p0 + t] - r0 : kRows;
      const uint32_t v = p0 + t + 1 < nnz ? col[p0 + t + 1] - r0 : kRows;
      ids[t / 2] = u * size | (v * size << 16);
    }
  }
  template <class T>
  static __device__ __forceinline__ T at(const T* base, const uint32_t (&ids)[E / 2], uint32_t t) {
    const uint32_t o = t % 2 ? ids[t / 2] >> 16 : ids[t / 2] & 0xFFFFu;
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + o);
  }

  // Step 1: value(t) of the lane's edge t; a barrier has to follow
  template <class F>
  static __device__ __forceinline__ void prefix(Shared& S, const Lane& L, F&& value) {
    unsigned long long s = 0ull;
    uint32_t rank = L.first;
#pragma unroll
    for (uint32_t t = 0; t < E; ++t) {
      s += value(t);
      if (L.ends >> t & 1u) S.pre[rank++] = s;
    }
    const unsigned long long inc = wave_inclusive_scan(s);
    S.lpre[threadIdx.x] = inc - s;
    if ((threadIdx.x & 63u) == 63u) S.wtot[threadIdx.x >> 6] = inc;
  }
  // Step 2: the sum of the lane's row r, which has edges
  static __device__ __forceinline__ unsigned long long row_sum(const Shared& S, const Lane& L, uint32_t r) {
    const uint32_t t1 = L.lanes[r] & 0xFFFFu, t0 = L.lanes[r] >> 16;
    unsigned long long d = S.pre[L.rk[r]] + S.lpre[t1];
    if (L.rk[r]) d -= S.pre[L.rk[r] - 1] + S.lpre[t0];
    for (uint32_t w = t0 >> 6; w < t1 >> 6; ++w) d += S.wtot[w];
    return d;
  }
};

template <uint32_t NT, uint32_t E>
__global__ __launch_bounds__(NT) void small_solve_kernel(SmallParams P, uint64_t k0, uint64_t k1) {
  using H = Shape<NT, E>;
  __shared__ typename H::Shared S;
  __shared__ unsigned long long q[H::kRows + 1];  // contributions; the last one is 0, for lanes past the edges
  __shared__ unsigned long long werr[H::kWaves];
  const uint32_t tid = threadIdx.x, g = blockIdx.x;
  if (P.bad) {
    const uint32_t b0 = P.bad[0], b1 = P.bad[1];
    if (g == 0 && tid < 2) P.bad_mail[tid] = tid ? b1 : b0;
    if (b0 | b1) return;
  }
  const uint32_t r0 = P.voff ? P.voff[g] : 0u;
  const uint32_t n = P.voff ? P.voff[g + 1] - r0 : P.n;
  if (!n) {
    for (uint64_t k = k0 + tid; k < k1; k += NT) P.acc[k * P.ngraphs + g] = 0ull;
    return;
  }
  const bool done = k0 > 0 && fixed_to_err(P.acc[(k0 - 1) * P.ngraphs + g]) < P.threshold;
  const uint32_t eb = P.rp[r0], nnz = P.rp[r0 + n] - eb;
  const float init = (float)(1.0 / n);  // page_rank.hpp:93
  float x[kR], b[kR];
  uint32_t dg[kR];
  CutNote cut;
#pragma unroll
  for (uint32_t r = 0; r < kR; ++r) {
    const uint32_t i = tid + r * NT;
    x[r] = 0.f;
    b[r] = 0.f;
    dg[r] = 0u;
    if (i < n) {
      dg[r] = P.deg[r0 + i];
      b[r] = P.basev ? P.basev[r0 + i] : P.base;
      x[r] = k0 ? P.x[r0 + i] : init;
      const float c = x[r] / (float)dg[r];
      q[i] = quantize(c);
      cut.note(c);
    }
  }
  if (tid == 0) q[H::kRows] = 0ull;
  uint32_t ids[E / 2];
  H::sources(ids, P.col + eb, r0, nnz, 8);
  typename H::Lane L;
  H::setup(S, L, P.rp + r0, n);  // with the barrier that q needs

  uint64_t k = k0;
  if (!done) {
    while (k < k1) {
      H::prefix(S, L, [&](uint32_t t) { return H::at(q, ids, t); });
      __syncthreads();
      unsigned long long err = 0ull;
#pragma unroll
      for (uint32_t r = 0; r < kR; ++r) {
        const uint32_t i = tid + r * NT;
        if (i < n) {
          const float z = L.rk[r] != kNone ? dequantize(H::row_sum(S, L, r)) : 0.f;
          const float xn = __builtin_fmaf(P.damp, z, b[r]);  // page_rank.hpp:133-135
          err += quantize(fabsf(xn - x[r]));  // in units of 2^-60
          x[r] = xn;
          const float c = xn / (float)dg[r];
          q[i] = quantize(c);
          cut.note(c);
        }
      }
      err = wave_sum(err);
      if ((tid & 63u) == 0) werr[tid >> 6] = err;
      __syncthreads();
      unsigned long long total = 0ull;
#pragma unroll
      for (uint32_t w = 0; w < H::kWaves; ++w) total += werr[w];
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
  if (__syncthreads_or(cut.cuts()) && tid == 0) *P.cut = 1ull;
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

// The weighted sweep (WItemParams in items.hpp): the iterate in LDS, the weights in registers, products
// quantized edge by edge, the L1 change a double.
template <uint32_t NT, uint32_t E>
__global__ __launch_bounds__(NT) void small_weighted_kernel(SmallWeighted P, uint64_t k0, uint64_t k1) {
  using H = Shape<NT, E>;
  __shared__ typename H::Shared S;
  __shared__ float xs[H::kRows + 1];  // the last one is 0, for lanes past the edges
  __shared__ double werr[H::kWaves];
  const uint32_t tid = threadIdx.x, n = P.n, nnz = P.rp[n];
  const double stop = P.thr_scale ? P.threshold * *P.thr_scale : P.threshold;
  const int qs = *P.qshift;
  float x[kR], b[kR];
#pragma unroll
  for (uint32_t r = 0; r < kR; ++r) {
    const uint32_t i = tid + r * NT;
    x[r] = 0.f;
    b[r] = 0.f;
    if (i < n) {
      b[r] = P.base[i];
      x[r] = k0 ? P.state[i] : P.y0 ? P.y0[i] : P.uniform;
      xs[i] = x[r];
    }
  }
  if (tid == 0) xs[H::kRows] = 0.f;
  uint32_t ids[E / 2];
  H::sources(ids, P.col, 0, nnz, 4);
  float w[E];
#pragma unroll
  for (uint32_t t = 0; t < E; ++t) w[t] = tid * E + t < nnz ? P.w[tid * E + t] : 0.f;
  typename H::Lane L;
  H::setup(S, L, P.rp, n);
  uint64_t k = k0;
  CutNote cut;
  while (k < k1) {
    H::prefix(S, L, [&](uint32_t t) {
      const float f = w[t] * H::at(xs, ids, t);
      cut.note(f);
      return quantize_signed(f, qs);
    });
    __syncthreads();
    double err = 0.0;
#pragma unroll
    for (uint32_t r = 0; r < kR; ++r) {
      const uint32_t i = tid + r * NT;
      if (i < n) {
        const float z = L.rk[r] != kNone ? dequantize_signed(H::row_sum(S, L, r), qs) : 0.f;
        const float xn = __builtin_fmaf(P.damp, z, b[r]);
        err += (double)fabsf(xn - x[r]);
        x[r] = xn;
        xs[i] = xn;
      }
    }
    err = wave_scan_dpp(err);
    if ((tid & 63u) == 63u) werr[tid >> 6] = err;
    __syncthreads();
    double total = 0.0;
#pragma unroll
    for (uint32_t v = 0; v < H::kWaves; ++v) total += werr[v];
    if (tid == 0) {
      P.err[k] = total;
      if (P.mail) P.mail[2 + k] = __double_as_longlong(total);
    }
    ++k;
    if (total < stop) break;
  }
  for (k += tid; k < k1; k += NT) {
    P.err[k] = 0.0;
    if (P.mail) P.mail[2 + k] = 0ull;
  }
  if (__syncthreads_or(cut.cuts(qs)) && tid == 0) *P.cut = 1ull;
  if (P.mail && tid < 2) P.mail[tid] = P.scale[tid];
#pragma unroll
  for (uint32_t r = 0; r < kR; ++r) {
    const uint32_t i = tid + r * NT;
    if (i < n) {
      P.state[i] = x[r];
      P.out[i] = x[r];
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
// 107 / 167, 96 of 256 to 2048 (up to 22 K edges) 146 / 201.  Weighted solve and its adjoint: 257 vertices
// 199 / 516, 1000 with 7 K edges 176 / 424, 2000 with 11 K 188 / 315.
bool small_fits(uint64_t n, uint64_t nnz, bool many) {
  return many ? fits<1024, 24>(n, nnz) : fits<1024, 20>(n, nnz);
}

void small_enqueue(hipStream_t s, const SmallParams& P, uint64_t n, uint64_t nnz, uint64_t k0, uint64_t k1) {
  NWG_REQUIRE(small_fits(n, nnz, true) && k1 - k0 <= kSmallSweeps, "graph too large for one workgroup");
  if (fits<256, 16>(n, nnz)) small_solve_kernel<256, 16><<<P.ngraphs, 256, 0, s>>>(P, k0, k1);
  else if (fits<1024, 8>(n, nnz)) small_solve_kernel<1024, 8><<<P.ngraphs, 1024, 0, s>>>(P, k0, k1);
  else if (fits<1024, 16>(n, nnz)) small_solve_kernel<1024, 16><<<P.ngraphs, 1024, 0, s>>>(P, k0, k1);
  else if (fits<1024, 20>(n, nnz)) small_solve_kernel<1024, 20><<<P.ngraphs, 1024, 0, s>>>(P, k0, k1);
  else small_solve_kernel<1024, 24><<<P.ngraphs, 1024, 0, s>>>(P, k0, k1);
  NWG_LAUNCH_CHECK();
}

void small_weighted_enqueue(hipStream_t s, const SmallWeighted& P, uint64_t nnz, uint64_t k0, uint64_t k1) {
  NWG_REQUIRE(small_fits(P.n, nnz, false) && k1 - k0 <= kSmallSweeps, "graph too large for one workgroup");
  if (fits<256, 16>(P.n, nnz)) small_weighted_kernel<256, 16><<<1, 256, 0, s>>>(P, k0, k1);
  else if (fits<1024, 8>(P.n, nnz)) small_weighted_kernel<1024, 8><<<1, 1024, 0, s>>>(P, k0, k1);
  else if (fits<1024, 16>(P.n, nnz)) small_weighted_kernel<1024, 16><<<1, 1024, 0, s>>>(P, k0, k1);
  else small_weighted_kernel<1024, 20><<<1, 1024, 0, s>>>(P, k0, k1);
  NWG_LAUNCH_CHECK();
}

}  // namespace nwg
