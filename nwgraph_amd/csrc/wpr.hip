// wpr.hip -- weighted PageRank forward, implicit adjoint and edge gradient.
//
// Forward (same fixed-point form as the reference loop, page_rank.hpp:121-147, with a
// per-edge transition weight instead of 1/outdeg and a teleport vector v):
//   x_i <- fma(d, z_i, (1-d) v_i),   z_i = sum_{p in CSC row i} w[p] * x[col[p]]
// Jacobi, x double-buffered, stop at the first sweep with L1 change < threshold.
// Adjoint of L(x) with g = dL/dx at the fixed point x = (1-d) v + d A x, A[i][u] = w(u->i):
//   lambda = g + d A^T lambda   -- solved by the same sweep in pull form over the CSR
// (row u gathers its out-edges u -> i: lambda_u <- fma(d, sum w(u->i) lambda_i, g_u)), so
// no unrolled forward iterate is stored and no atomics are needed.  Then
//   dL/dw(u->i) = d * lambda_i * x_u,   dL/dv = (1-d) lambda,
// and, for raw weights normalised per source (w = w~ / s_u, s_u = sum_k w~(u->k)),
//   dL/dw~(u->k) = (dL/dw(u->k) - sum_j dL/dw(u->j) w(u->j)) / s_u.
//
// Sweeps (weighted_sweep): one workgroup for small graphs (small.hip), the item sweep (items.hip), the
// binned sweep (binned.hip), all with exact fixed-point row sums; and the pull sweep here, in float, for
// what their bound does not cover: weights that are negative, not normalised or undefined, a teleport or
// gradient that is not finite, and large graphs whose plan is not binned.
//
// The pull sweep: the rows are cut into work items of up to 256 consecutive rows with at most
// kItemNnz nonzeros (values staged in LDS; one lane per short row, one wave per row of more than
// kLaneRow nonzeros) or one longer row (whole-workgroup reduction); a persistent grid walks the
// items round-robin.  Its L1 change is summed in double with a fixed order: every workgroup stores
// its partial, and the last workgroup to finish (a counter per sweep) adds all partials in
// workgroup order and stores err[k] (the other sweeps' changes are doubles too).  The adjoint's changes have no a-priori bound (a
// loss such as -sum log x gives |grad_x| ~ n), so a fixed-point accumulator of bounded
// range could wrap; this sum cannot, and it does not depend on completion order, so the
// sweep count is reproducible.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "device_utils.hpp"
#include "nwg_internal.hpp"
#include "small.hpp"

namespace nwg {

namespace {

constexpr int kThreads = 256;
constexpr uint32_t kItemNnz = 4096;
constexpr uint32_t kItemRows = 256;
constexpr uint32_t kGather = 8;    // gathers a lane issues before it uses them
constexpr uint32_t kLaneRow = 16;  // longest row summed by one lane; longer rows take a wave

struct WParams {
  const uint32_t* rp;
  const uint32_t* col;
  const float* w;
  const uint32_t* item_r0;
  const uint32_t* item_r1;
  uint32_t n_items;
  const float* base;  // per row: (1-d) v_i forward, g_u adjoint
  const float* xin;
  float* xout;
  float damp;
  double* part;    // per workgroup: L1 partial of the current sweep
  uint32_t* done;  // per sweep: workgroups that stored their partial
  double* err;     // per sweep: L1 change, stored by the sweep's last workgroup
  uint32_t iter;
  double threshold;
  const double* thr_scale;  // relative threshold: the stop compares with threshold * *thr_scale
};

__device__ __forceinline__ double stop_threshold(const WParams& P) {
  return P.thr_scale ? P.threshold * *P.thr_scale : P.threshold;
}

// Workgroup-order sum of the per-workgroup partials `e` (valid in thread 0) of sweep
// P.iter into P.err[P.iter], by whichever workgroup finishes last.
__device__ __forceinline__ void fold_sweep_error(const WParams& P, double e, double* red_d) {
  __shared__ uint32_t last;
  if (threadIdx.x == 0) {
    P.part[blockIdx.x] = e;
    __threadfence();  // release the partial before counting it
    last = atomicAdd(P.done + P.iter, 1u) == gridDim.x - 1 ? 1u : 0u;
  }
  __syncthreads();
  if (!last) return;
  __threadfence();  // acquire every other workgroup's partial
  double s = 0.0;
  for (uint32_t b = threadIdx.x; b < gridDim.x; b += kThreads)
    s += __hip_atomic_load(P.part + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  s = block_sum<kThreads>(s, red_d);
  if (threadIdx.x == 0) P.err[P.iter] = s;
}

__global__ __launch_bounds__(kThreads) void wsweep_kernel(WParams P) {
  if (P.iter > 0 && P.err[P.iter - 1] < stop_threshold(P)) return;
  __shared__ float vals[kItemNnz];
  __shared__ uint32_t lrows[kItemRows];   // an item's long rows (offsets from its first row)
  __shared__ uint32_t wlong[kThreads / 64];
  __shared__ float red_f[kThreads / 64];
  __shared__ double red_d[kThreads / 64];
  double e = 0.0;
  for (uint32_t it = blockIdx.x; it < P.n_items; it += gridDim.x) {
    const uint32_t r0 = P.item_r0[it], r1 = P.item_r1[it];
    const uint32_t p0 = P.rp[r0], p1 = P.rp[r1];
    if (p1 - p0 > kItemNnz) {
      // one long row: a lane's edges p0 + lane + t * kThreads, kGather gathers in flight,
      // added in that order
      float z = 0.f;
      for (uint32_t p = p0 + threadIdx.x; p < p1; p += kThreads * kGather) {
        uint32_t c[kGather];
        float wv[kGather], xv[kGather];
#pragma unroll
        for (uint32_t t = 0; t < kGather; ++t) {
          const uint32_t q = p + t * kThreads;
          c[t] = q < p1 ? P.col[q] : 0u;
          wv[t] = q < p1 ? P.w[q] : 0.f;
        }
#pragma unroll
        for (uint32_t t = 0; t < kGather; ++t) xv[t] = p + t * kThreads < p1 ? P.xin[c[t]] : 0.f;
#pragma unroll
        for (uint32_t t = 0; t < kGather; ++t)
          if (p + t * kThreads < p1) z = __builtin_fmaf(wv[t], xv[t], z);
      }
      z = block_sum<kThreads>(z, red_f);
      if (threadIdx.x == 0) {
        const float xn = __builtin_fmaf(P.damp, z, P.base[r0]);
        e += (double)fabsf(xn - P.xin[r0]);
        P.xout[r0] = xn;
      }
    } else {
      // stage the item's products w * x[col], kGather gathers of a lane in flight
      const uint32_t m = p1 - p0;
      for (uint32_t q0 = threadIdx.x; q0 < m; q0 += kThreads * kGather) {
        uint32_t c[kGather];
        float wv[kGather], xv[kGather];
#pragma unroll
        for (uint32_t t = 0; t < kGather; ++t) {
          const uint32_t q = q0 + t * kThreads;
          c[t] = q < m ? P.col[p0 + q] : 0u;
          wv[t] = q < m ? P.w[p0 + q] : 0.f;
        }
#pragma unroll
        for (uint32_t t = 0; t < kGather; ++t) xv[t] = q0 + t * kThreads < m ? P.xin[c[t]] : 0.f;
#pragma unroll
        for (uint32_t t = 0; t < kGather; ++t)
          if (q0 + t * kThreads < m) vals[q0 + t * kThreads] = wv[t] * xv[t];
      }
      __syncthreads();
      // rows of up to kLaneRow entries: one lane each, in row order; longer rows: one wave
      // each (lane-strided partial sums, then a butterfly), listed in row order through a
      // ballot so that every row's sum is computed the same way on every run
      const uint32_t i = r0 + threadIdx.x;
      uint32_t a = 0, b = 0;
      if (i < r1) {
        a = P.rp[i] - p0;
        b = P.rp[i + 1] - p0;
      }
      const bool longrow = b - a > kLaneRow;
      if (i < r1 && !longrow) {
        float z = 0.f;
        for (uint32_t q = a; q < b; ++q) z += vals[q];
        const float xn = __builtin_fmaf(P.damp, z, P.base[i]);
        e += (double)fabsf(xn - P.xin[i]);
        P.xout[i] = xn;
      }
      const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
      const unsigned long long lm = __ballot(longrow);
      if (lane == 0) wlong[wv] = (uint32_t)__popcll(lm);
      __syncthreads();
      uint32_t off = 0, nlong = 0;
      for (uint32_t q = 0; q < kThreads / 64; ++q) {
        off += q < wv ? wlong[q] : 0u;
        nlong += wlong[q];
      }
      if (longrow)
        lrows[off + __builtin_amdgcn_mbcnt_hi((uint32_t)(lm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)lm, 0u))] =
            threadIdx.x;
      __syncthreads();
      for (uint32_t k = wv; k < nlong; k += kThreads / 64) {
        const uint32_t ri = r0 + lrows[k];
        const uint32_t la = P.rp[ri] - p0, lb = P.rp[ri + 1] - p0;
        float z = 0.f;
        for (uint32_t q = la + lane; q < lb; q += 64) z += vals[q];
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) z += __shfl_xor(z, o, 64);
        if (lane == 0) {
          const float xn = __builtin_fmaf(P.damp, z, P.base[ri]);
          e += (double)fabsf(xn - P.xin[ri]);
          P.xout[ri] = xn;
        }
      }
      __syncthreads();
    }
  }
  e = block_sum<kThreads>(e, red_d);
  fold_sweep_error(P, e, red_d);
}

// y = v (src null) or y = src; the per-sweep counters and errors cleared
__global__ __launch_bounds__(kThreads) void winit_kernel(uint32_t n, const float* __restrict__ src, float v,
                                                         float* __restrict__ dst, uint32_t* __restrict__ done,
                                                         double* __restrict__ err, uint64_t iters) {
  const uint64_t t = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  if (t < n) dst[t] = src ? src[t] : v;
  if (t < iters) {
    done[t] = 0u;
    err[t] = 0.0;
  }
}

// What a solve scales its stop and its fixed point by, made on the device before its sweeps.
struct WScale {
  double scale;  // of a relative threshold: ||b||_1 / (1 - d), 1 for the uniform teleport and for b = 0
  int qshift;    // products are summed in units of 2^(-60 - qshift)
  int finite;    // b is finite
};

// The fixed point's constant term b into dst -- (float)((1-d) * v_i) for a forward solve (v null:
// uniform 1/n), v itself for an adjoint -- and per workgroup, over a contiguous range, the sum and
// the largest of |b| (NaN or infinity shows in the sum).
constexpr uint32_t kNormBlocks = 256;
__global__ __launch_bounds__(kThreads) void wprep_kernel(uint32_t n, const float* __restrict__ v, bool forward,
                                                         double omd, float* __restrict__ dst,
                                                         double* __restrict__ out) {
  __shared__ double red_d[kThreads / 64];
  const uint64_t per = ((uint64_t)n + gridDim.x - 1) / gridDim.x;
  const uint64_t i0 = (uint64_t)blockIdx.x * per, i1 = i0 + per < n ? i0 + per : n;
  double sum = 0.0, mx = 0.0;
  for (uint64_t i = i0 + threadIdx.x; i < i1; i += kThreads) {
    const float b = !forward ? v[i] : v ? (float)(omd * (double)v[i]) : (float)(omd / (double)n);
    dst[i] = b;
    const double a = (double)fabsf(b);
    sum += a;
    mx = a > mx ? a : mx;
  }
  sum = block_sum<kThreads>(sum, red_d);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const double y = __shfl_xor(mx, o, 64);
    mx = y > mx ? y : mx;
  }
  if ((threadIdx.x & 63) == 0) red_d[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t q = 0; q < kThreads / 64; ++q) mx = red_d[q] > mx ? red_d[q] : mx;
    out[2 * blockIdx.x] = sum;
    out[2 * blockIdx.x + 1] = mx;
  }
}

// Scale of the fixed point: 2^t with 2^t * 2M in [1/2, 1), M a bound of every product and partial
// row sum, from b (the constant term) in exact arithmetic:
//   forward  x' = b + d A x, x0 = 1/n: |sum_u w(u->i) x_u| <= ||x||_1 <= max(1, ||b||_1 / (1-d))
//            (A is column-stochastic: ||A x||_1 <= ||x||_1);
//   adjoint  l' = b + d A^T l, l0 = b: |sum_i w(u->i) l_i| <= ||l||_inf <= ||b||_inf / (1-d)
//            (each row of A^T sums to 1).
// The factor 2 covers the FP32 rounding of the iterates.  One workgroup, a fixed tree.
__global__ __launch_bounds__(kNormBlocks) void wscale_kernel(const double* __restrict__ stats, bool forward,
                                                             bool uniform, double omd, WScale* __restrict__ out) {
  __shared__ double red_d[kNormBlocks / 64];
  double mx = stats[2 * threadIdx.x + 1];
  const double sum = block_sum<kNormBlocks>(stats[2 * threadIdx.x], red_d);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const double y = __shfl_xor(mx, o, 64);
    mx = y > mx ? y : mx;
  }
  if ((threadIdx.x & 63) == 0) red_d[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t q = 0; q < kNormBlocks / 64; ++q) mx = red_d[q] > mx ? red_d[q] : mx;
    const double M = forward ? fmax(1.0, sum / omd) : mx / omd;
    int t = 0;
    if (M > 0.0 && isfinite(M)) (void)frexp(2.0 * M, &t);
    out->scale = uniform || !(sum > 0.0) ? 1.0 : sum / omd;
    out->qshift = -t;
    out->finite = isfinite(sum) ? 1 : 0;
  }
}

// out = the iterate of the solve's last sweep: sweep k leaves it in y[(k + 1) & 1], and the solve ended
// with the first sweep whose change is below the threshold, or after iters
__global__ __launch_bounds__(kThreads) void wout_kernel(uint32_t n, const float* __restrict__ y0,
                                                        const float* __restrict__ y1, const double* __restrict__ err,
                                                        uint32_t iters, double threshold,
                                                        const double* __restrict__ thr_scale,
                                                        float* __restrict__ out) {
  const double stop = thr_scale ? threshold * *thr_scale : threshold;
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t ended = iters;
  for (uint32_t k = 0; k < iters; k += 64) {
    const unsigned long long m = __ballot(k + lane < iters && err[k + lane] < stop);
    if (m) {
      ended = k + (uint32_t)__builtin_ctzll(m) + 1;
      break;
    }
  }
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n) out[i] = (ended & 1u) ? y1[i] : y0[i];
}

// the raw weights kept, and *bad = 1 when some weight is negative or not finite
__global__ __launch_bounds__(kThreads) void weight_copy_kernel(uint64_t nnz, const float* __restrict__ w,
                                                               float* __restrict__ raw, uint32_t* __restrict__ bad) {
  const uint64_t p = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  if (p >= nnz) return;
  const float v = w[p];
  raw[p] = v;
  if (!(v >= 0.f && v <= 3.402823466e38f)) *bad = 1u;
}

// row of every CSC position (upper bound in the row pointers)
__global__ __launch_bounds__(kThreads) void row_of_kernel(uint32_t n, uint64_t nnz, const uint32_t* __restrict__ rp,
                                                          uint32_t* __restrict__ row) {
  const uint64_t p = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  if (p >= nnz) return;
  uint32_t lo = 0, hi = n;  // first r with rp[r + 1] > p
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (rp[mid + 1] <= p) lo = mid + 1;
    else hi = mid;
  }
  row[p] = lo;
}

__global__ __launch_bounds__(64) void wclear_kernel(uint32_t* __restrict__ p) {
  if (threadIdx.x < 2) p[threadIdx.x] = 0u;
}

// *undefined = 1 when some weight is NaN: its source's raw weights sum to 0, or to no finite float
__global__ __launch_bounds__(kThreads) void normalise_kernel(uint64_t nnz, const uint32_t* __restrict__ col,
                                                             const float* __restrict__ w_raw,
                                                             const float* __restrict__ s, float* __restrict__ w,
                                                             uint32_t* __restrict__ undefined) {
  const uint64_t p = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  if (p >= nnz) return;
  const float v = w_raw[p] / s[col[p]];
  w[p] = v;
  if (v != v) *undefined = 1u;
}

__global__ __launch_bounds__(kThreads) void gather_kernel(uint64_t nnz, const uint32_t* __restrict__ perm,
                                                          const float* __restrict__ src, float* __restrict__ dst) {
  const uint64_t q = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  if (q < nnz) dst[q] = src[perm[q]];
}

// grad_w[p] = d * lambda[row(p)] * x[col[p]], one thread per CSC position
__global__ __launch_bounds__(kThreads) void edge_grad_kernel(uint64_t nnz, const uint32_t* __restrict__ row,
                                                             const uint32_t* __restrict__ col, float d,
                                                             const float* __restrict__ lambda,
                                                             const float* __restrict__ x, float* __restrict__ gw) {
  const uint64_t p = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  if (p < nnz) gw[p] = (d * lambda[row[p]]) * x[col[p]];
}

// The raw-weight gradient of edge p from u = col[p]:
//   (d lambda_row x_u - t_u) / s_u,  t_u = x_u m_u,  m_u = sum_j d lambda_j w(u->j),
// as (x_u / s_u) * (d lambda_row - m_u) with quotient and sum made once per source (ab): one gather of 8
// bytes per edge, and exactly 0 where the source has no other edge (w = 1, m_u = d lambda_row), as the
// three passes below gave.  Edge gradient, row sums over a gathered copy and chain rule as
// three passes took 885 us for 16 M edges on MI355X (the row sums 647: two scattered reads per edge,
// long rows one load at a time); row sums over items with the products made in place and this
// pass take 206 us.
__global__ __launch_bounds__(kThreads) void raw_grad_kernel(uint64_t nnz, const uint32_t* __restrict__ row,
                                                            const uint32_t* __restrict__ col, float d,
                                                            const float* __restrict__ lambda,
                                                            const float2* __restrict__ ab, float* __restrict__ gw) {
#pragma clang fp contract(off)  // the difference is of the rounded products that m_u adds up
  const uint64_t p = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  if (p >= nnz) return;
  const float2 q = ab[col[p]];
  gw[p] = q.x * (d * lambda[row[p]] - q.y);
}

__global__ __launch_bounds__(kThreads) void scale_kernel(uint32_t n, float a, const float* __restrict__ src,
                                                         float* __restrict__ dst) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n) dst[i] = a * src[i];
}

inline uint32_t grid1(uint64_t m) { return (uint32_t)ceil_div(m ? m : 1, kThreads); }

}  // namespace

// Work items over a compressed structure (host-side, from its row pointers).
void build_items(hipStream_t s, const uint32_t* rp_dev, uint32_t n, DevBuf<uint32_t>& r0, DevBuf<uint32_t>& r1,
                 uint32_t* count) {
  std::vector<uint32_t> rp((size_t)n + 1);
  NWG_HIP(hipMemcpyAsync(rp.data(), rp_dev, ((size_t)n + 1) * 4, hipMemcpyDeviceToHost, s));
  NWG_HIP(hipStreamSynchronize(s));
  std::vector<uint32_t> a, b;
  uint64_t r = 0;
  while (r < n) {
    uint64_t e = r + 1;
    if (rp[e] - rp[r] <= kItemNnz)
      while (e < n && e - r < kItemRows && rp[e + 1] - rp[r] <= kItemNnz) ++e;
    a.push_back((uint32_t)r);
    b.push_back((uint32_t)e);
    r = e;
  }
  r0.alloc(std::max<size_t>(a.size(), 1));
  r1.alloc(std::max<size_t>(b.size(), 1));
  if (!a.empty()) {
    NWG_HIP(hipMemcpyAsync(r0.p, a.data(), a.size() * 4, hipMemcpyHostToDevice, s));
    NWG_HIP(hipMemcpyAsync(r1.p, b.data(), b.size() * 4, hipMemcpyHostToDevice, s));
  }
  NWG_HIP(hipStreamSynchronize(s));
  *count = (uint32_t)a.size();
}

static uint32_t persistent_grid(uint32_t n_items) {
  int dev = 0, cus = 0;
  NWG_HIP(hipGetDevice(&dev));
  NWG_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(n_items, (uint64_t)cus * 8));
}

// the class items of the pull sweep over a compressed structure, built on first use
static void ensure_pull_items(hipStream_t s, nwg_graph* g, bool csr) {
  uint32_t& count = csr ? g->w_items_csr_n : g->w_items_csc_n;
  if (count || !g->n) return;
  if (csr) build_items(s, g->csr_ptr.p, g->n, g->w_items_csr_r0, g->w_items_csr_r1, &count);
  else build_items(s, g->csc_ptr.p, g->n, g->w_items_csc_r0, g->w_items_csc_r1, &count);
}

// items (items.hip) of the CSC or CSR, built on first use
static const WItems& ensure_items(hipStream_t s, nwg_graph* g, bool csr) {
  WItems& it = csr ? g->wi_csr : g->wi_csc;
  if (!it.desc.n) {
    it.count = item_count(g->n, g->nnz);
    it.desc.alloc(it.count);
    items_build(s, g->n, g->nnz, csr ? g->csr_ptr.p : g->csc_ptr.p, it.desc.p, nullptr);
  }
  return it;
}

// s_u over the CSR's rows (items.hip, RowSumParams)
static void csr_row_sums(hipStream_t s, nwg_graph* g, const uint32_t* idx, const float* src, const float* gather,
                         float d, const RowSumOut& out) {
  const WItems& it = ensure_items(s, g, true);
  DevBuf<double> pieces(2ull * it.count);
  RowSumParams R{};
  R.desc = it.desc.p;
  R.rp = g->csr_ptr.p;
  R.idx = idx;
  R.src = src;
  R.gather = gather;
  R.d = d;
  R.nnz = (uint32_t)g->nnz;
  R.count = it.count;
  R.head = pieces.p;
  R.tail = pieces.p + it.count;
  row_sums_enqueue(s, R, out);
}

void weights_set(hipStream_t s, nwg_graph* g, const float* w_dev, bool normalize) {
  const uint64_t nnz = g->nnz;
  build_csr_device(s, g);
  g->w_raw.ensure(nnz ? nnz : 1);
  g->w_csc.ensure(nnz ? nnz : 1);
  g->w_csr.ensure(nnz ? nnz : 1);
  g->w_rowsum.ensure(g->n);
  // raw weights all finite and >= 0, and every source's sum finite and above 0: the fixed-point bound of
  // the exact weighted sweeps holds
  DevBuf<uint32_t> bad(2);
  wclear_kernel<<<1, 64, 0, s>>>(bad.p);
  if (nnz) weight_copy_kernel<<<grid1(nnz), kThreads, 0, s>>>(nnz, w_dev, g->w_raw.p, bad.p);
  NWG_LAUNCH_CHECK();
  if (normalize) {
    RowSumOut o{};
    o.out = g->w_rowsum.p;
    csr_row_sums(s, g, g->csr_to_csc.p, g->w_raw.p, nullptr, 0.f, o);
    if (nnz)
      normalise_kernel<<<grid1(nnz), kThreads, 0, s>>>(nnz, g->csc_idx.p, g->w_raw.p, g->w_rowsum.p, g->w_csc.p,
                                                       bad.p + 1);
    NWG_LAUNCH_CHECK();
  } else {
    std::vector<float> ones(g->n, 1.0f);
    NWG_HIP(hipMemcpyAsync(g->w_rowsum.p, ones.data(), (size_t)g->n * 4, hipMemcpyHostToDevice, s));
    if (nnz) NWG_HIP(hipMemcpyAsync(g->w_csc.p, w_dev, nnz * 4, hipMemcpyDeviceToDevice, s));
    NWG_HIP(hipStreamSynchronize(s));  // before ones goes
  }
  if (nnz) gather_kernel<<<grid1(nnz), kThreads, 0, s>>>(nnz, g->csr_to_csc.p, g->w_csc.p, g->w_csr.p);
  NWG_LAUNCH_CHECK();
  uint32_t hb[2] = {0, 0};
  NWG_HIP(hipMemcpyAsync(hb, bad.p, sizeof hb, hipMemcpyDeviceToHost, s));
  NWG_HIP(hipStreamSynchronize(s));
  g->has_weights = true;
  g->w_normalized = normalize;
  g->w_nonneg = hb[0] == 0;
  g->w_undefined = hb[1] != 0;
  if (g->wst) {  // the weighted layouts carry the old weights
    g->wst->bl_csc.reset();
    g->wst->bl_csr.reset();
  }
}

// Items up to which every workgroup adds the previous sweep's parts itself (16 KiB of them, behind
// its gathers).
constexpr uint32_t kItemsFolding = 1024;

// The sweep a weighted solve runs.  The exact sweeps (items, binned) need the weights normalised per
// source from non-negative raw weights: then every weight is in [0, 1] and each source's out-weights
// sum to 1, which the fixed-point bound (wscale_kernel) relies on.
enum class WSweep { kPull, kItems, kBinned };

// One fixed point y <- fma(d, sum w y, b) to solve: over the CSC (forward) or the CSR (adjoint).
struct WSolve {
  bool csr;
  const uint32_t* rp;
  const uint32_t* col;
  const float* w;
  const float* base;  // b
  const float* y0;    // first iterate; null: uniform 1/n
  bool uniform;       // b is the uniform teleport's (a relative threshold is then absolute)
  float damping, threshold;
  uint64_t max_iters;
  float* out;
};

// Runs the fixed point in the cached buffers of `st` and leaves the last iterate in q.out.  L: the layout
// of a binned sweep.  The init and the max_iters sweeps run as HIP graphs of a segment of sweeps each,
// captured into caps (again when a buffer, the layout or a parameter changes), so the host launches
// one graph per segment; base and y0 must be buffers that stay the same from call to call.  st.scale
// holds the solve's WScale.  Between segments the host reads the sweeps' changes.  `then` queues
// what follows the solve; with eager it is queued behind every segment before the changes are
// read, so that a solve that ends in its first segment waits for the device once.  one: a small graph's
// solve is one workgroup's.
enum class WEnd {
  kDone,
  kNotFinite,  // b was not finite: an exact sweep is then no answer
  kCut,        // the one workgroup's fixed point was too coarse: the item sweep is not
};
template <class F>
static WEnd fixed_point(nwg_ctx* ctx, nwg_graph* g, WState& st, std::vector<std::unique_ptr<Captured>>& caps,
                        const WSolve& q, WSweep kind, const BinnedLayout* L, nwg_pr_info* info, bool one, bool eager,
                        F&& then) {
  hipStream_t s = ctx->stream;
  const uint32_t n = g->n;
  const uint64_t max_iters = q.max_iters;
  st.y0.ensure(n);
  st.y1.ensure(n);
  st.done.ensure(std::max<uint64_t>(max_iters, 1));
  st.err.ensure(std::max<uint64_t>(max_iters, 1));
  float* y[2] = {st.y0.p, st.y1.p};
  const bool relative = info && (info->flags & NWG_INFO_RELATIVE_THRESHOLD);
  const double* thr_scale = relative ? &reinterpret_cast<const WScale*>(st.scale.p)->scale : nullptr;
  const int* qshift = &reinterpret_cast<const WScale*>(st.scale.p)->qshift;
  const WItems* it = nullptr;
  uint32_t grid = 0;
  if (kind == WSweep::kItems) {
    it = &ensure_items(s, g, q.csr);
    st.ihsum.ensure(it->count);
    st.ihcnt.ensure(it->count);
    st.ipart.ensure(4ull * it->count);
  } else if (kind == WSweep::kBinned) {
    st.bvals.ensure(L->pairs);
    st.bpart.ensure(std::max<uint64_t>((uint64_t)L->n_slots << L->bin_bits, 1));
    st.wpart.ensure(std::max<uint64_t>((uint64_t)L->n_items2 + L->n_items3, 1));
  } else {
    ensure_pull_items(s, g, q.csr);
    grid = persistent_grid(q.csr ? g->w_items_csr_n : g->w_items_csc_n);
    st.part.ensure(grid);
  }
  unsigned long long* const mail = kind != WSweep::kPull && max_iters && max_iters + 2 <= kMailWords ? ctx->mail : nullptr;
  auto segment_mail = [&](uint64_t k0) {
    return WMail{mail, reinterpret_cast<const unsigned long long*>(st.scale.p), (uint32_t)k0};
  };
  // sweeps [k0, k1) (and the init with k0 = 0) on stream t
  const float uniform = (float)(1.0 / n);
  auto enqueue = [&](hipStream_t t, uint64_t k0, uint64_t k1) {
    const float* src = q.y0;
    if (kind == WSweep::kItems) {
      WItemParams I{};
      I.desc = it->desc.p;
      I.rp = q.rp;
      I.col = q.col;
      I.w = q.w;
      I.basev = q.base;
      I.damp = q.damping;
      I.n = n;
      I.nnz = (uint32_t)g->nnz;
      I.count = it->count;
      I.qshift = qshift;
      I.hsum = st.ihsum.p;
      I.hcnt = st.ihcnt.p;
      I.part = st.ipart.p;
      I.err = st.err.p;
      I.threshold = (double)q.threshold;
      I.thr_scale = thr_scale;
      if (k0 == 0) witems_enqueue_init(t, I, src, uniform, y[0], max_iters);
      I.folded = it->count > kItemsFolding;
      for (uint64_t k = k0; k < k1; ++k) {
        I.iter = (uint32_t)k;
        I.xin = y[k & 1];
        I.xout = y[(k + 1) & 1];
        witems_enqueue_sweep(t, I);
        if (I.folded && k + 1 < k1) witems_enqueue_fold(t, I, (uint32_t)k, WMail{});
      }
      if (k1 > k0) witems_enqueue_fold(t, I, (uint32_t)(k1 - 1), segment_mail(k0));
      return;
    }
    if (k0 == 0) {
      winit_kernel<<<grid1(std::max<uint64_t>(n, max_iters)), kThreads, 0, t>>>(n, src, uniform, y[0], st.done.p,
                                                                               st.err.p, max_iters);
      NWG_LAUNCH_CHECK();
    }
    if (kind == WSweep::kBinned) {
      // x double-buffered as y[k & 1] -> y[(k + 1) & 1]; the L1 change goes to st.err
      BinParams B{};
      B.brow = L->brow.p;
      B.bsrc = L->bsrc.p;
      B.bpid = L->bpid.p;
      B.vals = st.bvals.p;
      B.items2 = L->items2.p;
      B.items1 = L->items1.p;
      B.items3 = L->items3.p;
      B.seg_start = L->seg_start.p;
      B.seg_flat = L->seg_flat.p;
      B.part = st.bpart.p;
      B.item_he = L->item_he.p;
      B.item_hd = L->item_hd.p;
      B.hsrc = L->hsrc.p;
      B.n_hot = L->n_hot;
      B.basev = q.base;
      B.damp = q.damping;
      B.n = n;
      B.n_items1 = L->n_items1;
      B.n_items2 = L->n_items2;
      B.bin_bits = L->bin_bits;
      B.n_items3 = L->n_items3;
      B.threshold = (double)q.threshold;
      B.thr_scale = thr_scale;
      B.bw = L->bw.p;
      B.qshift = qshift;
      B.wpart = st.wpart.p;
      B.werr = st.err.p;
      for (uint64_t k = k0; k < k1; ++k) {
        B.iter = (uint32_t)k;
        B.cin = y[k & 1];
        B.x = y[(k + 1) & 1];
        binned_enqueue_weighted_sweep(t, B);
      }
      if (k1 > k0) binned_enqueue_weighted_fold(t, B, segment_mail(k0));
      return;
    }
    WParams P{};
    P.rp = q.rp;
    P.col = q.col;
    P.w = q.w;
    P.item_r0 = q.csr ? g->w_items_csr_r0.p : g->w_items_csc_r0.p;
    P.item_r1 = q.csr ? g->w_items_csr_r1.p : g->w_items_csc_r1.p;
    P.n_items = q.csr ? g->w_items_csr_n : g->w_items_csc_n;
    P.base = q.base;
    P.damp = q.damping;
    P.part = st.part.p;
    P.done = st.done.p;
    P.err = st.err.p;
    P.threshold = (double)q.threshold;
    P.thr_scale = thr_scale;
    for (uint64_t k = k0; k < k1; ++k) {
      P.iter = (uint32_t)k;
      P.xin = y[k & 1];
      P.xout = y[(k + 1) & 1];
      wsweep_kernel<<<grid, kThreads, 0, t>>>(P);
      NWG_LAUNCH_CHECK();
    }
  };
  CaptureKey key;
  const void* ptrs[CaptureKey::kPtrs] = {st.y0.p, st.y1.p, q.base, q.y0, st.err.p, st.done.p, q.rp, q.col, q.w,
                                         st.scale.p, kind == WSweep::kPull ? (void*)st.part.p : (void*)mail,
                                         L ? st.bvals.p : nullptr, L ? st.bpart.p : nullptr, L ? st.wpart.p : nullptr,
                                         it ? st.ihsum.p : nullptr, it ? (void*)st.ipart.p : nullptr};
  for (int k = 0; k < CaptureKey::kPtrs; ++k) key.ptrs[k] = ptrs[k];
  key.iters = max_iters;
  key.damping = q.damping;
  key.threshold = q.threshold;
  // the layout's device arrays stand behind its build number: a layout made after the weights
  // changed may sit at the old one's host address
  key.plan_version = L ? L->build_id : grid;
  key.extra = (relative ? 1u : 0u) | (q.y0 ? 0u : 2u) | ((uint32_t)kind << 2);
  const uint64_t first = kind == WSweep::kBinned ? kSegFirstBinned : kSegFirst;
  // a small graph: all sweeps in one launch
  const bool small = one && kind == WSweep::kItems && small_fits(n, g->nnz, false);
  SmallWeighted sp{};
  if (small) {
    sp.rp = q.rp;
    sp.col = q.col;
    sp.w = q.w;
    sp.base = q.base;
    sp.y0 = q.y0;
    sp.uniform = uniform;
    sp.damp = q.damping;
    sp.n = n;
    sp.state = st.y0.p;
    sp.out = q.out;
    sp.qshift = qshift;
    sp.err = st.err.p;
    sp.mail = mail;
    sp.cut = ctx->mail + kMailCut;
    *sp.cut = 0ull;
    sp.scale = reinterpret_cast<const unsigned long long*>(st.scale.p);
    sp.threshold = (double)q.threshold;
    sp.thr_scale = thr_scale;
  }
  std::vector<double> h(std::max<uint64_t>(max_iters, 1), 0.0);
  WScale sc{1.0, 0, 1};
  double stop = (double)q.threshold;
  uint64_t iters = max_iters, seg = 0;
  NWG_HIP(hipEventRecord(ctx->ev0, s));
  auto end_of = [&](uint64_t k0) {
    return small ? std::min(k0 + kSmallSweeps, max_iters) : segment_end(k0, max_iters, first);
  };
  for (uint64_t k0 = 0;; k0 = end_of(k0), ++seg) {
    const uint64_t k1 = end_of(k0);
    if (small) small_weighted_enqueue(s, sp, g->nnz, k0, k1);
    else run_segment(ctx, caps, seg, key, [&](hipStream_t t) { enqueue(t, k0, k1); });
    NWG_HIP(hipEventRecord(ctx->ev1, s));
    if (!small)
      wout_kernel<<<grid1(n), kThreads, 0, s>>>(n, y[0], y[1], st.err.p, (uint32_t)k1, (double)q.threshold, thr_scale,
                                             q.out);
    NWG_LAUNCH_CHECK();
    if (eager) then();
    if (!mail && k0 == 0 && (relative || kind != WSweep::kPull))
      NWG_HIP(hipMemcpyAsync(&sc, st.scale.p, sizeof sc, hipMemcpyDeviceToHost, s));
    if (!mail && k1 > k0)
      NWG_HIP(hipMemcpyAsync(h.data() + k0, st.err.p + k0, (k1 - k0) * sizeof(double), hipMemcpyDeviceToHost, s));
    NWG_HIP(hipStreamSynchronize(s));
    if (mail) {
      std::memcpy(&sc, mail, sizeof sc);
      std::memcpy(h.data() + k0, mail + 2 + k0, (k1 - k0) * sizeof(double));
    }
    if (kind != WSweep::kPull && !sc.finite) return WEnd::kNotFinite;
    if (small && *sp.cut) return WEnd::kCut;
    if (relative) stop = (double)q.threshold * sc.scale;
    bool ended = k1 >= max_iters;
    for (uint64_t k = k0; k < k1; ++k)
      if (h[k] < stop) {
        iters = k + 1;
        ended = true;
        break;
      }
    if (ended) break;
  }
  if (!eager) then();
  if (info) {
    float ms = 0.f;
    NWG_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    info->iterations = iters;
    info->final_error = iters ? h[iters - 1] : 0.0;
    info->ms_total = ms;
    info->ms_per_iter = iters ? ms / (double)iters : 0.0;
    info->sweep_ms_avg = 0.0;
    info->threshold_used = stop;
    if (info->error_trace)
      for (uint64_t k = 0; k < iters && k < info->error_trace_len; ++k) info->error_trace[k] = h[k];
  }
  return WEnd::kDone;
}

static WState& wstate(nwg_graph* g) {
  if (!g->wst) g->wst.reset(new WState());
  return *g->wst;
}

// Weighted sweeps over items up to kItemsWeighted items (2.6 M rows and edges).  Measured on MI355X
// (RMAT, us per sweep, items / binned): 53 K edges 5.9 / 19.9, 228 K 7.2 / 23.1, 842 K 9.9 / 20.3, 1.9 M 17.7 / 23.5,
// 3.9 M 32.1 / 26.2.
// Above, and where the plan names a bin size, the binned sweep when the plan (or, before any plan,
// its size) asks for it.  Weights that are undefined (0 / 0) show as NaN in the pull sweep, which takes the
// items' place for them; the binned layout carries them as 0, so that its sweeps drop their sources' mass.
constexpr uint32_t kItemsWeighted = 2560;
static WSweep weighted_sweep(const nwg_graph* g, float damping) {
  if (!g->w_normalized || !g->w_nonneg || g->nnz == 0) return WSweep::kPull;
  const nwg_plan_params pp = g->plan.built ? g->plan.params : default_plan_for(g);
  if (pp.binned && pp.bin_bits) return WSweep::kBinned;
  if (!g->w_undefined && item_count(g->n, g->nnz) <= kItemsWeighted && damping >= 0.f && damping < 1.f) return WSweep::kItems;
  return pp.binned ? WSweep::kBinned : WSweep::kPull;
}

static const BinnedLayout* weighted_layout(hipStream_t s, nwg_graph* g, WState& st, bool csr) {
  std::unique_ptr<BinnedLayout>& L = csr ? st.bl_csr : st.bl_csc;
  const int bits = (int)(g->plan.built ? g->plan.params : default_plan_for(g)).bin_bits;
  if (L && bits && L->bin_bits != bits) L.reset();  // the plan asks for other bins
  if (!L) {
    L.reset(new BinnedLayout());
    const ActiveCsc a = csr ? ActiveCsc{g->csr_ptr.p, g->csr_idx.p, nullptr, nullptr}
                            : ActiveCsc{g->csc_ptr.p, g->csc_idx.p, g->outdeg.p, nullptr};
    try {
      binned_build(s, a, g->n, g->nnz, *L, true, csr ? g->w_csr.p : g->w_csc.p, bits);
      L->build_id = ++st.layouts_built;
    } catch (...) {
      L.reset();
      throw;
    }
  }
  return L.get();
}

// b, its scale and statistics, on the device
static void prepare_scale(hipStream_t s, WState& st, uint32_t n, const float* v, bool forward, float damping,
                          float* b) {
  const double omd = 1.0 - (double)damping;
  st.stats.ensure(2 * kNormBlocks);
  st.scale.ensure(sizeof(WScale) / sizeof(double));
  wprep_kernel<<<kNormBlocks, kThreads, 0, s>>>(n, v, forward, omd, b, st.stats.p);
  wscale_kernel<<<1, kNormBlocks, 0, s>>>(st.stats.p, forward, forward && !v, omd,
                                          reinterpret_cast<WScale*>(st.scale.p));
  NWG_LAUNCH_CHECK();
}

// solves q with the graph's sweep, or with the pull sweep when b was not finite (which shows the NaN /
// infinity as the reference would).  again: `then` can be queued more than once.
template <class F>
static void weighted_solve(nwg_ctx* ctx, nwg_graph* g, WState& st, std::vector<std::unique_ptr<Captured>>& caps,
                           const WSolve& q, nwg_pr_info* info, bool again, F&& then) {
  const WSweep kind = weighted_sweep(g, q.damping);
  const BinnedLayout* L = kind == WSweep::kBinned ? weighted_layout(ctx->stream, g, st, q.csr) : nullptr;
  const bool eager = again && kind == WSweep::kItems;
  WEnd end = fixed_point(ctx, g, st, caps, q, kind, L, info, true, eager, then);
  if (end == WEnd::kCut) end = fixed_point(ctx, g, st, caps, q, kind, L, info, false, eager, then);
  if (end == WEnd::kNotFinite)
    (void)fixed_point(ctx, g, st, caps, q, WSweep::kPull, nullptr, info, false, false, then);
}

void wpr_forward(nwg_ctx* ctx, nwg_graph* g, const float* teleport_dev, float* x_dev, float damping, float threshold,
                 uint64_t max_iters, nwg_pr_info* info) {
  hipStream_t s = ctx->stream;
  NWG_REQUIRE(g->has_weights, "graph has no weights (nwg_graph_set_weights)");
  NWG_REQUIRE(max_iters < (1ull << 31), "max_iters too large");
  WState& st = wstate(g);
  st.base.ensure(g->n);
  prepare_scale(s, st, g->n, teleport_dev, true, damping, st.base.p);
  WSolve q{};
  q.rp = g->csc_ptr.p;
  q.col = g->csc_idx.p;
  q.w = g->w_csc.p;
  q.base = st.base.p;
  q.uniform = !teleport_dev;
  q.damping = damping;
  q.threshold = threshold;
  q.max_iters = max_iters;
  q.out = x_dev;
  weighted_solve(ctx, g, st, st.cap_fwd, q, info, true, [] {});
  NWG_HIP(hipStreamSynchronize(s));
}

void wpr_backward(nwg_ctx* ctx, nwg_graph* g, const float* x_dev, const float* gx_dev, float* gw_dev, float* gv_dev,
                  float damping, float threshold, uint64_t max_iters, bool raw, nwg_pr_info* info) {
  hipStream_t s = ctx->stream;
  NWG_REQUIRE(g->has_weights, "graph has no weights (nwg_graph_set_weights)");
  NWG_REQUIRE(max_iters < (1ull << 31), "max_iters too large");
  NWG_REQUIRE(!raw || g->w_normalized, "raw-weight gradients need weights set with normalize=1");
  build_csr_device(s, g);
  const uint32_t n = g->n;
  const uint64_t nnz = g->nnz;
  WState& st = wstate(g);
  st.lambda.ensure(n);
  // adjoint fixed point: lambda = g + d A^T lambda, started from g; grad_x in a fixed buffer, so
  // that the captured loop serves every call
  st.gin.ensure(n);
  prepare_scale(s, st, n, gx_dev, false, damping, st.gin.p);
  WSolve q{};
  q.csr = true;
  q.rp = g->csr_ptr.p;
  q.col = g->csr_idx.p;
  q.w = g->w_csr.p;
  q.base = st.gin.p;
  q.y0 = st.gin.p;
  q.damping = damping;
  q.threshold = threshold;
  q.max_iters = max_iters;
  q.out = st.lambda.p;
  const bool edges = gw_dev && nnz;
  if (edges && !st.row_of.n) {
    st.row_of.alloc(nnz);
    row_of_kernel<<<grid1(nnz), kThreads, 0, s>>>(n, nnz, g->csc_ptr.p, st.row_of.p);
    NWG_LAUNCH_CHECK();
  }
  if (edges && raw) st.ab.ensure(n);
  weighted_solve(ctx, g, st, st.cap_adj, q, info, gv_dev != x_dev, [&] {
    if (edges && raw) {
      RowSumOut o{};
      o.x = x_dev;
      o.norm = g->w_rowsum.p;
      o.ab = st.ab.p;
      o.gv = gv_dev;
      o.omd = 1.0f - damping;
      csr_row_sums(s, g, g->csr_idx.p, g->w_csr.p, st.lambda.p, damping, o);
      raw_grad_kernel<<<grid1(nnz), kThreads, 0, s>>>(nnz, st.row_of.p, g->csc_idx.p, damping, st.lambda.p, st.ab.p,
                                                      gw_dev);
    } else {
      if (edges)
        edge_grad_kernel<<<grid1(nnz), kThreads, 0, s>>>(nnz, st.row_of.p, g->csc_idx.p, damping, st.lambda.p, x_dev,
                                                         gw_dev);
      if (gv_dev) scale_kernel<<<grid1(n), kThreads, 0, s>>>(n, 1.0f - damping, st.lambda.p, gv_dev);
    }
    NWG_LAUNCH_CHECK();
  });
  NWG_HIP(hipStreamSynchronize(s));
}

}  // namespace nwg
