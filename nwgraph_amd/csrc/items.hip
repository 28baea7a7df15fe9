// items.hip -- PageRank sweep over edge-balanced work items, one launch per sweep.
//
// The sweep is the reference's (include/nwgraph/algorithms/page_rank.hpp:121-147, Jacobi form
// experimental/algorithms/page_rank.hpp:397-430).  It serves graphs whose contributions stay in
// L2, where a sweep is bound by launches, by load latency and by its longest rows, not by bytes:
// row classes with a launch each take up to seven launches per sweep, and one wave on a row of
// thousands of in-edges outlasts everything else.
//
// Row i starts at unit D(i) = i + rp[i] of n + nnz units (one per edge, one per row), and item c
// owns the units [c S, (c + 1) S), S = 4 * threads:
//   * every row of at most S in-edges that starts in the window, whole (its edges may reach
//     into the next window: at most 2 S edges are staged);
//   * of a longer row, the edges whose units fall in the window.  Its pieces lie in consecutive
//     items; each adds its exact sum to the counter of the item the row starts in, and the
//     last piece to arrive finishes the row.
// So no item walks more than 2 S edges or S rows, whatever the degrees.
//
// An item is one workgroup.  Lane t takes 4 (or 8) consecutive edges: one 16-byte load of ids
// each, all gathers in flight together; the values, in 64-bit fixed point, are summed into a
// running prefix over the item (lane, then wave, then workgroup), and row i's sum is the
// difference of the prefix at its two ends.  The sums are exact integers, so the difference is
// the row's exact sum: short and long rows cost the same, nothing diverges, and the result
// depends on no order (fixed_point.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_utils.hpp"
#include "fixed_point.hpp"
#include "items.hpp"
#include "nwg_internal.hpp"

namespace nwg {

namespace {

constexpr uint32_t kHeadPiece = 1u << 30;  // the item's first edges belong to a long row begun before it
constexpr uint32_t kTailPiece = 1u << 31;  // its last edges to a long row that goes on after it
constexpr uint32_t kRowMask = kHeadPiece - 1;

// units per item; an item stages at most 2 span - 2 edges, and 3 before them for alignment, in
// the 8 NT places it has
__host__ __device__ constexpr uint32_t item_span(uint32_t threads) { return 4u * threads - 4u; }

// first row i in [0, n] with i + rp[i] >= unit (n if none)
__device__ __forceinline__ uint32_t first_row_from(const uint32_t* __restrict__ rp, uint32_t n, uint64_t unit) {
  uint32_t lo = 0, hi = n;
  while (lo < hi) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    if ((uint64_t)mid + rp[mid] >= unit) hi = mid;
    else lo = mid + 1;
  }
  return lo;
}

// One thread per item.  desc = {e0, e1, r0, rows | flags}: rows [r0, r0 + rows) are finished by
// the item, their edges lie in [e0, e1) after the head piece (of row r0 - 1) and before the
// tail piece (of row r0 + rows).
__global__ __launch_bounds__(256) void item_desc_kernel(uint32_t n, uint64_t nnz, const uint32_t* __restrict__ rp,
                                                        uint32_t span, uint32_t count, uint4* __restrict__ desc) {
  const uint32_t c = blockIdx.x * 256 + threadIdx.x;
  if (c >= count) return;
  const uint64_t u0 = (uint64_t)c * span, u1 = u0 + span;
  const uint32_t r0 = first_row_from(rp, n, u0), r1 = first_row_from(rp, n, u1);
  const uint32_t p0 = rp[r0], p1 = rp[r1];
  uint32_t e0 = p0, e1 = p1, rows = r1 - r0, flags = 0;
  // row r0 - 1: a long one whose last edge (unit r0 - 1 + p0 - 1) is not before the window
  if (r0 > 0 && p0 - rp[r0 - 1] > span && (uint64_t)(r0 - 1) + p0 > u0) {
    flags |= kHeadPiece;
    e0 = (uint32_t)(u0 - (r0 - 1));
    if (!rows) e1 = (uint32_t)min((uint64_t)p0, u1 - (r0 - 1));  // no row starts here: it may go on after the window
  }
  if (rows && p1 - rp[r1 - 1] > span) {  // the last row that starts here is a long one
    --rows;
    flags |= kTailPiece;
    e1 = (uint32_t)(u1 - (r1 - 1));
  }
  desc[c] = make_uint4(e0, e1, r0, rows | flags);
}

// page_rank.hpp:133-135 -> the row's L1 change in fixed point
__device__ __forceinline__ unsigned long long item_update(const ItemParams& P, uint32_t i, float z, float xo, float b,
                                                          uint32_t dg) {
  const float xn = __builtin_fmaf(P.damp, z, b);
  P.x[i] = xn;
  P.cout[i] = xn / (float)dg;
  return err_to_fixed((double)fabsf(xn - xo));
}

// position of prefix entry q in LDS: one word skipped every 8, so that a lane's 8 stores and
// the next lane's do not fall on the same banks
__device__ __forceinline__ uint32_t pos(uint32_t q) { return q + (q >> 3); }

// K values per lane: inclusive fixed-point prefix of the edges [e0, e1), entry q of it for edge
// b0 + q (b0 = e0 rounded down to 4; entries before e0 are 0)
template <int NT, int K>
__device__ __forceinline__ void item_prefix(const ItemParams& P, uint32_t b0, uint32_t e0, uint32_t e1,
                                            unsigned long long* pre, unsigned long long* wsum) {
  const uint32_t q0 = threadIdx.x * K;
  uint32_t u[K];
#pragma unroll
  for (int h = 0; h < K; h += 4) {
    const uint32_t p = b0 + q0 + h;
    if ((uint64_t)p + 4 <= P.nnz && p < e1) {  // a whole 16-byte group inside the array
      const u32x4 v = *reinterpret_cast<const u32x4*>(P.col + p);
      u[h] = v.x;
      u[h + 1] = v.y;
      u[h + 2] = v.z;
      u[h + 3] = v.w;
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) u[h + t] = p + t < e1 ? P.col[p + t] : 0u;
    }
  }
  float c[K];
#pragma unroll
  for (int t = 0; t < K; ++t) c[t] = P.cin[u[t]];  // ids outside [e0, e1) are ids too, or 0
  unsigned long long v[K], s = 0;
#pragma unroll
  for (int t = 0; t < K; ++t) {
    const uint32_t p = b0 + q0 + t;
    s += (p >= e0 && p < e1) ? quantize(c[t]) : 0ull;
    v[t] = s;
  }
  unsigned long long inc = wave_inclusive_scan(s);
  unsigned long long off = inc - s;
  if constexpr (NT > 64) {
    if (lane_id() == 63) wsum[threadIdx.x >> 6] = inc;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NT / 64 - 1; ++w) off += (uint32_t)w < (threadIdx.x >> 6) ? wsum[w] : 0ull;
  }
#pragma unroll
  for (int t = 0; t < K; ++t) pre[pos(q0 + t)] = off + v[t];
  __syncthreads();
}

template <int NT>
__global__ __launch_bounds__(NT) void pr_item_kernel(ItemParams P) {
  constexpr uint32_t S = item_span(NT);
  static_assert(kItemLanes == 64, "one lane counter per wavefront lane");
  __shared__ unsigned long long pre[9 * NT];
  __shared__ unsigned long long wsum[NT / 64];
  const uint32_t lane = threadIdx.x & 63u;
  const uint4 d = P.desc[blockIdx.x];
  // the previous sweep's L1 change: loaded now, looked at once the gathers are done (a check
  // first would put its latency in front of theirs)
  unsigned long long ch = 0ull;
  if (P.iter > 0) ch = P.lanes[((P.iter - 1) % 3) * kItemLaneSlot + lane * kItemLanePad];
  const uint32_t e0 = d.x, e1 = d.y, r0 = d.z, rows = d.w & kRowMask;
  // the first round of rows: issued beside the ids
  uint32_t ra = 0, rb = 0, dg = 0;
  float xo = 0.f, bv = P.base;
  if (threadIdx.x < rows) {
    const uint32_t i = r0 + threadIdx.x;
    ra = P.rp[i];
    rb = P.rp[i + 1];
    xo = P.x[i];
    dg = P.deg[i];
    if (P.basev) bv = P.basev[i];
  }
  // lane 0 handles the head piece, lane 1 the tail piece: row h, edges [ha, hb) of the item
  const bool piece = (threadIdx.x == 0 && (d.w & kHeadPiece)) || (threadIdx.x == 1 && (d.w & kTailPiece));
  uint32_t h = 0, hp0 = 0, hp1 = 0;
  if (piece) {
    h = threadIdx.x == 0 ? r0 - 1 : r0 + rows;
    hp0 = P.rp[h];
    hp1 = P.rp[h + 1];
  }
  const uint32_t b0 = e0 & ~3u;
  if (e1 - b0 <= 4u * NT) item_prefix<NT, 4>(P, b0, e0, e1, pre, wsum);
  else item_prefix<NT, 8>(P, b0, e0, e1, pre, wsum);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) ch += __shfl_xor(ch, m, 64);
  if (blockIdx.x == 0) {
    if (threadIdx.x < 64) P.lanes[((P.iter + 1) % 3) * kItemLaneSlot + lane * kItemLanePad] = 0ull;
    if (threadIdx.x == 0 && P.iter > 0) P.acc[P.iter - 1] = ch;
  }
  if (P.iter > 0 && fixed_to_err(ch) < P.threshold) return;
  auto sum = [&](uint32_t a, uint32_t b) -> unsigned long long {  // edges [a, b)
    if (a >= b) return 0ull;
    const unsigned long long hi = pre[pos(b - 1 - b0)];
    return a == b0 ? hi : hi - pre[pos(a - 1 - b0)];
  };
  unsigned long long err = 0ull;
  if (threadIdx.x < rows) err = item_update(P, r0 + threadIdx.x, dequantize(sum(ra, rb)), xo, bv, dg);
  for (uint32_t q = threadIdx.x + NT; q < rows; q += NT) {
    const uint32_t i = r0 + q;
    err += item_update(P, i, dequantize(sum(P.rp[i], P.rp[i + 1])), P.x[i], P.basev ? P.basev[i] : P.base, P.deg[i]);
  }
  if (piece) {
    // the row's pieces are those of the items its edges' units lie in
    const uint32_t a = (uint32_t)(((uint64_t)h + hp0) / S), b = (uint32_t)(((uint64_t)h + hp1 - 1) / S);
    const unsigned long long mine = sum(max(hp0, e0), min(hp1, e1));
    unsigned long long old = __hip_atomic_fetch_add(P.hsum + a, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the sum has been added (its old value is back) before the piece is counted
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(old) : : "memory");
    if (__hip_atomic_fetch_add(P.hcnt + a, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == b - a) {
      // every piece is in: take the sum and leave both counters at 0 for the next sweep
      const unsigned long long z =
          __hip_atomic_exchange(P.hsum + a, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(P.hcnt + a, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      err += item_update(P, h, dequantize(z), P.x[h], P.basev ? P.basev[h] : P.base, P.deg[h]);
    }
  }
  err = wave_sum(err);
  if constexpr (NT > 64) {
    if (lane == 0) wsum[threadIdx.x >> 6] = err;
    __syncthreads();
    err = 0ull;
    for (int w = 0; w < NT / 64; ++w) err += wsum[w];
  }
  if (threadIdx.x == 0 && err)
    atomicAdd(P.lanes + (P.iter % 3) * kItemLaneSlot + (blockIdx.x % kItemLanes) * kItemLanePad, err);
}

__global__ __launch_bounds__(256) void item_init_kernel(ItemParams P, uint32_t count, float init, float* __restrict__ c0,
                                                        uint64_t iters) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < P.n) {
    P.x[i] = init;
    if (c0) c0[i] = init / (float)P.deg[i];
  }
  if (i < count) {
    P.hsum[i] = 0ull;
    P.hcnt[i] = 0u;
  }
  if (i < kItemLaneWords) P.lanes[i] = 0ull;
  if (i < iters) P.acc[i] = 0ull;
}

__global__ __launch_bounds__(64) void item_fold_kernel(const unsigned long long* __restrict__ lanes,
                                                       unsigned long long* __restrict__ acc, uint32_t k) {
  unsigned long long v = lanes[(k % 3) * kItemLaneSlot + threadIdx.x * kItemLanePad];
  v = wave_sum(v);
  if (threadIdx.x == 0) acc[k] = v;
}

}  // namespace

ItemShape item_shape(uint32_t n, uint64_t nnz, uint64_t max_items) {
  const uint64_t units = (uint64_t)n + nnz;
  ItemShape sh;
  sh.threads = units <= (1ull << 18) ? 64u : 256u;
  const uint64_t count = ceil_div(units, item_span(sh.threads));
  if (nnz >= (1ull << 31) || count > max_items) sh.threads = 0;
  else sh.count = (uint32_t)count;
  return sh;
}

void items_build(hipStream_t s, uint32_t n, uint64_t nnz, const uint32_t* rp, const ItemShape& sh, uint4* desc) {
  item_desc_kernel<<<(uint32_t)ceil_div(sh.count, 256), 256, 0, s>>>(n, nnz, rp, item_span(sh.threads), sh.count, desc);
  NWG_LAUNCH_CHECK();
}

void items_enqueue_init(hipStream_t s, const ItemShape& sh, const ItemParams& P, float init, float* c0,
                        uint64_t iters) {
  const uint64_t m = std::max<uint64_t>({P.n, sh.count, kItemLaneWords, iters});
  item_init_kernel<<<(uint32_t)ceil_div(m, 256), 256, 0, s>>>(P, sh.count, init, c0, iters);
  NWG_LAUNCH_CHECK();
}

void items_enqueue_sweep(hipStream_t s, const ItemShape& sh, const ItemParams& P) {
  if (sh.threads == 64) pr_item_kernel<64><<<sh.count, 64, 0, s>>>(P);
  else pr_item_kernel<256><<<sh.count, 256, 0, s>>>(P);
  NWG_LAUNCH_CHECK();
}

void items_enqueue_fold(hipStream_t s, const ItemParams& P, uint32_t k) {
  item_fold_kernel<<<1, 64, 0, s>>>(P.lanes, P.acc, k);
  NWG_LAUNCH_CHECK();
}

}  // namespace nwg
