// items.hip -- PageRank sweep over edge-balanced work items, one launch per sweep.
//
// The sweep is the reference's (include/nwgraph/algorithms/page_rank.hpp:121-147, Jacobi form
// experimental/algorithms/page_rank.hpp:397-430).  It is the pull sweep of every size, and made for graphs
// whose contributions stay in L2, where a sweep is bound by launches, by load latency and by its longest
// rows, not by bytes: row classes with a launch each take up to seven launches per sweep, and one wave
// on a row of thousands of in-edges outlasts everything else.
//
// Row i starts at unit D(i) = i + rp[i] of n + nnz units (one per edge, one per row), and item c
// owns the units [c S, (c + 1) S), S = kSpan = 1020:
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
// depends on no order (fixed_point.hpp).  Where cut-off bits could show (scores far below the others:
// long personalised solves, damping 1), a row is added up once more in double from its gathers.  The form
// that looks for them takes 1 to 3 % longer (20 sweeps, RMAT-12 101.3 / 102.9 us, RMAT-16 @@ / 168.2), so it runs
// where the base does not rule them out.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_utils.hpp"
#include "fixed_point.hpp"
#include "items.hpp"
#include "nwg_internal.hpp"

namespace nwg {

namespace {

// Lanes of an item.  Measured on MI355X, us per sweep with 128 / 256 / 512 / 1024 lanes: RMAT-12
// 6.0 / 5.4 / 5.7 / 7.2, RMAT-16 8.9 / 8.8 / 9.5 / 9.7, RMAT-18 21.8 / 21.3 / 21.6 / 30.6; with 64 RMAT-12
// took 6.1: its span of 252 units cuts more rows into pieces, whose sums meet in atomics.
constexpr uint32_t kNT = 256;

constexpr uint32_t kHeadPiece = 1u << 30;  // the item's first edges belong to a long row begun before it
constexpr uint32_t kTailPiece = 1u << 31;  // its last edges to a long row that goes on after it
constexpr uint32_t kRowMask = kHeadPiece - 1;
constexpr uint32_t kCutRow = 1u << 31;     // in a long row's count of pieces: some value was cut

// units per item; an item stages at most 2 kSpan - 2 edges, and 3 before them for alignment, in
// the 8 kNT places it has
constexpr uint32_t kSpan = 4u * kNT - 4u;

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
__global__ __launch_bounds__(256) void item_desc_kernel(uint32_t n, const uint32_t* __restrict__ rp,
                                                        uint32_t count, uint4* __restrict__ desc,
                                                        uint32_t* __restrict__ longest) {
  const uint32_t c = blockIdx.x * 256 + threadIdx.x;
  if (c >= count) return;
  const uint64_t u0 = (uint64_t)c * kSpan, u1 = u0 + kSpan;
  const uint32_t r0 = first_row_from(rp, n, u0), r1 = first_row_from(rp, n, u1);
  const uint32_t p0 = rp[r0], p1 = rp[r1];
  uint32_t e0 = p0, e1 = p1, rows = r1 - r0, flags = 0;
  // row r0 - 1: a long one whose last edge (unit r0 - 1 + p0 - 1) is not before the window
  if (r0 > 0 && p0 - rp[r0 - 1] > kSpan && (uint64_t)(r0 - 1) + p0 > u0) {
    flags |= kHeadPiece;
    e0 = (uint32_t)(u0 - (r0 - 1));
    if (!rows) e1 = (uint32_t)min((uint64_t)p0, u1 - (r0 - 1));  // no row starts here: it may go on after the window
  }
  if (rows && p1 - rp[r1 - 1] > kSpan) {  // the last row that starts here is a long one
    --rows;
    flags |= kTailPiece;
    e1 = (uint32_t)(u1 - (r1 - 1));
    if (longest) atomicMax(longest, p1 - rp[r1 - 1]);
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

// ids of the K entries p0 .. p0 + K of a lane (p0 a multiple of 4): 16-byte loads where whole
// groups lie in the array, 0 for entries from e1 on
template <int K>
__device__ __forceinline__ void item_ids(const uint32_t* __restrict__ ids, uint32_t nnz, uint32_t p0, uint32_t e1,
                                         uint32_t (&u)[K]) {
#pragma unroll
  for (int h = 0; h < K; h += 4) {
    const uint32_t p = p0 + h;
    if ((uint64_t)p + 4 <= nnz && p < e1) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(ids + p);
      u[h] = v.x;
      u[h + 1] = v.y;
      u[h + 2] = v.z;
      u[h + 3] = v.w;
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) u[h + t] = p + t < e1 ? ids[p + t] : 0u;
    }
  }
}

// K values per lane: inclusive fixed-point prefix of the edges [e0, e1), entry q of it for edge
// b0 + q (b0 = e0 rounded down to 4; entries before e0 are 0).  w null: value cin[id]; else
// w * cin[id] scaled by 2^qs.  kLook: cuts, per wave, whether some value lost bits.
template <int K, bool W, bool kLook>
__device__ __forceinline__ void item_prefix(const uint32_t* __restrict__ col, const float* w, int qs,
                                            const float* cin, uint32_t nnz, uint32_t b0, uint32_t e0, uint32_t e1,
                                            unsigned long long* pre, unsigned long long* wsum, uint32_t* cuts) {
  const uint32_t q0 = threadIdx.x * K;
  uint32_t u[K];
  item_ids<K>(col, nnz, b0 + q0, e1, u);
  uint32_t wt[W ? K : 1];
  if constexpr (W) item_ids<K>(reinterpret_cast<const uint32_t*>(w), nnz, b0 + q0, e1, wt);
  float c[K];
#pragma unroll
  for (int t = 0; t < K; ++t) c[t] = cin[u[t]];  // ids outside [e0, e1) are ids too, or 0
  unsigned long long v[K], s = 0;
  CutNote cut;  // entries outside [e0, e1) too: noting one that cuts costs time only
#pragma unroll
  for (int t = 0; t < K; ++t) {
    const uint32_t p = b0 + q0 + t;
    unsigned long long q;
    if constexpr (W) {
      const float f = __uint_as_float(wt[t]) * c[t];
      q = quantize_signed(f, qs);
      if constexpr (kLook) cut.note(f);
    } else {
      q = quantize(c[t]);
      if constexpr (kLook) cut.note(c[t]);
    }
    s += (p >= e0 && p < e1) ? q : 0ull;
    v[t] = s;
  }
  uint64_t any_cut = 0;
  if constexpr (kLook) any_cut = __ballot(cut.cuts(qs));
  unsigned long long inc = wave_inclusive_scan(s);
  unsigned long long off = inc - s;
  if (lane_id() == 63) {
    wsum[threadIdx.x >> 6] = inc;
    if constexpr (kLook) cuts[threadIdx.x >> 6] = any_cut != 0;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t w2 = 0; w2 < kNT / 64 - 1; ++w2) off += w2 < (threadIdx.x >> 6) ? wsum[w2] : 0ull;
#pragma unroll
  for (int t = 0; t < K; ++t) pre[pos(q0 + t)] = off + v[t];
  __syncthreads();
}

// exact sum of the edges [a, b) of an item
__device__ __forceinline__ unsigned long long item_sum(const unsigned long long* pre, uint32_t b0, uint32_t a,
                                                       uint32_t b) {
  if (a >= b) return 0ull;
  const unsigned long long hi = pre[pos(b - 1 - b0)];
  return a == b0 ? hi : hi - pre[pos(a - 1 - b0)];
}

static_assert(kNT == 256, "cuts of four waves");
__device__ __forceinline__ bool item_cuts(const uint32_t* cuts) { return (cuts[0] | cuts[1] | cuts[2] | cuts[3]) != 0; }

// sum of the entries a, a + step, ... below b of a row, as item_prefix's without the rounding to units
template <bool W>
__device__ __forceinline__ double direct_sum(const uint32_t* __restrict__ col, const float* w, const float* cin,
                                             uint64_t a, uint64_t b, uint32_t step) {
  double s = 0.0;
#pragma unroll 4
  for (uint64_t p = a; p < b; p += step) {
    const double c = (double)cin[col[p]];
    if constexpr (W) s += (double)w[p] * c;
    else s += c;
  }
  return s;
}
// The sums of the long rows whose lanes ask for them (entries [a, b) each), by the whole wave.
template <bool W>
__device__ __forceinline__ void direct_long_sums(const uint32_t* __restrict__ col, const float* w, const float* cin,
                                                 uint32_t a, uint32_t b, bool ask, float* z) {
  for (uint64_t m = __ballot(ask); __builtin_expect(m != 0, 0); m &= m - 1) {
    const int l = __builtin_ctzll(m);
    const uint32_t ra = (uint32_t)__shfl((int)a, l, 64), rb = (uint32_t)__shfl((int)b, l, 64);
    const double s = wave_sum(direct_sum<W>(col, w, cin, (uint64_t)ra + lane_id(), rb, 64));
    if ((int)lane_id() == l) *z = (float)s;
  }
}

// Adds a piece of long row h (entries [hp0, hp1), this piece's sum `mine`) to the row's counter, that
// of the item it starts in; true for the last piece, which gets the row's sum and leaves the
// counters at 0 for the next sweep.  *start: the item the row starts in.  cut: in, whether a value of
// this piece was cut; out, of any piece.
template <bool kLook>
__device__ __forceinline__ bool add_piece(unsigned long long* hsum, uint32_t* hcnt, uint32_t h, uint32_t hp0,
                                          uint32_t hp1, unsigned long long mine, unsigned long long* z,
                                          uint32_t* start, bool& cut) {
  // the row's pieces are those of the items its edges' units lie in
  const uint32_t a = (uint32_t)(((uint64_t)h + hp0) / kSpan), b = (uint32_t)(((uint64_t)h + hp1 - 1) / kSpan);
  *start = a;
  unsigned long long old = __hip_atomic_fetch_add(hsum + a, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // in the word of the count, so before it
  if (kLook && cut) (void)__hip_atomic_fetch_or(hcnt + a, kCutRow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // the sum has been added (its old value is back) before the piece is counted
  asm volatile("s_waitcnt vmcnt(0)" : "+v"(old) : : "memory");
  const uint32_t counted = __hip_atomic_fetch_add(hcnt + a, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if ((counted & ~kCutRow) != b - a) return false;
  cut = kLook && (counted & kCutRow);
  *z = __hip_atomic_exchange(hsum + a, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(hcnt + a, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// the sum of a row's entries [a, b): s in fixed point, or in double where that is too coarse for it
template <bool kLook>
__device__ __forceinline__ float item_row_sum(const ItemParams& P, unsigned long long s, uint32_t a, uint32_t b,
                                              float base, const uint32_t* cuts) {
  const float z = dequantize(s);
  if constexpr (kLook)
    if (__builtin_expect(item_cuts(cuts), 0) && sum_is_coarse(__builtin_fmaf(P.damp, z, base), b - a))
      return (float)direct_sum<false>(P.col, nullptr, P.cin, a, b, 1);
  return z;
}

// kLook: rows may be too small for the fixed point (looks)
template <bool kLook>
__global__ __launch_bounds__(kNT) void pr_item_kernel(ItemParams P) {
  static_assert(kItemLanes == 64 && kNT == 256, "one lane counter per wavefront lane, four waves");
  __shared__ unsigned long long pre[9 * kNT];
  __shared__ unsigned long long wsum[kNT / 64];
  __shared__ uint32_t cuts[kNT / 64];
  const uint32_t lane = threadIdx.x & 63u;
  const uint4 d = P.desc[blockIdx.x];
  // a solve that stopped before the previous sweep gathers nothing more (9 of 20 sweeps, allocation-free:
  // uniform random with 18 M edges 2.55 to 1.48 ms, with 3 M 0.39 to 0.24; resident, 1.9 M 0.23 to 0.14)
  if (P.iter > 1 && fixed_to_err(P.acc[P.iter - 2]) < P.threshold) return;
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
  if (e1 - b0 <= 4u * kNT) item_prefix<4, false, kLook>(P.col, nullptr, 0, P.cin, P.nnz, b0, e0, e1, pre, wsum, cuts);
  else item_prefix<8, false, kLook>(P.col, nullptr, 0, P.cin, P.nnz, b0, e0, e1, pre, wsum, cuts);
  ch = wave_sum(ch);
  if (blockIdx.x == 0) {
    if (threadIdx.x < 64) P.lanes[((P.iter + 1) % 3) * kItemLaneSlot + lane * kItemLanePad] = 0ull;
    if (threadIdx.x == 0 && P.iter > 0) P.acc[P.iter - 1] = ch;
  }
  if (P.iter > 0 && fixed_to_err(ch) < P.threshold) return;
  auto sum = [&](uint32_t a, uint32_t b) { return item_sum(pre, b0, a, b); };
  unsigned long long err = 0ull;
  for (uint32_t q = threadIdx.x; q < rows;) {
    err += item_update(P, r0 + q, item_row_sum<kLook>(P, sum(ra, rb), ra, rb, bv, cuts), xo, bv, dg);
    if ((q += kNT) >= rows) break;
    const uint32_t i = r0 + q;
    ra = P.rp[i];
    rb = P.rp[i + 1];
    xo = P.x[i];
    dg = P.deg[i];
    if (P.basev) bv = P.basev[i];
  }
  float hz = 0.f, hb = 0.f;
  bool last = false, ask = false;
  if (piece) {
    unsigned long long z;
    uint32_t a;
    bool cut = kLook && item_cuts(cuts);
    last = add_piece<kLook>(P.hsum, P.hcnt, h, hp0, hp1, sum(max(hp0, e0), min(hp1, e1)), &z, &a, cut);
    if (last) {
      hz = dequantize(z);
      hb = P.basev ? P.basev[h] : P.base;
      ask = cut && sum_is_coarse(__builtin_fmaf(P.damp, hz, hb), hp1 - hp0);
    }
  }
  if constexpr (kLook) direct_long_sums<false>(P.col, nullptr, P.cin, hp0, hp1, ask, &hz);
  if (last) err += item_update(P, h, hz, P.x[h], hb, P.deg[h]);
  err = wave_sum(err);
  if (lane == 0) wsum[threadIdx.x >> 6] = err;
  __syncthreads();
  err = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
  if (threadIdx.x == 0 && err)
    atomicAdd(P.lanes + (P.iter % 3) * kItemLaneSlot + (blockIdx.x % kItemLanes) * kItemLanePad, err);
}

// ---- many graphs ----
// L1 change of graph g in sweep k
__device__ __forceinline__ unsigned long long many_change(const ItemParams& P, const ManyParams& M, uint32_t k,
                                                          uint32_t g) {
  const uint32_t stride = many_stride(M.ngraphs);
  const unsigned long long* l = P.lanes + (uint64_t)(k % 3) * kManyLanes * stride + g;
  unsigned long long s = 0ull;
#pragma unroll
  for (uint32_t q = 0; q < kManyLanes; ++q) s += l[(uint64_t)q * stride];
  return s;
}

// The sweep over the union of many graphs: items are cut from it as from one graph, so one may hold rows
// of several.  The L1 changes of its first kManyLocal graphs meet in LDS, those of further ones
// (graphs of a few vertices) go to memory row by row.  Measured on MI355X, ms for 20 sweeps here / with
// workgroups of up to 4096 edges that add up a row per lane / binned: 63 graphs of 256 to 1024
// vertices (0.4 M edges) 0.17 / 0.42 / 0.39, 12 of 2^12 to 2^18 (9.5 M) 0.87 / 4.7 / 1.53, 80 of 2^12 to 2^16
// (18.7 M) 1.47 / 4.5 / 1.63.
constexpr uint32_t kManyLocal = 64;
template <bool kLook>
__global__ __launch_bounds__(kNT) void pr_item_many_kernel(ItemParams P, ManyParams M) {
  __shared__ unsigned long long pre[9 * kNT];
  __shared__ unsigned long long wsum[kNT / 64];
  __shared__ uint32_t cuts[kNT / 64];
  __shared__ unsigned long long errs[kManyLocal];
  __shared__ uint32_t done[kManyLocal];
  // the previous sweep's changes, for the host, and the next sweep's lanes
  if (P.iter > 0)
    for (uint32_t q = blockIdx.x * kNT + threadIdx.x; q < M.ngraphs; q += gridDim.x * kNT)
      P.acc[(uint64_t)(P.iter - 1) * M.ngraphs + q] = many_change(P, M, P.iter - 1, q);
  const uint64_t slot = (uint64_t)kManyLanes * many_stride(M.ngraphs);
  for (uint64_t q = blockIdx.x * kNT + threadIdx.x; q < slot; q += gridDim.x * kNT)
    P.lanes[(P.iter + 1) % 3 * slot + q] = 0ull;
  const uint4 d = P.desc[blockIdx.x];
  const uint32_t e0 = d.x, e1 = d.y, r0 = d.z, rows = d.w & kRowMask;
  const bool head = d.w & kHeadPiece, tail = d.w & kTailPiece;
  if (!rows && !head && !tail) return;
  uint32_t ra = 0, rb = 0, dg = 0, rg = 0;
  float xo = 0.f, bv = 0.f;
  if (threadIdx.x < rows) {
    const uint32_t i = r0 + threadIdx.x;
    ra = P.rp[i];
    rb = P.rp[i + 1];
    xo = P.x[i];
    dg = P.deg[i];
    bv = P.basev[i];
    rg = M.row_graph[i];
  }
  const uint32_t g0 = M.row_graph[head ? r0 - 1 : r0], g1 = M.row_graph[tail ? r0 + rows : r0 + rows - 1];
  if (threadIdx.x < kManyLocal) {
    const uint32_t g = g0 + threadIdx.x;
    errs[threadIdx.x] = 0ull;
    done[threadIdx.x] = P.iter > 0 && g <= g1 && fixed_to_err(many_change(P, M, P.iter - 1, g)) < P.threshold;
  }
  const bool piece = (threadIdx.x == 0 && head) || (threadIdx.x == 1 && tail);
  uint32_t h = 0, hp0 = 0, hp1 = 0;
  if (piece) {
    h = threadIdx.x == 0 ? r0 - 1 : r0 + rows;
    hp0 = P.rp[h];
    hp1 = P.rp[h + 1];
  }
  const uint32_t b0 = e0 & ~3u;
  if (e1 - b0 <= 4u * kNT) item_prefix<4, false, kLook>(P.col, nullptr, 0, P.cin, P.nnz, b0, e0, e1, pre, wsum, cuts);
  else item_prefix<8, false, kLook>(P.col, nullptr, 0, P.cin, P.nnz, b0, e0, e1, pre, wsum, cuts);
  if (g0 == g1 && done[0]) return;
  unsigned long long* const lane =
      P.lanes + P.iter % 3 * slot + (uint64_t)(blockIdx.x % kManyLanes) * many_stride(M.ngraphs);
  auto sum = [&](uint32_t a, uint32_t b) { return item_sum(pre, b0, a, b); };
  auto solved = [&](uint32_t g) {
    return g - g0 < kManyLocal ? done[g - g0] != 0
                               : P.iter > 0 && fixed_to_err(many_change(P, M, P.iter - 1, g)) < P.threshold;
  };
  unsigned long long err = 0ull;  // with one graph only
  auto add = [&](uint32_t g, unsigned long long e) {
    if (g0 == g1) err += e;
    else if (!e) return;
    else if (g - g0 < kManyLocal) atomicAdd(&errs[g - g0], e);
    else atomicAdd(lane + g, e);
  };
  for (uint32_t q = threadIdx.x; q < rows;) {
    if (!solved(rg)) add(rg, item_update(P, r0 + q, item_row_sum<kLook>(P, sum(ra, rb), ra, rb, bv, cuts), xo, bv, dg));
    if ((q += kNT) >= rows) break;
    const uint32_t i = r0 + q;
    ra = P.rp[i];
    rb = P.rp[i + 1];
    xo = P.x[i];
    dg = P.deg[i];
    bv = P.basev[i];
    rg = M.row_graph[i];
  }
  float hz = 0.f, hb = 0.f;
  bool last = false, ask = false;
  uint32_t hg = 0;
  if (piece) {
    // all pieces of a row see the same change, so they are all added or none is
    hg = M.row_graph[h];
    unsigned long long z;
    uint32_t a;
    bool cut = kLook && item_cuts(cuts);
    last = !solved(hg) && add_piece<kLook>(P.hsum, P.hcnt, h, hp0, hp1, sum(max(hp0, e0), min(hp1, e1)), &z, &a, cut);
    if (last) {
      hz = dequantize(z);
      hb = P.basev[h];
      ask = cut && sum_is_coarse(__builtin_fmaf(P.damp, hz, hb), hp1 - hp0);
    }
  }
  if constexpr (kLook) direct_long_sums<false>(P.col, nullptr, P.cin, hp0, hp1, ask, &hz);
  if (last) add(hg, item_update(P, h, hz, P.x[h], hb, P.deg[h]));
  if (g0 == g1) {
    err = wave_sum(err);
    if (lane_id() == 0) wsum[threadIdx.x >> 6] = err;
    __syncthreads();
    err = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
    if (threadIdx.x == 0 && err) atomicAdd(lane + g0, err);
  } else {
    __syncthreads();
    if (threadIdx.x < kManyLocal && errs[threadIdx.x]) atomicAdd(lane + g0 + threadIdx.x, errs[threadIdx.x]);
  }
}

__global__ __launch_bounds__(256) void item_many_init_kernel(ItemParams P, ManyParams M) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < P.count) {
    P.hsum[i] = 0ull;
    P.hcnt[i] = 0u;
  }
  if (i < 3ull * kManyLanes * many_stride(M.ngraphs)) P.lanes[i] = 0ull;
}

__global__ __launch_bounds__(256) void item_many_fold_kernel(ItemParams P, ManyParams M, uint32_t k) {
  const uint32_t g = blockIdx.x * 256 + threadIdx.x;
  if (g < M.ngraphs) P.acc[(uint64_t)k * M.ngraphs + g] = many_change(P, M, k, g);
}

// ---- weighted ----
// The L1 changes of a weighted sweep have no bound (fixed_point.hpp's scale covers row sums), so
// they stay doubles: every item stores its own and, where a long row starts in it, that row's; every
// workgroup of the next sweep adds them all in one fixed order and stops or goes on, which takes
// the place of a launch that folds them (with more items than that is worth, the launch does).

__device__ __forceinline__ double witem_stop(const WItemParams& P) {
  return P.thr_scale ? P.threshold * *P.thr_scale : P.threshold;
}

// L1 change of sweep k from its items' parts; the whole workgroup, result in every lane
__device__ __forceinline__ double witem_change(const WItemParams& P, uint32_t k, double* red) {
  const double* part = P.part + (uint64_t)(k & 1u) * 2 * P.count;
  double e = 0.0;
  for (uint32_t q = threadIdx.x; q < 2 * P.count; q += kNT) e += part[q];
  e = wave_sum(e);
  if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = e;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ __launch_bounds__(kNT) void wpr_item_kernel(WItemParams P) {
  __shared__ unsigned long long pre[9 * kNT];
  __shared__ unsigned long long wsum[kNT / 64];
  __shared__ uint32_t cuts[kNT / 64];
  __shared__ double red[kNT / 64], red2[kNT / 64];
  const double stop = witem_stop(P);
  // a solve that stopped before the previous sweep: that sweep stored no parts
  if (P.folded ? P.iter > 0 && P.err[P.iter - 1] < stop : P.iter > 1 && P.err[P.iter - 2] < stop) return;
  const uint4 d = P.desc[blockIdx.x];
  const uint32_t e0 = d.x, e1 = d.y, r0 = d.z, rows = d.w & kRowMask;
  const int qs = *P.qshift;
  uint32_t ra = 0, rb = 0;
  float xo = 0.f, bv = 0.f;
  if (threadIdx.x < rows) {
    const uint32_t i = r0 + threadIdx.x;
    ra = P.rp[i];
    rb = P.rp[i + 1];
    xo = P.xin[i];
    bv = P.basev[i];
  }
  const bool piece = (threadIdx.x == 0 && (d.w & kHeadPiece)) || (threadIdx.x == 1 && (d.w & kTailPiece));
  uint32_t h = 0, hp0 = 0, hp1 = 0;
  if (piece) {
    h = threadIdx.x == 0 ? r0 - 1 : r0 + rows;
    hp0 = P.rp[h];
    hp1 = P.rp[h + 1];
  }
  const uint32_t b0 = e0 & ~3u;
  if (e1 - b0 <= 4u * kNT) item_prefix<4, true, true>(P.col, P.w, qs, P.xin, P.nnz, b0, e0, e1, pre, wsum, cuts);
  else item_prefix<8, true, true>(P.col, P.w, qs, P.xin, P.nnz, b0, e0, e1, pre, wsum, cuts);
  if (P.iter > 0 && !P.folded) {
    const double ch = witem_change(P, P.iter - 1, red);
    if (blockIdx.x == 0 && threadIdx.x == 0) P.err[P.iter - 1] = ch;
    if (ch < stop) return;
  }
  auto coarse = [&](float z, float b, uint32_t m) { return sum_is_coarse(__builtin_fmaf(P.damp, z, b), m, qs); };
  auto update = [&](uint32_t i, float z, float old, float b) -> double {
    const float xn = __builtin_fmaf(P.damp, z, b);
    P.xout[i] = xn;
    return (double)fabsf(xn - old);
  };
  auto row_sum = [&](uint32_t a, uint32_t b, float base) -> float {
    const float z = dequantize_signed(item_sum(pre, b0, a, b), qs);
    if (__builtin_expect(item_cuts(cuts), 0) && coarse(z, base, b - a)) return (float)direct_sum<true>(P.col, P.w, P.xin, a, b, 1);
    return z;
  };
  double e = 0.0;
  for (uint32_t q = threadIdx.x; q < rows;) {
    e += update(r0 + q, row_sum(ra, rb, bv), xo, bv);
    if ((q += kNT) >= rows) break;
    const uint32_t i = r0 + q;
    ra = P.rp[i];
    rb = P.rp[i + 1];
    xo = P.xin[i];
    bv = P.basev[i];
  }
  double* part = P.part + (uint64_t)(P.iter & 1u) * 2 * P.count;
  float hz = 0.f, hb = 0.f;
  uint32_t ha = 0;
  bool last = false, ask = false;
  if (piece) {
    unsigned long long z;
    bool cut = item_cuts(cuts);
    last = add_piece<true>(P.hsum, P.hcnt, h, hp0, hp1, item_sum(pre, b0, max(hp0, e0), min(hp1, e1)), &z, &ha, cut);
    if (last) {
      hz = dequantize_signed(z, qs);
      hb = P.basev[h];
      ask = cut && coarse(hz, hb, hp1 - hp0);
    }
  }
  direct_long_sums<true>(P.col, P.w, P.xin, hp0, hp1, ask, &hz);
  if (last) part[P.count + ha] = update(h, hz, P.xin[h], hb);
  e = wave_sum(e);
  if ((threadIdx.x & 63u) == 0) red2[threadIdx.x >> 6] = e;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (red2[0] + red2[1]) + (red2[2] + red2[3]);
}

__global__ __launch_bounds__(256) void witem_init_kernel(WItemParams P, const float* __restrict__ src, float v,
                                                         float* __restrict__ dst, uint64_t iters) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < P.n) dst[i] = src ? src[i] : v;
  if (i < P.count) {
    P.hsum[i] = 0ull;
    P.hcnt[i] = 0u;
  }
  if (i < 4ull * P.count) P.part[i] = 0.0;
  if (i < iters) P.err[i] = 0.0;
}

__global__ __launch_bounds__(kNT) void witem_fold_kernel(WItemParams P, uint32_t k, WMail mail) {
  __shared__ double red[kNT / 64];
  double ch = 0.0;
  if (k == 0 || !(P.err[k - 1] < witem_stop(P))) {  // else sweep k did nothing
    ch = witem_change(P, k, red);
    if (threadIdx.x == 0) P.err[k] = ch;
  }
  wmail_post(mail, P.err, k, ch);
}

// ---- row sums ----
// Sums in double, with no value of one row ever added to another's (signed values of any magnitude: a
// running prefix would cancel): lane t adds its 4 or 8 consecutive values up to the row starts
// among them, and a segmented scan over the lanes carries what is open.
__device__ __forceinline__ void seg_scan_step(double& v, uint32_t& f, double pv, uint32_t pf) {
  if (!f) v += pv;
  f |= pf;
}

template <int K>
__device__ __forceinline__ void item_row_sums(const RowSumParams& P, uint32_t b0, uint32_t e0, uint32_t e1,
                                              const uint8_t* start, double* pre, double* wv, uint32_t* wf) {
  const uint32_t q0 = threadIdx.x * K;
  uint32_t u[K];
  item_ids<K>(P.idx, P.nnz, b0 + q0, e1, u);
  double val[K];
  if (P.gather) {
    uint32_t wt[K];
    item_ids<K>(reinterpret_cast<const uint32_t*>(P.src), P.nnz, b0 + q0, e1, wt);
#pragma unroll
    for (int t = 0; t < K; ++t) val[t] = (double)(P.d * P.gather[u[t]]) * (double)__uint_as_float(wt[t]);
  } else {
#pragma unroll
    for (int t = 0; t < K; ++t) val[t] = (double)P.src[u[t]];
  }
  double run = 0.0;
  uint32_t open = 0;  // a row starts in the lane's values
#pragma unroll
  for (int t = 0; t < K; ++t) {
    const uint32_t p = b0 + q0 + t;
    const bool in = p >= e0 && p < e1;
    if (in && start[q0 + t]) {
      run = 0.0;
      open = 1u;
    }
    run += in ? val[t] : 0.0;
    val[t] = run;
  }
  // inclusive segmented scan of (run, open) over the wave, then the waves
  double v = run;
  uint32_t f = open;
  const uint32_t lane = lane_id(), w = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double pv = __shfl_up(v, o, 64);
    const uint32_t pf = (uint32_t)__shfl_up((int)f, o, 64);
    if (lane >= (uint32_t)o) seg_scan_step(v, f, pv, pf);
  }
  if (lane == 63) {
    wv[w] = v;
    wf[w] = f;
  }
  double cv = __shfl_up(v, 1, 64);
  uint32_t cf = (uint32_t)__shfl_up((int)f, 1, 64);
  if (lane == 0) {
    cv = 0.0;
    cf = 0u;
  }
  __syncthreads();
  double ov = 0.0;  // open sum before this wave
  for (uint32_t q = 0; q < w; ++q) ov = wf[q] ? wv[q] : ov + wv[q];
  const double carry = cf ? cv : ov + cv;  // open sum before this lane
  bool fresh = false;
#pragma unroll
  for (int t = 0; t < K; ++t) {
    const uint32_t p = b0 + q0 + t;
    fresh |= p >= e0 && p < e1 && start[q0 + t];
    pre[pos(q0 + t)] = fresh ? val[t] : carry + val[t];
  }
  __syncthreads();
}

__device__ __forceinline__ void row_sum_out(const RowSumParams& P, const RowSumOut& o, uint32_t u, double s) {
  if (!P.gather) {
    const float f = (float)s;
    o.out[u] = __builtin_isinf(f) ? __builtin_nanf("") : f;  // past the floats: the weights it divides would be 0
    return;
  }
  // a source without out-edges has no edge that reads its pair; a quotient past the floats stays finite, as
  // a source of one edge multiplies it by 0
  float a = o.x[u] / o.norm[u];
  if (__builtin_isinf(a) && o.norm[u] != 0.f && !__builtin_isinf(o.x[u])) a = __builtin_copysignf(3.402823466e38f, a);
  o.ab[u] = make_float2(a, (float)s);
  if (o.gv) o.gv[u] = o.omd * P.gather[u];
}

__global__ __launch_bounds__(kNT) void row_sum_kernel(RowSumParams P, RowSumOut o) {
  __shared__ double pre[9 * kNT];
  __shared__ uint8_t start[8 * kNT];
  __shared__ double wv[kNT / 64];
  __shared__ uint32_t wf[kNT / 64];
  const uint4 d = P.desc[blockIdx.x];
  const uint32_t e0 = d.x, e1 = d.y, r0 = d.z, rows = d.w & kRowMask, b0 = e0 & ~3u;
  for (uint32_t q = threadIdx.x; q < 2 * kNT; q += kNT) reinterpret_cast<uint32_t*>(start)[q] = 0u;
  __syncthreads();
  // rows with entries mark their first; the tail piece's row too (r0 + rows)
  const uint32_t marks = rows + ((d.w & kTailPiece) ? 1u : 0u);
  for (uint32_t q = threadIdx.x; q < marks; q += kNT) {
    const uint32_t a = P.rp[r0 + q];
    if (P.rp[r0 + q + 1] > a) start[a - b0] = 1;
  }
  __syncthreads();
  if (e1 - b0 <= 4u * kNT) item_row_sums<4>(P, b0, e0, e1, start, pre, wv, wf);
  else item_row_sums<8>(P, b0, e0, e1, start, pre, wv, wf);
  for (uint32_t q = threadIdx.x; q < rows; q += kNT) {
    const uint32_t a = P.rp[r0 + q], b = P.rp[r0 + q + 1];
    row_sum_out(P, o, r0 + q, b > a ? pre[pos(b - 1 - b0)] : 0.0);
  }
  if (threadIdx.x == 0 && (d.w & kHeadPiece)) {
    const uint32_t end = rows || (d.w & kTailPiece) ? P.rp[r0] : e1;
    P.head[blockIdx.x] = pre[pos(end - 1 - b0)];
  }
  if (threadIdx.x == 1 && (d.w & kTailPiece)) P.tail[blockIdx.x] = pre[pos(e1 - 1 - b0)];
}

// One wave per item: the long row that starts in it, if any, from its pieces (lane-strided, then a
// fixed tree).
__global__ __launch_bounds__(256) void row_sum_long_kernel(RowSumParams P, RowSumOut o) {
  const uint32_t a = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
  if (a >= P.count) return;
  const uint4 d = P.desc[a];
  if (!(d.w & kTailPiece)) return;
  const uint32_t h = d.z + (d.w & kRowMask);
  const uint32_t b = (uint32_t)(((uint64_t)h + P.rp[h + 1] - 1) / kSpan);
  double s = lane == 0 ? P.tail[a] : 0.0;
  for (uint32_t c = a + 1 + lane; c <= b; c += 64) s += P.head[c];
  s = wave_sum(s);
  if (lane == 0) row_sum_out(P, o, h, s);
}

__global__ __launch_bounds__(256) void item_init_kernel(ItemParams P, float init, float* __restrict__ c0,
                                                        uint64_t iters) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < P.n) {
    P.x[i] = init;
    if (c0) c0[i] = init / (float)P.deg[i];
  }
  if (i < P.count) {
    P.hsum[i] = 0ull;
    P.hcnt[i] = 0u;
  }
  if (i < kItemLaneWords) P.lanes[i] = 0ull;
  if (i < iters) P.acc[i] = 0ull;
}

__global__ __launch_bounds__(64) void item_fold_kernel(const unsigned long long* __restrict__ lanes,
                                                       unsigned long long* __restrict__ acc, uint32_t first,
                                                       uint32_t k, double threshold,
                                                       unsigned long long* __restrict__ mail) {
  unsigned long long v = lanes[(k % 3) * kItemLaneSlot + threadIdx.x * kItemLanePad];
  v = wave_sum(v);
  if (k > 0 && fixed_to_err(acc[k - 1]) < threshold) v = 0ull;  // sweep k did nothing, its lanes are older
  if (threadIdx.x == 0) acc[k] = v;
  if (!mail) return;
  for (uint32_t q = first + threadIdx.x; q < k; q += 64) mail[q] = acc[q];
  if (threadIdx.x == 0) mail[k] = v;
}

}  // namespace

uint32_t item_count(uint32_t n, uint64_t nnz) {
  return (uint32_t)ceil_div((uint64_t)n + nnz, kSpan);
}

void witems_enqueue_init(hipStream_t s, const WItemParams& P, const float* src, float v, float* dst, uint64_t iters) {
  const uint64_t m = std::max<uint64_t>({P.n, 4ull * P.count, iters});
  witem_init_kernel<<<(uint32_t)ceil_div(m, 256), 256, 0, s>>>(P, src, v, dst, iters);
  NWG_LAUNCH_CHECK();
}

void witems_enqueue_sweep(hipStream_t s, const WItemParams& P) {
  wpr_item_kernel<<<P.count, kNT, 0, s>>>(P);
  NWG_LAUNCH_CHECK();
}

void witems_enqueue_fold(hipStream_t s, const WItemParams& P, uint32_t k, const WMail& mail) {
  witem_fold_kernel<<<1, kNT, 0, s>>>(P, k, mail);
  NWG_LAUNCH_CHECK();
}

void row_sums_enqueue(hipStream_t s, const RowSumParams& P, const RowSumOut& o) {
  if (!P.count) return;
  row_sum_kernel<<<P.count, kNT, 0, s>>>(P, o);
  row_sum_long_kernel<<<(P.count + 3) / 4, 256, 0, s>>>(P, o);
  NWG_LAUNCH_CHECK();
}

void items_build(hipStream_t s, uint32_t n, uint64_t nnz, const uint32_t* rp, uint4* desc, uint32_t* longest) {
  const uint32_t count = item_count(n, nnz);
  item_desc_kernel<<<(uint32_t)ceil_div(count, 256), 256, 0, s>>>(n, rp, count, desc, longest);
  NWG_LAUNCH_CHECK();
}

void items_enqueue_init(hipStream_t s, const ItemParams& P, float init, float* c0, uint64_t iters) {
  const uint64_t m = std::max<uint64_t>({P.n, P.count, kItemLaneWords, iters});
  item_init_kernel<<<(uint32_t)ceil_div(m, 256), 256, 0, s>>>(P, init, c0, iters);
  NWG_LAUNCH_CHECK();
}

// A row's result is at least its base, and no row of m entries is too small for the fixed point where that is
// m * 2^-34 or more (sum_is_coarse): with the uniform teleport at damping 0.85, rows of an item's span in
// graphs of up to 2.5 M vertices, rows of 65,536 in graphs of 39,000.
static bool looks(float base, uint32_t longest) { return !(base >= (float)std::max(kSpan, longest) * 0x1p-34f); }

void items_enqueue_sweep(hipStream_t s, const ItemParams& P) {
  if (P.basev || looks(P.base, P.longest)) pr_item_kernel<true><<<P.count, kNT, 0, s>>>(P);
  else pr_item_kernel<false><<<P.count, kNT, 0, s>>>(P);
  NWG_LAUNCH_CHECK();
}

void items_many_enqueue_init(hipStream_t s, const ItemParams& P, const ManyParams& M) {
  const uint64_t m = std::max<uint64_t>(P.count, 3ull * kManyLanes * many_stride(M.ngraphs));
  item_many_init_kernel<<<(uint32_t)ceil_div(m, 256), 256, 0, s>>>(P, M);
  NWG_LAUNCH_CHECK();
}

void items_many_enqueue_sweep(hipStream_t s, const ItemParams& P, const ManyParams& M) {
  if (looks(M.least_base, P.longest)) pr_item_many_kernel<true><<<P.count, kNT, 0, s>>>(P, M);
  else pr_item_many_kernel<false><<<P.count, kNT, 0, s>>>(P, M);
  NWG_LAUNCH_CHECK();
}

void items_many_enqueue_fold(hipStream_t s, const ItemParams& P, const ManyParams& M, uint32_t k) {
  item_many_fold_kernel<<<(uint32_t)ceil_div(M.ngraphs, 256), 256, 0, s>>>(P, M, k);
  NWG_LAUNCH_CHECK();
}

void items_enqueue_fold(hipStream_t s, const ItemParams& P, uint32_t first, uint32_t k, unsigned long long* mail) {
  item_fold_kernel<<<1, 64, 0, s>>>(P.lanes, P.acc, first, k, P.threshold, mail);
  NWG_LAUNCH_CHECK();
}

}  // namespace nwg
