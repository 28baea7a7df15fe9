// items.hpp -- the item sweep (items.hip): one launch per PageRank sweep over edge-balanced
// work items of a CSC.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nwg {

// Lanes the L1 change of a sweep is spread over (one counter per 64 bytes), and the sweeps
// whose lanes are kept: sweep k reads sweep k-1's, adds to its own and clears sweep k+1's.
constexpr uint32_t kItemLanes = 64;
constexpr uint32_t kItemLanePad = 8;
constexpr uint32_t kItemLaneSlot = kItemLanes * kItemLanePad;
constexpr uint32_t kItemLaneWords = 3 * kItemLaneSlot;

// Work items of one CSC: `threads` lanes per item (64 or 256), count items.
struct ItemShape {
  uint32_t threads = 0;
  uint32_t count = 0;
};

struct ItemParams {
  const uint4* desc;         // per item: {first edge, end edge, first row, rows | flags} (items.hip)
  const uint32_t* rp;
  const uint32_t* col;       // 16-byte aligned
  const uint32_t* deg;
  const float* cin;          // contributions gathered
  float* cout;               // contributions written (cin itself for the in-place schedule)
  float* x;
  const float* basev;        // personalised base per row, or null
  float base;
  float damp;
  uint32_t n;
  uint32_t nnz;
  unsigned long long* hsum;  // per item: fixed-point sum of the long row that starts in it
  uint32_t* hcnt;            // per item: pieces of that row added so far
  unsigned long long* lanes; // kItemLaneWords
  unsigned long long* acc;   // per sweep: L1 change, fixed point
  uint32_t iter;
  double threshold;
};

// The weighted sweep over items: x' = fma(d, sum w * xin, basev), products scaled by 2^(*qshift) and
// summed in signed fixed point (fixed_point.hpp).
struct WItemParams {
  const uint4* desc;
  const uint32_t* rp;
  const uint32_t* col;    // 16-byte aligned
  const float* w;         // 16-byte aligned, in the order of col
  const float* basev;
  const float* xin;
  float* xout;
  float damp;
  uint32_t n;
  uint32_t nnz;
  uint32_t count;
  const int* qshift;
  unsigned long long* hsum;
  uint32_t* hcnt;
  double* part;           // 4 * count: per sweep parity, every item's L1 change and its long row's
  double* err;            // per sweep: L1 change
  uint32_t iter;
  double threshold;
  const double* thr_scale;  // relative threshold: the stop compares with threshold * *thr_scale
};

// Row sums of a compressed structure over its items, s_u = sum of a value per entry q:
//   gather == null  src[perm[q]]
//   else            gather[col[q]] * src[q], d times
struct RowSumParams {
  const uint4* desc;
  const uint32_t* rp;
  const uint32_t* idx;  // perm or col; 16-byte aligned
  const float* src;     // 16-byte aligned
  const float* gather;
  uint32_t n;
  uint32_t nnz;
  uint32_t count;
  double* head;         // count: an item's piece of the long row begun before it
  double* tail;         // count: and of the one that goes on after it
};
// what becomes of s_u: out[u] = s_u, or with gather
//   ab[u] = {x[u] / norm[u], x[u] * d * s_u / norm[u]} and (nullable) gv[u] = omd * gather[u]
struct RowSumOut {
  float* out;
  const float* x;
  const float* norm;
  float2* ab;
  float* gv;
  float d, omd;
};

// Shape for a CSC of n rows and nnz entries; threads is 0 when it takes more than max_items items
// (or 2^32 entries or more).
ItemShape item_shape(uint32_t n, uint64_t nnz, uint64_t max_items);
// desc (count entries) from the row pointers
// The same with 256-lane items whatever the size.
ItemShape item_shape_wide(uint32_t n, uint64_t nnz, uint64_t max_items);
void items_build(hipStream_t s, uint32_t n, uint64_t nnz, const uint32_t* rp, const ItemShape& sh, uint4* desc);
// x = init, c0 (nullable) = init / outdeg, and the solve's counters cleared: acc[0 .. iters), the lanes,
// hsum and hcnt (count each)
void items_enqueue_init(hipStream_t s, const ItemShape& sh, const ItemParams& P, float init, float* c0,
                        uint64_t iters);
void items_enqueue_sweep(hipStream_t s, const ItemShape& sh, const ItemParams& P);
// Weighted: xin[0] = src (null: v), err[0 .. iters) and the items' counters cleared; a sweep; err[k]
// of sweep k, the last one launched.
void witems_enqueue_init(hipStream_t s, const WItemParams& P, const float* src, float v, float* dst, uint64_t iters);
void witems_enqueue_sweep(hipStream_t s, const WItemParams& P);
void witems_enqueue_fold(hipStream_t s, const WItemParams& P, uint32_t k);
void row_sums_enqueue(hipStream_t s, const RowSumParams& P, const RowSumOut& o);
// acc[k] of sweep k, the last one launched (the others' are stored by the sweep after them)
void items_enqueue_fold(hipStream_t s, const ItemParams& P, uint32_t k);

}  // namespace nwg
