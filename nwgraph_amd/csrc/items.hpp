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

// Shape for a CSC of n rows and nnz entries; threads is 0 when it takes more than max_items items
// (or 2^31 entries or more).
ItemShape item_shape(uint32_t n, uint64_t nnz, uint64_t max_items);
// desc (count entries) from the row pointers
void items_build(hipStream_t s, uint32_t n, uint64_t nnz, const uint32_t* rp, const ItemShape& sh, uint4* desc);
// x = init, c0 (nullable) = init / outdeg, and the solve's counters cleared: acc[0 .. iters), the lanes,
// hsum and hcnt (count each)
void items_enqueue_init(hipStream_t s, const ItemShape& sh, const ItemParams& P, float init, float* c0,
                        uint64_t iters);
void items_enqueue_sweep(hipStream_t s, const ItemShape& sh, const ItemParams& P);
// acc[k] of sweep k, the last one launched (the others' are stored by the sweep after them)
void items_enqueue_fold(hipStream_t s, const ItemParams& P, uint32_t k);

}  // namespace nwg
