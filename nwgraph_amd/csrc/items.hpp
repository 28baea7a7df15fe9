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
  uint32_t count;            // items
  unsigned long long* hsum;  // per item: fixed-point sum of the long row that starts in it
  uint32_t* hcnt;            // per item: pieces of that row added so far
  unsigned long long* lanes; // kItemLaneWords
  unsigned long long* acc;   // per sweep: L1 change, fixed point
  uint32_t iter;
  double threshold;
  uint32_t longest;          // in-edges of the longest row above an item's span (items_build), or 0
};

// Many graphs in one block-diagonal CSC: every row has its graph's base (ItemParams::basev), and every
// graph its own L1 changes and stopping rule.  ItemParams::acc is iters x ngraphs, and lanes are
// 3 slots (as in ItemParams) of kManyLanes lanes of many_stride(ngraphs) counters: whole 128-byte lines, as
// atomics to one line take some 12 ns each (3 graphs with 9.7 M edges, 20 sweeps: 8 lanes side by side
// 2.22 ms, in lines of their own 0.82; 32 lanes, which every item reads, 1.02).
constexpr uint32_t kManyLanes = 8;
__host__ __device__ constexpr uint32_t many_stride(uint32_t ngraphs) { return (ngraphs + 15u) / 16u * 16u; }
struct ManyParams {
  const uint32_t* row_graph;  // non-decreasing
  uint32_t ngraphs;
  float least_base;           // of ItemParams::basev
};

// Where a segment of weighted sweeps leaves what the host reads: the solve's two words of scales, then
// err[k] at words[2 + k], k in [first, last] of the segment (words null: nowhere).
struct WMail {
  unsigned long long* words = nullptr;
  const unsigned long long* scale = nullptr;
  uint32_t first = 0;
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
  uint32_t folded;        // err[iter - 1] is folded by a launch between the sweeps, else by the sweep
};

// Row sums of a compressed structure over its items, s_u = sum of a value per entry q:
//   gather == null  src[perm[q]]
//   else            (d gather[col[q]]) * src[q]
struct RowSumParams {
  const uint4* desc;
  const uint32_t* rp;
  const uint32_t* idx;  // perm or col; 16-byte aligned
  const float* src;     // 16-byte aligned
  const float* gather;
  float d;
  uint32_t nnz;
  uint32_t count;
  double* head;         // count: an item's piece of the long row begun before it
  double* tail;         // count: and of the one that goes on after it
};
// what becomes of s_u: out[u] = s_u, or with gather
//   ab[u] = {x[u] / norm[u], s_u} and (nullable) gv[u] = omd * gather[u]
struct RowSumOut {
  float* out;
  const float* x;
  const float* norm;
  float2* ab;
  float* gv;
  float omd;
};

// items of a CSC of n rows and nnz entries
uint32_t item_count(uint32_t n, uint64_t nnz);
// their descriptions (item_count of them) from the row pointers; longest (nullable, 0 before): the most
// in-edges of a row above an item's span.  Reads within rp[0 .. n] whatever it holds.
void items_build(hipStream_t s, uint32_t n, uint64_t nnz, const uint32_t* rp, uint4* desc, uint32_t* longest);
// x = init, c0 (nullable) = init / outdeg, and the solve's counters cleared: acc[0 .. iters), the lanes,
// hsum and hcnt (count each)
void items_enqueue_init(hipStream_t s, const ItemParams& P, float init, float* c0, uint64_t iters);
void items_enqueue_sweep(hipStream_t s, const ItemParams& P);
// Many graphs: hsum, hcnt and the lanes cleared; a sweep; acc of sweep k, the last one launched
void items_many_enqueue_init(hipStream_t s, const ItemParams& P, const ManyParams& M);
void items_many_enqueue_sweep(hipStream_t s, const ItemParams& P, const ManyParams& M);
void items_many_enqueue_fold(hipStream_t s, const ItemParams& P, const ManyParams& M, uint32_t k);
// Weighted: xin[0] = src (null: v), err[0 .. iters) and the items' counters cleared; a sweep; err[k]
// of sweep k, the last one launched.
void witems_enqueue_init(hipStream_t s, const WItemParams& P, const float* src, float v, float* dst, uint64_t iters);
void witems_enqueue_sweep(hipStream_t s, const WItemParams& P);
void witems_enqueue_fold(hipStream_t s, const WItemParams& P, uint32_t k, const WMail& mail);
void row_sums_enqueue(hipStream_t s, const RowSumParams& P, const RowSumOut& o);
// acc[k] of sweep k, the last one launched (the others' are stored by the sweep after them); with mail,
// acc[first .. k] there too
void items_enqueue_fold(hipStream_t s, const ItemParams& P, uint32_t first, uint32_t k, unsigned long long* mail);

}  // namespace nwg
