// build.hip -- on-device edge list -> CSC / CSR construction.
//
// Pipeline (reference semantics in brackets, pnnl/NWGraph):
//   1. the first pass of the sort reads the edges, packs key = (row << b) | entry, b =
//      bits(n-1), and with clean=1 drops u == v [remove_self_loops, build.hpp:404-410] --
//      dropping before the sort gives the same edge set as the reference's sort -> uniq ->
//      remove order (tc.cpp:66-68)
//   2. stable LSD radix sort of the 2b-bit keys [lexical_sort_by, build.hpp:57-70]
//   3. row pointers from the sorted keys and entries = low bits
//      [fill_directed<idx> + sort_to_be_indexed, build.hpp:209-232,
//       compressed.hpp:491-502: each row ascending makes the layout unique]; with clean=1 of
//      equal keys only the first [uniq, build.hpp:392-402]
//   4. out-degree = histogram of sources [build_degrees, bench/gapbs/common.hpp:110-121]
#include <algorithm>

#include "device_utils.hpp"
#include "nwg_internal.hpp"

namespace nwg {

namespace {

inline int bits_for(uint32_t n) {
  int b = 1;
  while (b < 32 && (1ull << b) < (uint64_t)n) ++b;
  return b;
}

// Sorted keys (row << b | entry) -> row pointers and entries, in tiles of kCsxTile keys; with
// uniq, equal neighbours count once [uniq, build.hpp:392-402].  A wave takes kCsxItems x 64
// consecutive keys, 64 at a time.  One pass counts a tile's distinct keys, a scan places the
// tiles, the second pass writes: 20 bytes moved per key (flags, their scan, a compacted copy and
// the row pointers as passes of their own moved 56: 0.86 ms for 67 M keys on MI355X, against
// 0.29 ms now).
constexpr int kCsxItems = 8;
constexpr int kCsxTile = 256 * kCsxItems;

// key q is the first of its run of equal keys
__device__ __forceinline__ bool csx_first(const uint64_t* __restrict__ keys, uint64_t q, bool uniq) {
  return !uniq || q == 0 || keys[q] != keys[q - 1];
}

__global__ __launch_bounds__(256) void csx_count_kernel(const uint64_t* __restrict__ keys, uint64_t m,
                                                        uint32_t* __restrict__ count) {
  __shared__ uint32_t red[4];
  const uint64_t base = (uint64_t)blockIdx.x * kCsxTile + threadIdx.x;
  uint32_t c = 0;
#pragma unroll
  for (int j = 0; j < kCsxItems; ++j) {
    const uint64_t q = base + (uint64_t)j * 256;
    if (q < m && csx_first(keys, q, true)) ++c;
  }
  c = block_sum<256>(c, red);
  if (threadIdx.x == 0) count[blockIdx.x] = c;
}

// before: distinct keys before each tile (null without uniq: the keys before it).  Rows up to the
// last key's get their pointer here, the rows after it in csx_tail_kernel.
__global__ __launch_bounds__(256) void csx_write_kernel(const uint64_t* __restrict__ keys, uint64_t m, int b,
                                                        const uint32_t* __restrict__ before,
                                                        uint32_t* __restrict__ ptr, uint32_t* __restrict__ ent) {
  __shared__ uint32_t wave_total[4];
  const uint32_t w = threadIdx.x >> 6, lane = lane_id();
  const uint64_t base = (uint64_t)blockIdx.x * kCsxTile + w * (kCsxItems * 64) + lane;
  uint64_t k[kCsxItems], prev[kCsxItems], first[kCsxItems];
#pragma unroll
  for (int j = 0; j < kCsxItems; ++j) {
    const uint64_t q = base + 64 * j;
    k[j] = q < m ? keys[q] : 0ull;
    prev[j] = q < m && q ? keys[q - 1] : ~0ull;  // no key: ids take fewer than 64 bits
  }
  uint32_t total = 0;
#pragma unroll
  for (int j = 0; j < kCsxItems; ++j) {
    first[j] = __ballot(base + 64 * j < m && (!before || k[j] != prev[j]));
    total += (uint32_t)__popcll(first[j]);
  }
  if (lane == 0) wave_total[w] = total;
  __syncthreads();
  uint32_t pos = before ? before[blockIdx.x] : blockIdx.x * (uint32_t)kCsxTile;
  for (uint32_t q = 0; q < w; ++q) pos += wave_total[q];
  const uint64_t lt = __lanemask_lt();
#pragma unroll
  for (int j = 0; j < kCsxItems; ++j) {
    const bool mine = (first[j] >> lane) & 1ull;
    const uint32_t at = pos + (uint32_t)__popcll(first[j] & lt);
    pos += (uint32_t)__popcll(first[j]);
    // rows (row of the key before, row of this key] begin here
    const uint32_t row = (uint32_t)(k[j] >> b);
    const uint32_t lo = prev[j] == ~0ull ? 0u : (uint32_t)(prev[j] >> b) + 1u;
    if (mine) ent[at] = (uint32_t)(k[j] & ((1ull << b) - 1));
    const bool wide = mine && row >= lo && row - lo >= 32u;  // a long run of empty rows: by the whole wave
    if (mine && !wide && row >= lo)
      for (uint32_t r = lo; r <= row; ++r) ptr[r] = at;
    uint64_t todo = __ballot(wide);
    while (todo) {
      const int l = __builtin_ctzll(todo);
      todo &= todo - 1;
      const uint32_t r0 = (uint32_t)__shfl((int)lo, l), r1 = (uint32_t)__shfl((int)row, l),
                     v = (uint32_t)__shfl((int)at, l);
      for (uint64_t r = (uint64_t)r0 + lane; r <= r1; r += 64) ptr[r] = v;
    }
  }
}

// ptr[r] = m_out for the rows after the last key's, and the end
__global__ __launch_bounds__(256) void csx_tail_kernel(const uint64_t* __restrict__ keys, uint64_t m, uint32_t n, int b,
                                                       uint32_t m_out, uint32_t* __restrict__ ptr) {
  const uint64_t r = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (r <= n && r > (keys[m - 1] >> b)) ptr[r] = m_out;
}

__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// One atomic per workgroup of at most kMaxBlocks: those to one address take some 12 ns each (one per
// wave of 1024 workgroups took 38 to 53 us).
constexpr uint64_t kMaxBlocks = 512;
__global__ __launch_bounds__(256) void max_u32_kernel(const uint32_t* __restrict__ v, uint64_t n,
                                                      uint32_t* __restrict__ out) {
  __shared__ uint32_t wm[4];
  uint32_t m = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) m = max(m, v[i]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, 64));
  if (lane_id() == 0) wm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) atomicMax(out, max(max(wm[0], wm[1]), max(wm[2], wm[3])));
}

// Out-degree histogram of the CSC's source ids [build_degrees, common.hpp:110-121].  A
// grid of 2 workgroups per CU walks contiguous ranges of the ids with 16-byte loads, four
// in flight per lane (16 ids), and adds one per id with a non-returning atomic.  Ids below
// kDegLds are counted in a per-workgroup LDS histogram and flushed once per workgroup: on
// skewed graphs the hubs take most entries, and a million global atomics on one hub's
// counter serialise.  (RMAT's hubs have low ids; in the degree-ordered numbering every hub
// does.)  The ids are read once, so they are loaded non-temporally.
constexpr uint32_t kDegLds = 16384;
constexpr uint32_t kDegThreads = 512;
constexpr uint32_t kDegVec = 4;  // 16-byte loads in flight per lane
__device__ __forceinline__ void degree_count(uint32_t u, uint32_t n, uint32_t* h, uint32_t* deg) {
  if (u < kDegLds) {
    if (u < n) atomicAdd(&h[u], 1u);
  } else if (u < n) {
    atomicAdd(&deg[u], 1u);
  }
}
__global__ __launch_bounds__(kDegThreads) void degree_kernel(const uint32_t* __restrict__ col, uint64_t nnz,
                                                             uint32_t n, uint64_t vec_per_block,
                                                             uint32_t* __restrict__ deg) {
  __shared__ uint32_t h[kDegLds];
  for (uint32_t q = threadIdx.x; q < kDegLds; q += kDegThreads) h[q] = 0u;
  __syncthreads();
  const uint64_t nv = nnz / 4;  // whole 16-byte groups; the nnz % 4 tail is counted by workgroup 0
  const u32x4* c4 = reinterpret_cast<const u32x4*>(col);
  const uint64_t v0 = (uint64_t)blockIdx.x * vec_per_block;
  const uint64_t v1 = v0 + vec_per_block < nv ? v0 + vec_per_block : nv;
  for (uint64_t v = v0 + threadIdx.x; v < v1; v += (uint64_t)kDegThreads * kDegVec) {
    u32x4 a[kDegVec];
#pragma unroll
    for (uint32_t t = 0; t < kDegVec; ++t) {
      const uint64_t q = v + (uint64_t)t * kDegThreads;
      a[t] = q < v1 ? __builtin_nontemporal_load(c4 + q) : u32x4{n, n, n, n};  // id n counts nothing
    }
#pragma unroll
    for (uint32_t t = 0; t < kDegVec; ++t) {
      degree_count(a[t].x, n, h, deg);
      degree_count(a[t].y, n, h, deg);
      degree_count(a[t].z, n, h, deg);
      degree_count(a[t].w, n, h, deg);
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < nnz - nv * 4) degree_count(col[nv * 4 + threadIdx.x], n, h, deg);
  __syncthreads();
  for (uint32_t q = threadIdx.x; q < kDegLds && q < n; q += kDegThreads)
    if (h[q]) atomicAdd(&deg[q], h[q]);
}

// Out-degrees of a small or middling CSC without global atomics: workgroup (w, r) counts the
// ids of range r (kHistIds of them, two 16-bit counters to an LDS word) in chunk w of the
// column ids, at most kHistChunk of them, so that no counter passes 16 bits, and stores its
// counts; a second kernel adds the chunks' counts per id.  (degree_kernel's flush of every
// workgroup's LDS counters into one array of global counters queues on the hubs': 142 us for
// 1.5 M ids and 100,003 vertices on MI355X, 247 us for 3.1 M and 200,003; this form takes 19
// and 22 us.)  It reads the ids once per range and moves 4 bytes per id and chunk, so it serves
// CSCs whose counts, kHistBytes at most, stay in the caches.
constexpr uint32_t kHistIds = 1u << 16;
constexpr uint32_t kHistThreads = 1024;
constexpr uint32_t kHistRound = kHistThreads * 4;        // ids a workgroup reads at a time
constexpr uint32_t kHistChunk = 15 * kHistRound;         // 61440 < 2^16
constexpr uint64_t kHistBytes = 32ull << 20;
__global__ __launch_bounds__(kHistThreads) void hist_count_kernel(const uint32_t* __restrict__ col, uint64_t nnz,
                                                                  uint32_t chunk, uint32_t words,
                                                                  uint32_t* __restrict__ part) {
  __shared__ uint32_t h[kHistIds / 2];
  u32x4* h4 = reinterpret_cast<u32x4*>(h);
  for (uint32_t q = threadIdx.x; q < kHistIds / 8; q += kHistThreads) h4[q] = u32x4{0u, 0u, 0u, 0u};
  __syncthreads();
  const uint32_t first = blockIdx.y * kHistIds;
  const uint64_t p0 = (uint64_t)blockIdx.x * chunk, p1 = p0 + chunk < nnz ? p0 + chunk : nnz;
  auto count = [&](uint32_t u) {
    const uint32_t k = u - first;
    if (k < kHistIds) atomicAdd(&h[k >> 1], 1u << (16u * (k & 1u)));
  };
  for (uint64_t p = p0 + 4ull * threadIdx.x; p < p1; p += kHistRound) {
    if (p + 4 <= p1) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(col + p);
      count(v.x);
      count(v.y);
      count(v.z);
      count(v.w);
    } else {
      for (uint64_t q = p; q < p1; ++q) count(col[q]);
    }
  }
  __syncthreads();
  const uint32_t w0 = first / 2, nw = words - w0 < kHistIds / 2 ? words - w0 : kHistIds / 2;
  uint32_t* out = part + (uint64_t)blockIdx.x * words + w0;
  for (uint32_t q = threadIdx.x; q < nw; q += kHistThreads) out[q] = h[q];
}

// deg[i] = the chunks' counts of id i added; with given, *bad |= 1 where given[i] is below it
__global__ __launch_bounds__(256) void hist_add_kernel(uint32_t n, uint32_t words, uint32_t chunks,
                                                       const uint32_t* __restrict__ part, uint32_t* __restrict__ deg,
                                                       const uint32_t* __restrict__ given, uint32_t* __restrict__ bad) {
  const uint32_t w = blockIdx.x * 256 + threadIdx.x;
  if (w >= words) return;
  uint32_t lo = 0, hi = 0;
#pragma unroll 8
  for (uint32_t c = 0; c < chunks; ++c) {
    const uint32_t v = part[(uint64_t)c * words + w];
    lo += v & 0xFFFFu;
    hi += v >> 16;
  }
  const uint32_t i = 2 * w;
  if (given) {
    if ((i < n && given[i] < lo) || (i + 1 < n && given[i + 1] < hi)) *bad = 1u;
  } else {
    if (i < n) deg[i] = lo;
    if (i + 1 < n) deg[i + 1] = hi;
  }
}

// Out-degrees of a large CSC without global atomics: the ids are grouped by id range
// (2^kDegRangeBits ids per range) with a radix sort of the range bits only, then every range is
// counted in LDS histograms.  With at most 256 ranges the sort is one pass that keeps just the
// ids' low 16 bits and knows where every range starts (12 bytes moved per id); with more, a sort of
// whole ids, whose range starts are then looked up.  A range's entries are shared by kDegSplit
// workgroups; when one of them gets all, it stores its counts, else they are added.  At RMAT-22
// (65 M ids on MI355X) 0.58 ms, against 1.29 ms for sorting whole ids, read-back starts and items of
// 2^20 entries read two bytes at a time, of which the count alone took 0.71 ms; shares below 2^19
// entries pay more for their flushes than they save (2^16: 0.84 ms).  The global-atomic
// histogram is bound by the device's atomic rate (~1.3e10 per second).
constexpr int kDegRangeBits = 14;
constexpr uint32_t kDegRange = 1u << kDegRangeBits;
constexpr uint64_t kDegSortMin = 1ull << 24;  // entries from which the range path is taken
constexpr uint32_t kDegSplit = 32;            // most workgroups of a range
constexpr uint32_t kDegMin = 1u << 19;        // entries that one workgroup takes alone
constexpr uint32_t kDegCountThreads = 1024;

// start[r] = first position whose id's range is >= r, r in [0, nr]; every r written once
__global__ __launch_bounds__(256) void range_start_kernel(const uint32_t* __restrict__ ids, uint64_t nnz, uint32_t nr,
                                                          uint32_t* __restrict__ start) {
  const uint64_t p = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (p > nnz) return;
  const uint32_t a = p == 0 ? 0u : (ids[p - 1] >> kDegRangeBits) + 1u;
  uint32_t b = p == nnz ? nr : (ids[p] >> kDegRangeBits);
  if (b > nr) b = nr;  // ids are below n (checked by the callers); never write past the table
  for (uint32_t r = a; r <= b; ++r) start[r] = (uint32_t)p;
}

// workgroup (r, y): LDS counts of its share of range r's ids
template <class Id>
__global__ __launch_bounds__(kDegCountThreads) void range_count_kernel(const Id* __restrict__ ids,
                                                                       const uint32_t* __restrict__ start, uint32_t n,
                                                                       uint32_t* __restrict__ deg) {
  __shared__ uint32_t h[kDegRange];
  const uint32_t e0 = start[blockIdx.x], e1 = start[blockIdx.x + 1];
  const uint32_t share = max(kDegMin, (uint32_t)(((uint64_t)(e1 - e0) + kDegSplit - 1) / kDegSplit));
  const uint64_t p0 = e0 + (uint64_t)blockIdx.y * share;
  if (blockIdx.y && p0 >= e1) return;
  const uint64_t p1 = p0 + share < e1 ? p0 + share : e1;
  for (uint32_t q = threadIdx.x; q < kDegRange; q += kDegCountThreads) h[q] = 0u;
  __syncthreads();
  // 16-byte loads: a workgroup alone on a range has its CU's bandwidth only with enough in flight
  constexpr uint32_t kPer = 16 / sizeof(Id);
  const uint64_t a0 = (p0 + kPer - 1) / kPer * kPer, a1 = p1 / kPer * kPer;  // whole 16-byte groups of [p0, p1)
  auto count = [&](uint32_t u) { atomicAdd(&h[u & (kDegRange - 1)], 1u); };
  auto ends = [&](uint64_t q0, uint64_t q1) {
    if (q0 + threadIdx.x < q1) count(ids[q0 + threadIdx.x]);
  };
  if (a0 >= a1) {
    ends(p0, p1);  // fewer than 2 kPer ids
  } else {
    ends(p0, a0);
    ends(a1, p1);
  }
  for (uint64_t p = a0 + (uint64_t)threadIdx.x * kPer; p < a1; p += (uint64_t)kDegCountThreads * kPer) {
    const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(ids + p));
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      count(w[t]);
      if constexpr (sizeof(Id) == 2) count(w[t] >> 16);
    }
  }
  __syncthreads();
  const uint32_t v0 = blockIdx.x << kDegRangeBits;
  const uint32_t cnt = n - v0 < kDegRange ? n - v0 : kDegRange;
  const bool split = e1 - e0 > share;
  for (uint32_t q = threadIdx.x; q < cnt; q += kDegCountThreads) {
    if (!split) deg[v0 + q] = h[q];
    else if (h[q]) atomicAdd(&deg[v0 + q], h[q]);
  }
}

// *bad = 1 when some given out-degree is below the number of entries of its vertex
__global__ __launch_bounds__(256) void outdeg_check_kernel(uint32_t n, const uint32_t* __restrict__ given,
                                                           const uint32_t* __restrict__ counted,
                                                           uint32_t* __restrict__ bad) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n && given[i] < counted[i]) *bad = 1u;
}

// CSR keys from a CSC: (source << b) | target, payload = CSC position; one thread per CSC row.
__global__ __launch_bounds__(256) void transpose_keys_kernel(uint32_t n, const uint32_t* __restrict__ ptr,
                                                             const uint32_t* __restrict__ col, int b,
                                                             uint64_t* __restrict__ keys,
                                                             uint32_t* __restrict__ pos) {
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  for (uint32_t p = ptr[r]; p < ptr[r + 1]; ++p) {
    keys[p] = ((uint64_t)col[p] << b) | r;
    pos[p] = p;
  }
}

inline uint32_t grid_for(uint64_t n) { return (uint32_t)ceil_div(n ? n : 1, 256); }

uint32_t read_back_u32(hipStream_t s, const uint32_t* d) {
  uint32_t h = 0;
  NWG_HIP(hipMemcpyAsync(&h, d, sizeof h, hipMemcpyDeviceToHost, s));
  NWG_HIP(hipStreamSynchronize(s));
  return h;
}

}  // namespace

static const char* const kBadCsc = "CSC: row pointers not monotone from 0 to nnz, or an entry >= n";

int key_bits_for(uint32_t n) { return bits_for(n); }

// row pointers and entries from m sorted keys; before (nullable): distinct keys before each tile
static void csx_write(hipStream_t s, const uint64_t* keys, uint64_t m, const uint32_t* before, uint32_t m_out,
                      uint32_t n, int b, uint32_t* ptr, uint32_t* ent) {
  if (m) {
    csx_write_kernel<<<(uint32_t)ceil_div(m, kCsxTile), 256, 0, s>>>(keys, m, b, before, ptr, ent);
    csx_tail_kernel<<<grid_for((uint64_t)n + 1), 256, 0, s>>>(keys, m, n, b, m_out, ptr);
  } else {
    fill_u32_kernel<<<grid_for((uint64_t)n + 1), 256, 0, s>>>(ptr, (uint64_t)n + 1, 0u);
  }
  NWG_LAUNCH_CHECK();
}

void sorted_keys_to_csx(hipStream_t s, const uint64_t* keys, uint64_t m, uint32_t n, int b, uint32_t* ptr,
                        uint32_t* ent) {
  csx_write(s, keys, m, nullptr, (uint32_t)m, n, b, ptr, ent);
}

// bad[0] = 1 for a CSC in device memory whose row pointers are not monotone from 0 to nnz or
// whose entries are not below n (a plain store of 1: every flagging thread writes the same)
__global__ __launch_bounds__(256) void csc_check_kernel(uint32_t n, uint64_t nnz, const uint32_t* __restrict__ ptr,
                                                        const uint32_t* __restrict__ idx, uint32_t* __restrict__ bad) {
  const uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  bool b = false;
  if (t < nnz) b = idx[t] >= n;
  if (t < n) b = b || ptr[t] > ptr[t + 1];
  if (t == 0) b = b || ptr[0] != 0u || ptr[n] != (uint32_t)nnz;
  if (b) *bad = 1u;
}

// Chunks of the private histograms of a CSC: ids per chunk and chunks; none when its counts
// would pass kHistBytes.
struct HistShape {
  uint32_t chunk = 0, chunks = 0, words = 0;
};
static HistShape hist_shape(uint32_t n, uint64_t nnz) {
  HistShape h;
  h.words = (n + 1) / 2;
  const uint64_t ranges = ceil_div(n, kHistIds);
  // about one workgroup per CU, in whole rounds
  const uint64_t want = ceil_div(ceil_div(nnz * ranges, 256), kHistRound) * kHistRound;
  h.chunk = (uint32_t)std::min<uint64_t>(std::max<uint64_t>(want, kHistRound), kHistChunk);
  const uint64_t chunks = ceil_div(nnz, h.chunk);
  if (nnz && ranges < 65536 && chunks * h.words * 4ull <= kHistBytes) h.chunks = (uint32_t)chunks;
  return h;
}

static void hist_enqueue(hipStream_t s, const HistShape& h, uint32_t n, uint64_t nnz, const uint32_t* col,
                         uint32_t* part, uint32_t* deg, const uint32_t* given, uint32_t* bad) {
  hist_count_kernel<<<dim3(h.chunks, (uint32_t)ceil_div(n, kHistIds)), kHistThreads, 0, s>>>(col, nnz, h.chunk, h.words,
                                                                                           part);
  hist_add_kernel<<<grid_for(h.words), 256, 0, s>>>(n, h.words, h.chunks, part, deg, given, bad);
  NWG_LAUNCH_CHECK();
}

// The range path for a large CSC (ids below n < 2^32 assumed checked).
static void out_degrees_by_range(hipStream_t s, uint32_t n, uint64_t nnz, const uint32_t* col, uint32_t* deg) {
  const uint32_t nr = (uint32_t)ceil_div(n, kDegRange);
  fill_u32_kernel<<<grid_for(n), 256, 0, s>>>(deg, n, 0u);
  NWG_LAUNCH_CHECK();
  const int bits = std::max(1, bits_for(n) - kDegRangeBits);
  const dim3 grid(nr, kDegSplit);
  if (bits <= 8) {
    DevBuf<uint16_t> low(nnz);
    DevBuf<uint32_t> start((1u << bits) + 1);
    radix_partition_low16(s, col, nnz, kDegRangeBits, bits, low.p, start.p);
    range_count_kernel<uint16_t><<<grid, kDegCountThreads, 0, s>>>(low.p, start.p, n, deg);
  } else {
    DevBuf<uint32_t> ids(nnz), tmp(nnz), start((uint64_t)nr + 1);
    radix_sort_keys_u32(s, ids, tmp, col, nnz, kDegRangeBits, bits_for(n));
    range_start_kernel<<<grid_for(nnz + 1), 256, 0, s>>>(ids.p, nnz, nr, start.p);
    range_count_kernel<uint32_t><<<grid, kDegCountThreads, 0, s>>>(ids.p, start.p, n, deg);
  }
  NWG_LAUNCH_CHECK();
}

static void degrees_aligned(const uint32_t* col) {
  NWG_REQUIRE(reinterpret_cast<uintptr_t>(col) % 16 == 0, "column ids must be 16-byte aligned");
}

// the LDS + global-atomic histogram
static void out_degrees_atomic(hipStream_t s, uint32_t n, uint64_t nnz, const uint32_t* col, uint32_t* deg) {
  fill_u32_kernel<<<grid_for(n), 256, 0, s>>>(deg, n, 0u);
  NWG_LAUNCH_CHECK();
  if (nnz) {
    int dev = 0, cus = 0;
    NWG_HIP(hipGetDevice(&dev));
    NWG_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    // ranges of whole lane rounds (kDegThreads x kDegVec groups of 4 ids), about 2 per CU
    const uint64_t round = (uint64_t)kDegThreads * kDegVec;
    const uint64_t nv = nnz / 4;
    const uint64_t per = std::max<uint64_t>(1, ceil_div(ceil_div(nv, 2ull * std::max(cus, 1)), round)) * round;
    const uint32_t blocks = (uint32_t)std::max<uint64_t>(1, ceil_div(nv, per));
    degree_kernel<<<blocks, kDegThreads, 0, s>>>(col, nnz, n, per, deg);
    NWG_LAUNCH_CHECK();
  }
}

void out_degrees_device(hipStream_t s, uint32_t n, uint64_t nnz, const uint32_t* col, uint32_t* deg) {
  degrees_aligned(col);
  const HistShape h = hist_shape(n, nnz);
  if (h.chunks) {
    DevBuf<uint32_t> part((uint64_t)h.chunks * h.words);
    hist_enqueue(s, h, n, nnz, col, part.p, deg, nullptr, nullptr);
    return;
  }
  if (nnz >= kDegSortMin && nnz < (1ull << 32)) {
    out_degrees_by_range(s, n, nnz, col, deg);
    return;
  }
  out_degrees_atomic(s, n, nnz, col, deg);
}

void check_device_csc(hipStream_t s, uint32_t n, uint64_t nnz, const uint32_t* ptr, const uint32_t* col,
                      const uint32_t* given, uint32_t* deg, const CscCheckScratch* scratch, bool wait) {
  NWG_REQUIRE(wait || scratch, "the check's flags outlive it in the caller's memory only");
  if (given || deg) degrees_aligned(col);
  DevBuf<uint32_t> own_flags, own_part, own_counted;
  uint32_t* flags = scratch ? scratch->flags : (own_flags.alloc(3), own_flags.p);
  fill_u32_kernel<<<1, 256, 0, s>>>(flags, 3, 0u);
  csc_check_kernel<<<grid_for(std::max<uint64_t>(nnz, n)), 256, 0, s>>>(n, nnz, ptr, col, flags);
  NWG_LAUNCH_CHECK();
  // the histograms count ids >= n nowhere, so they need not wait for the check above
  const HistShape h = hist_shape(n, nnz);
  const bool hist = h.chunks && (!scratch || (uint64_t)h.chunks * h.words * 4 <= scratch->part_bytes);
  if (given || deg) {
    uint32_t* counts = deg;
    if (!counts) counts = scratch ? scratch->counted : (own_counted.alloc(n), own_counted.p);
    if (hist) {
      uint32_t* part = scratch ? scratch->part : (own_part.alloc((uint64_t)h.chunks * h.words), own_part.p);
      hist_enqueue(s, h, n, nnz, col, part, counts, given, flags + 1);
    } else {
      if (!scratch && nnz >= kDegSortMin) {
        // the range path sorts and indexes by the ids: only once they are known to be in range
        if (read_back_u32(s, flags)) throw Error(NWG_EINVAL, kBadCsc);
        out_degrees_device(s, n, nnz, col, counts);
      } else {
        out_degrees_atomic(s, n, nnz, col, counts);
      }
      if (given) outdeg_check_kernel<<<grid_for(n), 256, 0, s>>>(n, given, counts, flags + 1);
      NWG_LAUNCH_CHECK();
    }
  }
  if (!wait) return;
  uint32_t bad[2] = {0, 0};
  NWG_HIP(hipMemcpyAsync(bad, flags, sizeof bad, hipMemcpyDeviceToHost, s));
  NWG_HIP(hipStreamSynchronize(s));
  csc_verdict(bad[0], bad[1]);
}

void csc_verdict(uint64_t bad_csc, uint64_t bad_outdeg) {
  if (bad_csc) throw Error(NWG_EINVAL, kBadCsc);
  if (bad_outdeg) throw Error(NWG_EINVAL, "outdeg: some vertex's out-degree is below its number of entries in the CSC");
}

void build_csc_device(hipStream_t s, uint32_t n, uint64_t ne, const uint32_t* src, const uint32_t* dst, bool clean,
                      nwg_graph* g) {
  NWG_REQUIRE(n >= 1, "graph needs at least one vertex");
  NWG_REQUIRE(ne < (1ull << 32), "edge count must be below 2^32 (uint32 indices)");
  const int b = bits_for(n);
  DevBuf<uint64_t> keys(ne ? ne : 1), tmp(ne ? ne : 1);
  DevBuf<uint32_t> bad(1);
  fill_u32_kernel<<<1, 256, 0, s>>>(bad.p, 1, 0u);
  const uint64_t m = radix_sort_edges(s, EdgeKeySource{src, dst, n, b, clean, bad.p}, ne, keys, tmp);
  uint64_t nnz = m;
  const uint32_t tiles = (uint32_t)ceil_div(m, kCsxTile);
  DevBuf<uint32_t> count, before;
  if (clean && m) {
    count.alloc(tiles);
    before.alloc((uint64_t)tiles + 1);
    csx_count_kernel<<<tiles, 256, 0, s>>>(keys.p, m, count.p);
    NWG_LAUNCH_CHECK();
    exclusive_scan_u32(s, count.p, before.p, tiles);
    nnz = read_back_u32(s, before.p + tiles);
  }
  g->csc_ptr.alloc((uint64_t)n + 1);
  g->csc_idx.alloc(nnz ? nnz : 1);
  csx_write(s, keys.p, m, before.p, (uint32_t)nnz, n, b, g->csc_ptr.p, g->csc_idx.p);
  g->n = n;
  g->nnz = nnz;
  g->outdeg.alloc(n);
  out_degrees_device(s, n, nnz, g->csc_idx.p, g->outdeg.p);
  if (g->nnz >= kSkewEdges) note_max_outdeg(s, g);  // waits
  else NWG_HIP(hipStreamSynchronize(s));
}

void note_max_outdeg(hipStream_t s, nwg_graph* g) {
  if (g->nnz < kSkewEdges) return;
  DevBuf<uint32_t> m(1);
  fill_u32_kernel<<<1, 256, 0, s>>>(m.p, 1, 0u);
  max_u32_kernel<<<(uint32_t)std::min<uint64_t>(grid_for(g->n), kMaxBlocks), 256, 0, s>>>(g->outdeg.p, g->n, m.p);
  NWG_LAUNCH_CHECK();
  g->max_outdeg = read_back_u32(s, m.p);
}

bool skewed_degrees(const nwg_graph* g) {
  return (double)g->max_outdeg > 64.0 + 8.0 * (double)g->nnz / (double)std::max<uint32_t>(g->n, 1);
}

void build_csr_device(hipStream_t s, nwg_graph* g) {
  if (g->has_csr) return;
  const uint32_t n = g->n;
  const uint64_t nnz = g->nnz;
  const int b = bits_for(n);
  DevBuf<uint64_t> keys(nnz ? nnz : 1), tmp(nnz ? nnz : 1);
  DevBuf<uint32_t> pos(nnz ? nnz : 1), pos_tmp(nnz ? nnz : 1);
  if (nnz) {
    transpose_keys_kernel<<<grid_for(n), 256, 0, s>>>(n, g->csc_ptr.p, g->csc_idx.p, b, keys.p, pos.p);
    NWG_LAUNCH_CHECK();
    // the CSC's positions ascend by target, and the sort is stable: by source is enough
    radix_sort_pairs(s, keys, tmp, &pos, &pos_tmp, nnz, b, 2 * b);
  }
  g->csr_ptr.alloc((uint64_t)n + 1);
  g->csr_idx.alloc(nnz ? nnz : 1);
  csx_write(s, keys.p, nnz, nullptr, (uint32_t)nnz, n, b, g->csr_ptr.p, g->csr_idx.p);
  g->csr_to_csc = std::move(pos);
  NWG_HIP(hipStreamSynchronize(s));
  g->has_csr = true;
}

}  // namespace nwg
