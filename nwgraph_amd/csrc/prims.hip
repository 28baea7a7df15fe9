// prims.hip -- device-wide exclusive scan and stable LSD radix sort.
//
// Scan: reduce-then-scan over 2048-element tiles (256 threads x 8 items), recursing on the tile
// sums.
#include "device_utils.hpp"
#include "nwg_internal.hpp"

namespace nwg {

namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__global__ __launch_bounds__(kScanThreads) void scan_reduce_kernel(const uint32_t* __restrict__ in, uint64_t n,
                                                                   uint32_t* __restrict__ sums) {
  __shared__ uint32_t lds[kScanThreads / 64];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile;
  uint32_t s = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    uint64_t i = base + (uint64_t)j * kScanThreads + threadIdx.x;
    if (i < n) s += in[i];
  }
  s = block_sum<kScanThreads>(s, lds);
  if (threadIdx.x == 0) sums[blockIdx.x] = s;
}

// out[i] = offsets[block] + exclusive prefix inside the tile; the last tile writes out[n].
__global__ __launch_bounds__(kScanThreads) void scan_tiles_kernel(const uint32_t* __restrict__ in,
                                                                  uint32_t* __restrict__ out, uint64_t n,
                                                                  const uint32_t* __restrict__ offsets) {
  __shared__ uint32_t lds[kScanThreads / 64 + 1];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
  uint32_t v[kScanItems];
  uint32_t s = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    uint64_t i = base + j;
    v[j] = i < n ? in[i] : 0u;
    s += v[j];
  }
  uint32_t total;
  uint32_t pre = block_exclusive_scan<kScanThreads>(s, lds, &total);
  const uint32_t off = offsets ? offsets[blockIdx.x] : 0u;
  pre += off;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    uint64_t i = base + j;
    if (i < n) out[i] = pre;
    pre += v[j];
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = off + total;
}

}  // namespace

void exclusive_scan_u32(hipStream_t s, const uint32_t* in, uint32_t* out, uint64_t n) {
  const uint64_t nb = ceil_div(n ? n : 1, kScanTile);
  if (nb == 1) {
    scan_tiles_kernel<<<1, kScanThreads, 0, s>>>(in, out, n, nullptr);
    NWG_LAUNCH_CHECK();
    return;
  }
  DevBuf<uint32_t> sums(nb), offs(nb + 1);
  scan_reduce_kernel<<<(uint32_t)nb, kScanThreads, 0, s>>>(in, n, sums.p);
  NWG_LAUNCH_CHECK();
  exclusive_scan_u32(s, sums.p, offs.p, nb);
  scan_tiles_kernel<<<(uint32_t)nb, kScanThreads, 0, s>>>(in, out, n, offs.p);
  NWG_LAUNCH_CHECK();
  // the temporaries go back to the call's pool, whose next user runs on s after these kernels
}

// ---------------------------------------------------------------------------
// radix sort
// ---------------------------------------------------------------------------
// A pass over digits of at most 8 bits: an upsweep counts every tile's digits, a scan of the
// digit-major counts gives each (digit, tile) its place in the output, and the scatter ranks the
// tile's keys, puts them in digit order in LDS and writes each digit's run out contiguously.
//
// Ranking.  Wave w takes kRsItems x 64 consecutive keys of the tile, 64 at a time in order, and
// keeps its own digit counters in LDS.  Lanes with the same digit find each other by ballots; the
// first of them reads and advances the counter.  No barrier is needed until all keys are
// ranked (a workgroup-wide counter took three barriers per 256 keys, 458 us for a pass of 67 M 64-bit
// keys on MI355X, 2.3 TB/s; this form takes 271 us, 4.0 TB/s).
namespace {

constexpr int kRsThreads = 512;
constexpr int kRsItems = 8;
constexpr int kRsTile = kRsThreads * kRsItems;
constexpr int kRsWaves = kRsThreads / 64;

// Where a pass reads its keys: an array, or the packed keys of an edge list, of which invalid
// edges are dropped (counted nowhere and written nowhere).
template <class K>
struct KeyArray {
  typedef K Key;
  const K* keys;
  uint64_t n;
  __device__ __forceinline__ bool get(uint64_t i, K& k) const {
    if (i >= n) return false;
    k = keys[i];
    return true;
  }
  __device__ __forceinline__ void note(uint64_t) const {}
};
struct EdgeKeys {
  typedef uint64_t Key;
  EdgeKeySource e;
  uint64_t n;
  __device__ __forceinline__ bool get(uint64_t i, uint64_t& k) const {
    if (i >= n) return false;
    const uint32_t u = e.src[i], v = e.dst[i];
    k = ((uint64_t)v << e.bits) | u;
    return u < e.n && v < e.n && !(e.drop_loops && u == v);
  }
  // *bad = 1 for an id out of range in an edge that would be kept
  __device__ __forceinline__ void note(uint64_t i) const {
    if (i >= n) return;
    const uint32_t u = e.src[i], v = e.dst[i];
    if ((u >= e.n || v >= e.n) && !(e.drop_loops && u == v)) *e.bad = 1u;
  }
};

template <class Src>
__global__ __launch_bounds__(kRsThreads) void rs_upsweep_kernel(Src src, int shift, uint32_t mask, uint32_t nb,
                                                                uint32_t* __restrict__ hist) {
  __shared__ uint32_t cnt[kRsWaves][256];  // a set per wave: fewer lanes on one counter
  for (uint32_t q = threadIdx.x; q < kRsWaves * 256; q += kRsThreads) (&cnt[0][0])[q] = 0u;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * kRsTile + threadIdx.x;
  uint32_t* mine = cnt[threadIdx.x >> 6];
  typename Src::Key k[kRsItems];
  bool ok[kRsItems];
#pragma unroll
  for (int j = 0; j < kRsItems; ++j) {
    ok[j] = src.get(base + (uint64_t)j * kRsThreads, k[j]);
    if (!ok[j]) src.note(base + (uint64_t)j * kRsThreads);
  }
#pragma unroll
  for (int j = 0; j < kRsItems; ++j)
    if (ok[j]) atomicAdd(&mine[(uint32_t)(k[j] >> shift) & mask], 1u);
  __syncthreads();
  if (threadIdx.x <= mask) {
    uint32_t c = 0;
#pragma unroll
    for (int w = 0; w < kRsWaves; ++w) c += cnt[w][threadIdx.x];
    hist[(uint64_t)threadIdx.x * nb + blockIdx.x] = c;
  }
}

// Out: what is written of a key (the key, or its low bits)
template <class Src, class Out, bool HasVals>
__global__ __launch_bounds__(kRsThreads) void rs_scatter_kernel(Src src, const uint32_t* __restrict__ vals_in,
                                                                Out* __restrict__ keys_out,
                                                                uint32_t* __restrict__ vals_out, int shift,
                                                                uint32_t mask, uint32_t nb,
                                                                const uint32_t* __restrict__ hist_scan) {
  typedef typename Src::Key K;
  __shared__ K sk[kRsTile];
  __shared__ uint32_t sv[HasVals ? kRsTile : 1];
  __shared__ uint32_t cnt[kRsWaves][256];
  __shared__ uint32_t gofs[256];  // a digit's place in the output, less its place in the tile
  __shared__ uint32_t scan_lds[kRsThreads / 64 + 1];

  const uint32_t tid = threadIdx.x, lane = lane_id(), w = tid / 64;
  for (uint32_t q = tid; q < kRsWaves * 256; q += kRsThreads) (&cnt[0][0])[q] = 0u;
  const uint64_t base = (uint64_t)blockIdx.x * kRsTile + w * (kRsItems * 64) + lane;
  K key[kRsItems];
  uint32_t val[HasVals ? kRsItems : 1];
  uint32_t rank[kRsItems];
  bool ok[kRsItems];
#pragma unroll
  for (int j = 0; j < kRsItems; ++j) {
    key[j] = 0;
    ok[j] = src.get(base + 64 * j, key[j]);
    if constexpr (HasVals) val[j] = ok[j] ? vals_in[base + 64 * j] : 0u;
  }
  uint32_t place = 0;
  if (tid <= mask) place = hist_scan[(uint64_t)tid * nb + blockIdx.x];
  __syncthreads();
  const uint64_t lt_mask = __lanemask_lt();
  volatile uint32_t* mine = cnt[w];  // read and written by this wave only, in program order
#pragma unroll
  for (int j = 0; j < kRsItems; ++j) {
    const uint32_t dg = (uint32_t)(key[j] >> shift) & mask;
    uint64_t peers = __ballot(ok[j]);
#pragma unroll
    for (int bit = 0; bit < 8; ++bit) {
      const bool set = (dg >> bit) & 1u;
      const uint64_t bb = __ballot(set);
      peers &= set ? bb : ~bb;
    }
    const uint32_t r = (uint32_t)__popcll(peers & lt_mask);
    const uint32_t pre = mine[dg];
    __builtin_amdgcn_wave_barrier();
    if (ok[j] && r == 0) mine[dg] = pre + (uint32_t)__popcll(peers);
    __builtin_amdgcn_wave_barrier();
    rank[j] = pre + r;
  }
  __syncthreads();
  // cnt[w][d] -> first place in the tile of wave w's keys of digit d
  uint32_t c[kRsWaves], sum = 0;
  if (tid < 256) {
#pragma unroll
    for (int q = 0; q < kRsWaves; ++q) {
      c[q] = sum;
      sum += cnt[q][tid];
    }
  }
  uint32_t total;
  const uint32_t first = block_exclusive_scan<kRsThreads>(sum, scan_lds, &total);
  if (tid < 256) {
#pragma unroll
    for (int q = 0; q < kRsWaves; ++q) cnt[q][tid] = first + c[q];
    gofs[tid] = place - first;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kRsItems; ++j) {
    if (!ok[j]) continue;
    const uint32_t lp = cnt[w][(uint32_t)(key[j] >> shift) & mask] + rank[j];
    sk[lp] = key[j];
    if constexpr (HasVals) sv[lp] = val[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kRsItems; ++j) {
    const uint32_t li = (uint32_t)j * kRsThreads + tid;
    if (li < total) {
      const K k = sk[li];
      const uint32_t o = gofs[(uint32_t)(k >> shift) & mask] + li;
      keys_out[o] = (Out)k;
      if constexpr (HasVals) vals_out[o] = sv[li];
    }
  }
}

// start[d] = where digit d begins in the output, d in [0, digits]
__global__ __launch_bounds__(256) void digit_start_kernel(uint32_t digits, uint32_t nb,
                                                          const uint32_t* __restrict__ scan,
                                                          uint32_t* __restrict__ start) {
  const uint32_t d = blockIdx.x * 256 + threadIdx.x;
  if (d <= digits) start[d] = scan[(uint64_t)d * nb];
}

// The tile counts of one sort's passes and their scan.
struct RadixSpace {
  uint32_t nb;
  DevBuf<uint32_t> hist, scan;
  explicit RadixSpace(uint64_t n) : nb((uint32_t)ceil_div(n, kRsTile)), hist(256ull * nb), scan(256ull * nb + 1) {}
};

template <class Src, class Out, bool HasVals>
void radix_pass(hipStream_t s, RadixSpace& sp, const Src& src, const uint32_t* vi, Out* ko, uint32_t* vo, int shift,
                int bits) {
  const uint32_t mask = (1u << bits) - 1u;
  rs_upsweep_kernel<Src><<<sp.nb, kRsThreads, 0, s>>>(src, shift, mask, sp.nb, sp.hist.p);
  NWG_LAUNCH_CHECK();
  exclusive_scan_u32(s, sp.hist.p, sp.scan.p, (uint64_t)sp.nb << bits);
  rs_scatter_kernel<Src, Out, HasVals><<<sp.nb, kRsThreads, 0, s>>>(src, vi, ko, vo, shift, mask, sp.nb, sp.scan.p);
  NWG_LAUNCH_CHECK();
}

// bits of the next pass over [shift, end): the passes share the bits evenly
int next_bits(int shift, int end) {
  const int left = end - shift, passes = (left + 7) / 8;
  return (left + passes - 1) / passes;
}

}  // namespace

void radix_sort_pairs(hipStream_t s, DevBuf<uint64_t>& keys, DevBuf<uint64_t>& keys_tmp, DevBuf<uint32_t>* vals,
                      DevBuf<uint32_t>* vals_tmp, uint64_t n, int first_bit, int end_bit) {
  if (n < 2 || end_bit <= first_bit) return;
  NWG_REQUIRE(n < (1ull << 32), "radix sort supports fewer than 2^32 keys");
  RadixSpace sp(n);
  for (int shift = first_bit; shift < end_bit;) {
    const int bits = next_bits(shift, end_bit);
    const KeyArray<uint64_t> src{keys.p, n};
    if (vals)
      radix_pass<KeyArray<uint64_t>, uint64_t, true>(s, sp, src, vals->p, keys_tmp.p, vals_tmp->p, shift, bits);
    else
      radix_pass<KeyArray<uint64_t>, uint64_t, false>(s, sp, src, nullptr, keys_tmp.p, nullptr, shift, bits);
    keys.swap(keys_tmp);
    if (vals) vals->swap(*vals_tmp);
    shift += bits;
  }
}

uint64_t radix_sort_edges(hipStream_t s, const EdgeKeySource& e, uint64_t ne, DevBuf<uint64_t>& keys,
                          DevBuf<uint64_t>& keys_tmp) {
  if (!ne) return 0;
  NWG_REQUIRE(ne < (1ull << 32), "radix sort supports fewer than 2^32 keys");
  const int end_bit = 2 * e.bits;
  const int bits = next_bits(0, end_bit);
  uint32_t back[2] = {0, 0};  // edges kept, bad
  {
    RadixSpace sp(ne);
    radix_pass<EdgeKeys, uint64_t, false>(s, sp, EdgeKeys{e, ne}, nullptr, keys.p, nullptr, 0, bits);
    NWG_HIP(hipMemcpyAsync(&back[0], sp.scan.p + ((uint64_t)sp.nb << bits), 4, hipMemcpyDeviceToHost, s));
    NWG_HIP(hipMemcpyAsync(&back[1], e.bad, 4, hipMemcpyDeviceToHost, s));
    NWG_HIP(hipStreamSynchronize(s));
  }
  if (back[1]) throw Error(NWG_EINVAL, "edge list holds a vertex id >= n");
  radix_sort_pairs(s, keys, keys_tmp, nullptr, nullptr, back[0], bits, end_bit);
  return back[0];
}

void radix_sort_keys_u32(hipStream_t s, DevBuf<uint32_t>& keys, DevBuf<uint32_t>& keys_tmp, const uint32_t* in,
                         uint64_t n, int first_bit, int end_bit) {
  NWG_REQUIRE(n >= 1 && n < (1ull << 32), "radix sort supports 1 to 2^32 - 1 keys");
  NWG_REQUIRE(first_bit >= 0 && end_bit <= 32 && first_bit < end_bit, "key bits must lie in [0, 32)");
  RadixSpace sp(n);
  const uint32_t* from = in;
  for (int shift = first_bit; shift < end_bit;) {
    const int bits = next_bits(shift, end_bit);
    radix_pass<KeyArray<uint32_t>, uint32_t, false>(s, sp, KeyArray<uint32_t>{from, n}, nullptr, keys_tmp.p, nullptr,
                                                    shift, bits);
    keys.swap(keys_tmp);
    from = keys.p;
    shift += bits;
  }
}

void radix_partition_low16(hipStream_t s, const uint32_t* in, uint64_t n, int shift, int bits, uint16_t* low,
                           uint32_t* start) {
  NWG_REQUIRE(n >= 1 && n < (1ull << 32) && bits >= 1 && bits <= 8, "partition of 1 to 2^32 - 1 keys by up to 8 bits");
  RadixSpace sp(n);
  radix_pass<KeyArray<uint32_t>, uint16_t, false>(s, sp, KeyArray<uint32_t>{in, n}, nullptr, low, nullptr, shift, bits);
  const uint32_t digits = 1u << bits;
  digit_start_kernel<<<(digits + 256) / 256, 256, 0, s>>>(digits, sp.nb, sp.scan.p, start);
  NWG_LAUNCH_CHECK();
}

}  // namespace nwg
