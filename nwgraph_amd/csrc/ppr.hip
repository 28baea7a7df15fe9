// ppr.hip -- k personalised PageRank vectors as one SpMM per sweep.
//
// Each vector j is the reference's PageRank loop (page_rank_v10 Jacobi schedule,
// include/nwgraph/experimental/algorithms/page_rank.hpp:377-432) with the uniform
// base (1-d)/N replaced by (1-d) v_j, v_j uniform over a small seed set, and its own
// stopping rule (first sweep with L1 change < threshold).  Contributions are tile-major,
// so one in-edge u of row i gathers the contiguous T-float slice C[tile][u][0..T) of the
// k-tile being served (T = 8/16/32/64) in one coalesced access.
// Scores are not kept during the solve: a row's old score is read back from its previous
// contribution (x / deg, or x itself for a row without out-edges), and the row-major N x k
// scores are written once at the end.
//
// Work split per sweep (one launch + one finishing launch), k-tile after k-tile, with T / 4 lanes of 16
// bytes per gathered slice (a lane group):
//   heavy pieces     at most 32 in-edges of one row with more than light_max, of one source slice
//                    (an eighth of the sources, one XCD's); the pieces of one row in a
//                    workgroup leave one partial vector
//   row workgroups   (1024/T) lane groups x 1 or 4 consecutive rows, over a compacted copy of the
//                    light rows
//   finish           heavy rows (partials added in order) and per-vector L1 changes folded
//                    (fixed point, order independent)
// A vector whose previous sweep converged is skipped (its lanes idle); a workgroup
// whose k-tile is entirely converged exits at once.  From the third sweep on, the rows
// after the last row with in-edges (their values fixed after one sweep) are not launched.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "device_utils.hpp"
#include "nwg_internal.hpp"

namespace nwg {

namespace {

constexpr int kThreads = 256;
constexpr uint32_t kSeedFlag = 0x80000000u;
// partials a finishing thread has in flight, and the vectors whose L1 changes its workgroup first adds
// in LDS
constexpr uint32_t kFinU = 8;
constexpr uint32_t kFinMaxK = 256;
constexpr uint32_t kFoldRows = 128;  // row-workgroup L1 partials per finishing workgroup, at most
// A workgroup adds its L1 changes to one of 8 lanes: atomics to one address take some 12 ns each
// on MI355X, and a solve has thousands of finishing workgroups.
constexpr uint32_t kErrLanes = 8;
// edges of a heavy row's piece (all their gathers are in flight at once)
constexpr uint32_t kPiece = 32;
struct PprParams {
  const uint32_t* rp;
  const uint32_t* lrp;   // light CSC: rows with in-degree <= light_max, heavy rows empty
  const uint32_t* lcol;
  const uint32_t* degflag;   // out-degree | kSeedFlag when the row is a seed of some vector
  const uint32_t* seed_row;  // sorted (row, vector) seed entries
  const uint32_t* seed_vec;
  const float* seed_base;    // (1-d) v_j[row] for the entry
  uint32_t n_seed;
  const float* cin;
  float* cout;
  uint32_t n, k;
  uint32_t tiles, kt_shift;  // k-tiles and log2 of their width
  float damp;
  uint32_t light_max;        // rows with in-degree <= light_max take the row path
  uint32_t row_blocks;       // workgroups of rows per k-tile
  uint32_t n_hub_rows;
  const uint32_t* hub_rows;
  const uint32_t* part_ptr;    // heavy row h's partials: hub_part rows [part_ptr[h], part_ptr[h + 1])
  const uint32_t* hcol;        // heavy rows' in-edges, source slice by source slice, row by row in each
  const uint2* pieces;         // piece p: edges [pieces[p].x, pieces[p + 1].x) of hcol, partial pieces[p].y
  uint32_t slice_off[kSlices + 1];  // slice x's pieces; whole workgroups of them
  uint32_t heavy_blocks;       // heavy workgroups per k-tile (a multiple of 8)
  uint32_t tile_blocks;        // workgroups per k-tile (a multiple of 8)
  uint32_t row_blocks_run;     // row workgroups per k-tile this sweep runs (and whose L1 partials are folded)
  uint32_t fold_rows;          // of whose L1 partials a finishing workgroup folds so many
  float* hub_part;           // n_parts x 4 kq
  double* blk_err;           // (row_blocks * tiles) x T
  unsigned long long* lanes;  // L1 changes: 3 rotating slots of kErrLanes lanes of kpad vectors
  unsigned long long* acc;   // iters x k: the lanes' sums, one sweep later
  uint32_t kpad;
  uint32_t kq;               // k in fours, rounded up
  uint32_t iter;
  double threshold;
};

// L1 change of vector j in sweep `iter`
__device__ __forceinline__ unsigned long long ppr_change(const unsigned long long* lanes, uint32_t kpad, uint32_t iter,
                                                         uint32_t j) {
  const unsigned long long* l = lanes + (uint64_t)(iter % 3) * kErrLanes * kpad + j;
  unsigned long long s = 0ull;
#pragma unroll
  for (uint32_t q = 0; q < kErrLanes; ++q) s += l[(uint64_t)q * kpad];
  return s;
}
__device__ __forceinline__ bool vec_done(const PprParams& P, uint32_t j) {
  return P.iter > 0 && fixed_to_err(ppr_change(P.lanes, P.kpad, P.iter - 1, j)) < P.threshold;
}

__device__ __forceinline__ float seed_base(const PprParams& P, uint32_t i, uint32_t j) {
  // lower_bound of i in seed_row, then scan the row's entries for vector j
  uint32_t lo = 0, hi = P.n_seed;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (P.seed_row[mid] < i) lo = mid + 1;
    else hi = mid;
  }
  float b = 0.f;
  for (uint32_t q = lo; q < P.n_seed && P.seed_row[q] == i; ++q)
    if (P.seed_vec[q] == j) b = P.seed_base[q];
  return b;
}

// Contributions are stored tile-major, [tile][row][T] (T = 1 << kt_shift vectors per tile),
// so that the gathers of one k-tile touch only that tile's array; scores stay row-major.
__device__ __forceinline__ uint64_t cidx(const PprParams& P, uint32_t i, uint32_t j) {
  return (((uint64_t)(j >> P.kt_shift) * P.n + i) << P.kt_shift) + (j & ((1u << P.kt_shift) - 1));
}

// Scores are not stored during the solve: the contribution array holds x / deg for a row with
// out-edges and x itself for a row without (no in-edge ever gathers it), and a row's old score
// is read back from the contributions of the previous sweep.
__device__ __forceinline__ float ppr_score(float c, uint32_t df) {
  const uint32_t d = df & ~kSeedFlag;
  return d ? c * (float)d : c;
}

// Four vectors of a tile at a time: a lane holds vectors j .. j + 3.
struct Four {
  float v[4];
};
__device__ __forceinline__ Four load4(const float* p) {
  const float4 f = *reinterpret_cast<const float4*>(p);
  return Four{{f.x, f.y, f.z, f.w}};
}

// Update of row i, vectors j .. j + 3 from their sums z, its degree/seed word df and the previous sweep's
// contributions xo (whose scores are within an ulp of the old ones).  Only the vectors in `live` change;
// err: their L1 changes, added.
__device__ __forceinline__ void ppr_update4(const PprParams& P, uint32_t i, uint32_t j, const Four& z, uint32_t df,
                                            const Four& xo, uint32_t live, double (&err)[4]) {
  const uint32_t d = df & ~kSeedFlag;
  float b[4] = {0.f, 0.f, 0.f, 0.f}, c[4];
  if (df & kSeedFlag)
#pragma unroll
    for (uint32_t a = 0; a < 4; ++a) b[a] = seed_base(P, i, j + a);
#pragma unroll
  for (uint32_t a = 0; a < 4; ++a) {
    const float xn = __builtin_fmaf(P.damp, z.v[a], b[a]);
    c[a] = d ? xn / (float)d : xn;
    if (live >> a & 1u) err[a] += (double)fabsf(xn - ppr_score(xo.v[a], df));
  }
  float* o = P.cout + cidx(P, i, j);
  if (live == 15u) {
    *reinterpret_cast<float4*>(o) = make_float4(c[0], c[1], c[2], c[3]);
  } else {  // converged vectors keep theirs
#pragma unroll
    for (uint32_t a = 0; a < 4; ++a)
      if (live >> a & 1u) o[a] = c[a];
  }
}

// per-vector sums over the workgroup's lane groups (G = T / 4 lanes each); vector q of the tile in
// thread q < T
template <int T>
__device__ __forceinline__ double slot_reduce(const double (&e)[4], double* lds /* 4*T */) {
  constexpr int G = T / 4;
  const uint32_t w = threadIdx.x / 64, l = threadIdx.x % 64;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    double v = e[q];
#pragma unroll
    for (int o = G; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
    if (l < (uint32_t)G) lds[w * T + l * 4 + q] = v;
  }
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x < (uint32_t)T)
    for (int q = 0; q < 4; ++q) r += lds[q * T + threadIdx.x];
  return r;
}

// What bounds it: the vector L1's misses.  Some 80 lines are in flight per CU at 510 cycles each (RMAT-22,
// k = 64: 142 M line reads, 72 M of them past the L2, 1.6 ms: 81 G lines/s, 9.3 TB/s into the L2s), whatever
// the tile, the wavefronts in flight or the L2's hit rate.  1.79 ms with one lane per float, rows of
// up to 256 in-edges on the row path and slices by the low bits of the source.
// kEven: the graph's rows are light up to kLightMaxWhole in-edges, which are added up kU at a time, then
// these sums (rows of 180, error against 64 bits with one running sum 2.0e-7, so 9.6e-8, in pieces of 32
// 8.7e-8).  Where light rows end at 32 it gains nothing and costs up to 9 % (RMAT-22, k = 64, 36.9 against 33.6 ms).
template <int T, int kR, bool kEven>
__global__ __launch_bounds__(kThreads) void ppr_sweep_kernel(PprParams P) {
  constexpr uint32_t G = T / 4;              // lanes per edge
  constexpr uint32_t kGroups = kThreads / G;
  constexpr uint32_t kU = G < 8 ? G : 8;     // gathers a lane has in flight on the row path
  __shared__ double red[4 * T];
  __shared__ float4 hub_red[kThreads];
  __shared__ uint32_t slot_of[kGroups];
  __shared__ uint32_t lives[2];
  // The k-tiles follow each other, so that the caches hold one tile's contributions at a time.
  // A tile's heavy workgroups come first: workgroup class c = b % 8 (its XCD: workgroup b runs on
  // XCD b % 8) serves source slice c, so that each XCD's L2 caches its eighth of the sources only.
  // Row workgroups follow.
  const uint32_t tile = blockIdx.x / P.tile_blocks;
  uint32_t b = blockIdx.x % P.tile_blocks, piece0 = 0;
  const bool heavy = b < P.heavy_blocks;
  if (!heavy) {
    b -= P.heavy_blocks;
    if (b >= P.row_blocks_run) return;
  } else {
    const uint32_t x = b % kSlices;
    piece0 = P.slice_off[x] + b / kSlices * kGroups;
    if (piece0 >= P.slice_off[x + 1]) return;
  }
  // the tile's vectors that are still solved
  if (threadIdx.x < 64) {
    const uint32_t j = tile * T + threadIdx.x;
    const unsigned long long m = __ballot(threadIdx.x < T && j < P.k && !vec_done(P, j));
    if (threadIdx.x == 0) {
      lives[0] = (uint32_t)m;
      lives[1] = (uint32_t)(m >> 32);
    }
  }
  __syncthreads();
  const uint64_t alive = ((uint64_t)lives[1] << 32) | lives[0];
  if (!alive) return;
  const uint32_t g = threadIdx.x / G, vl = threadIdx.x % G;
  const uint32_t j0 = tile * T + vl * 4;
  const uint32_t live = (uint32_t)(alive >> (vl * 4)) & 15u;
  const float* __restrict__ ctile = P.cin + (uint64_t)tile * P.n * T;
  // Sum of the contributions of the edges ids[p .. end), in edge order; c: the ids at p + vl, and
  // at the end those at end + vl (up to `last`).  kU gathers in flight, and the next ids with them.
  // Every lane gathers: lanes of converged vectors share their group's line, and past the end the last edge
  // is gathered again, whose line is there or under way (the next row's edges, gathered in its
  // place, were lines of their own: uniform random, 900,000 rows of 10, k = 64, 5.37 against 5.07 ms, 2 M,
  // k = 32, 6.21 against 5.89; RMAT-22, k = 64, 33.9 against 33.6).  Loads that a lane condition skipped made
  // the compiler drain every load in flight before each add.
  auto walk = [&](const uint32_t* __restrict__ ids, uint32_t p, uint32_t end, uint32_t last, uint32_t& c) {
    Four z{{0.f, 0.f, 0.f, 0.f}};
#pragma unroll 1
    while (p < end) {
      const uint32_t m = min(G, end - p);
      p += m;
      const uint32_t cn = p + vl < last ? ids[p + vl] : 0u;
#pragma unroll 1
      for (uint32_t q0 = 0; q0 < m; q0 += kU) {
        Four v[kU];
#pragma unroll
        for (uint32_t t = 0; t < kU; ++t)
          v[t] = load4(ctile + (uint64_t)(uint32_t)__shfl((int)c, (int)min(q0 + t, m - 1), (int)G) * T + vl * 4);
        if constexpr (kEven) {
          Four r{{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
          for (uint32_t t = 0; t < kU; ++t)
#pragma unroll
            for (int a = 0; a < 4; ++a) r.v[a] += q0 + t < m ? v[t].v[a] : 0.f;
#pragma unroll
          for (int a = 0; a < 4; ++a) z.v[a] += r.v[a];
        } else {
#pragma unroll
          for (uint32_t t = 0; t < kU; ++t)
#pragma unroll
            for (int a = 0; a < 4; ++a) z.v[a] += q0 + t < m ? v[t].v[a] : 0.f;
        }
      }
      c = cn;
    }
    return z;
  };
  if (!heavy) {
    // Light rows: each G-lane group takes kR consecutive rows, one after the other, over the compacted
    // light CSC (heavy rows are empty there)
    const uint32_t g0 = (b * kGroups + g) * kR;
    double e[4] = {0.0, 0.0, 0.0, 0.0};
    if (g0 < P.n) {
      uint32_t lp[kR + 1], rq[kR + 1], df[kR];
      Four xo[kR];
#pragma unroll
      for (uint32_t t = 0; t <= kR; ++t) {
        lp[t] = P.lrp[min(g0 + t, P.n)];
        rq[t] = P.rp[min(g0 + t, P.n)];
      }
      const uint32_t pend = lp[kR];
      uint32_t c = lp[0] + vl < pend ? P.lcol[lp[0] + vl] : 0u;
#pragma unroll
      for (uint32_t t = 0; t < kR; ++t) {
        const uint32_t i = min(g0 + t, P.n - 1);
        df[t] = P.degflag[i];
        xo[t] = load4(P.cin + cidx(P, i, j0));
      }
#pragma unroll
      for (uint32_t r = 0; r < kR; ++r) {
        const Four z = walk(P.lcol, lp[r], lp[r + 1], pend, c);
        if (g0 + r < P.n && rq[r + 1] - rq[r] <= P.light_max && live)  // heavy rows: the finishing launch
          ppr_update4(P, g0 + r, j0, z, df[r], xo[r], live, e);
      }
    }
    const double es = slot_reduce<T>(e, red);
    if (threadIdx.x < (uint32_t)T) P.blk_err[((uint64_t)tile * P.row_blocks + b) * T + threadIdx.x] = es;
  } else {
    // Heavy rows: lane group g takes piece piece0 + g (at most kPiece contiguous edges of one row and
    // slice) and adds its edges in order; the pieces of one row in this workgroup are added in order
    // and leave one partial
    const uint2 d = P.pieces[piece0 + g];
    const uint32_t m = P.pieces[piece0 + g + 1].x - d.x;  // 0 for a slice's padding
    uint32_t c = vl < m ? P.hcol[d.x + vl] : 0u;
    Four z = walk(P.hcol, d.x, d.x + m, d.x + m, c);
    hub_red[threadIdx.x] = make_float4(z.v[0], z.v[1], z.v[2], z.v[3]);
    if (vl == 0) slot_of[g] = m ? d.y : 0xFFFFFFFFu;
    __syncthreads();
    if (m && (g == 0 || slot_of[g - 1] != d.y)) {
      for (uint32_t h = g + 1; h < kGroups && slot_of[h] == d.y; ++h) {
        const float4 f = hub_red[h * G + vl];
        z.v[0] += f.x;
        z.v[1] += f.y;
        z.v[2] += f.z;
        z.v[3] += f.w;
      }
      if (j0 < P.k)
        *reinterpret_cast<float4*>(P.hub_part + (uint64_t)d.y * P.kq * 4 + j0) =
            make_float4(z.v[0], z.v[1], z.v[2], z.v[3]);
    }
  }
}

// finishing launch: heavy rows + fold of the per-workgroup, per-vector L1 partials.
// grid.x covers max(heavy rows * kq / kThreads, L1 partials / fold_rows).  One item (heavy row, four
// vectors) per thread: the longest rows' partials are a serial chain per item, and in degree order
// the first workgroups have all of them.  RMAT-22, k = 64: 97 us with one vector per item and eight
// items per thread.
template <int T>
__global__ __launch_bounds__(kThreads) void ppr_finish_kernel(PprParams P, uint32_t tiles) {
  __shared__ double red[kThreads];
  __shared__ unsigned long long errj[kFinMaxK];
  __shared__ uint8_t done[kFinMaxK];
  // part 1: heavy rows; their L1 changes are added per vector in LDS (fixed point: order
  // independent), then one atomic per vector
  const uint64_t items = (uint64_t)P.n_hub_rows * P.kq;
  const uint64_t t = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  const bool mine = t < items;
  uint32_t h = 0, j0 = 0, s0 = 0, s1 = 0, row = 0;
  if (mine) {
    if (items <= 0xFFFFFFFFull) {  // uniform over the launch: a 32-bit division is far cheaper
      h = (uint32_t)t / P.kq;
      j0 = ((uint32_t)t - h * P.kq) * 4;
    } else {
      h = (uint32_t)(t / P.kq);
      j0 = (uint32_t)(t % P.kq) * 4;
    }
    s0 = P.part_ptr[h];
    s1 = P.part_ptr[h + 1];
    row = P.hub_rows[h];
  }
  for (uint32_t q = threadIdx.x; q < kFinMaxK; q += kThreads) {
    errj[q] = 0ull;
    done[q] = q >= P.k || vec_done(P, q);
  }
  // the previous sweep's change: its sum for the host, and the next sweep's slot cleared
  if (P.iter > 0)
    for (uint32_t q = blockIdx.x * kThreads + threadIdx.x; q < P.k; q += gridDim.x * kThreads)
      P.acc[(uint64_t)(P.iter - 1) * P.k + q] = ppr_change(P.lanes, P.kpad, P.iter - 1, q);
  for (uint32_t q = blockIdx.x * kThreads + threadIdx.x; q < kErrLanes * P.kpad; q += gridDim.x * kThreads)
    P.lanes[(uint64_t)((P.iter + 1) % 3) * kErrLanes * P.kpad + q] = 0ull;
  unsigned long long* const lane = P.lanes + ((uint64_t)(P.iter % 3) * kErrLanes + blockIdx.x % kErrLanes) * P.kpad;
  __syncthreads();
  auto vdone = [&](uint32_t j) { return j < kFinMaxK ? done[j] != 0 : j >= P.k || vec_done(P, j); };
  auto add_err = [&](uint32_t j, double e) {
    if (j < kFinMaxK) atomicAdd(&errj[j], err_to_fixed(e));
    else atomicAdd(lane + j, err_to_fixed(e));
  };
  uint32_t live = 0;
  if (mine)
    for (uint32_t a = 0; a < 4; ++a) live |= vdone(j0 + a) ? 0u : 1u << a;
  if (live) {
    const uint32_t df = P.degflag[row];
    const Four xo = load4(P.cin + cidx(P, row, j0));
    // partials added in order, kFinU loads in flight
    Four z{{0.f, 0.f, 0.f, 0.f}};
    for (uint32_t s = s0; s < s1; s += kFinU) {
      Four v[kFinU];
#pragma unroll
      for (uint32_t r = 0; r < kFinU; ++r) v[r] = load4(P.hub_part + ((uint64_t)min(s + r, s1 - 1) * P.kq * 4 + j0));
#pragma unroll
      for (uint32_t r = 0; r < kFinU; ++r)
#pragma unroll
        for (int a = 0; a < 4; ++a) z.v[a] += s + r < s1 ? v[r].v[a] : 0.f;
    }
    double e[4] = {0.0, 0.0, 0.0, 0.0};
    ppr_update4(P, row, j0, z, df, xo, live, e);
#pragma unroll
    for (uint32_t a = 0; a < 4; ++a)
      if (e[a] > 0.0) add_err(j0 + a, e[a]);
  }
  // part 2: fold blk_err rows; this workgroup folds fold_rows workgroup rows of every tile
  const uint64_t r0 = (uint64_t)blockIdx.x * P.fold_rows;
  const uint64_t rows_total = min((uint64_t)P.row_blocks_run, r0 + P.fold_rows);
  for (uint32_t tl = 0; tl < tiles && r0 < rows_total; ++tl) {
    const uint32_t vl = threadIdx.x % T;
    const uint32_t slot = threadIdx.x / T;  // kThreads/T slots stride over the rows
    constexpr uint32_t kS = kThreads / T, kPer = (kFoldRows + kS - 1) / kS;
    double a[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
      const uint64_t r = r0 + slot + (uint64_t)q * kS;
      if (r < rows_total) a[q & 3] += P.blk_err[((uint64_t)tl * P.row_blocks + r) * T + vl];
    }
    red[threadIdx.x] = (a[0] + a[1]) + (a[2] + a[3]);
    __syncthreads();
    if (threadIdx.x < (uint32_t)T) {
      double sum = 0.0;
      for (uint32_t q = 0; q < kThreads / T; ++q) sum += red[q * T + threadIdx.x];
      const uint32_t jj = tl * T + threadIdx.x;
      if (jj < P.k && sum > 0.0 && !vdone(jj)) add_err(jj, sum);
    }
    __syncthreads();
  }
  __syncthreads();
  for (uint32_t q = threadIdx.x; q < kFinMaxK && q < P.k; q += kThreads)
    if (errj[q]) atomicAdd(lane + q, errj[q]);
}

// c0 = init / outdeg (init itself for a row without out-edges) for every vector of a tile, in the
// tile-major layout: blockIdx.y is the k-tile, and x runs over its n x T floats four by four (T is a
// multiple of 4; lanes past k are written and never read).
__global__ __launch_bounds__(kThreads) void ppr_init_kernel(uint32_t n, uint32_t kt_shift,
                                                            const uint32_t* __restrict__ deg, float init,
                                                            float4* __restrict__ c0) {
  const uint64_t q = (uint64_t)blockIdx.x * kThreads + threadIdx.x;  // offset inside the tile, in fours
  const uint32_t i = (uint32_t)(q >> (kt_shift - 2));
  if (i < n && (q >> (kt_shift - 2)) < n) {
    const uint32_t d = deg[i];
    const float c = d ? init / (float)d : init;
    c0[(((uint64_t)blockIdx.y * n << kt_shift) >> 2) + q] = make_float4(c, c, c, c);
  }
}

__global__ __launch_bounds__(kThreads) void ppr_zero_acc_kernel(unsigned long long* __restrict__ acc, uint64_t m) {
  const uint64_t t = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  if (t < m) acc[t] = 0ull;
}

// out[i] = deg[i] | kSeedFlag when row i appears in the sorted seed rows (binary search,
// so no two threads ever write the same entry)
__global__ __launch_bounds__(kThreads) void ppr_degflag_kernel(uint32_t n, const uint32_t* __restrict__ deg,
                                                               const uint32_t* __restrict__ seed_row, uint32_t ns,
                                                               uint32_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  uint32_t lo = 0, hi = ns;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (seed_row[mid] < i) lo = mid + 1;
    else hi = mid;
  }
  out[i] = deg[i] | ((lo < ns && seed_row[lo] == i) ? kSeedFlag : 0u);
}

__global__ __launch_bounds__(kThreads) void gather_u32_kernel(uint32_t m, const uint32_t* __restrict__ idx,
                                                              const uint32_t* __restrict__ table,
                                                              uint32_t* __restrict__ out) {
  const uint32_t q = blockIdx.x * kThreads + threadIdx.x;
  if (q < m) out[q] = table[idx[q]];
}

// sweeps vector j executed: the first t with acc[t][j] below the threshold, plus one (or all); the last
// sweep's change is still in its lanes
__global__ __launch_bounds__(kThreads) void ppr_its_kernel(uint32_t k, const unsigned long long* __restrict__ lanes,
                                                           uint32_t kpad, unsigned long long* __restrict__ acc,
                                                           uint64_t iters, double threshold,
                                                           uint32_t* __restrict__ its) {
  const uint32_t j = blockIdx.x * kThreads + threadIdx.x;
  if (j >= k) return;
  if (iters) acc[(iters - 1) * k + j] = ppr_change(lanes, kpad, (uint32_t)(iters - 1), j);
  uint64_t n_it = iters;
  for (uint64_t q = 0; q < iters; ++q)
    if (fixed_to_err(acc[q * k + j]) < threshold) {
      n_it = q + 1;
      break;
    }
  its[j] = (uint32_t)n_it;
}

// Final scores from the contributions: vector j's last sweep t = its[j] - 1 wrote c0 when t
// is odd, c1 when even (c0 before any sweep).  With a relabelled solve row r is original
// vertex order[r].
__global__ __launch_bounds__(kThreads) void ppr_scores_kernel(uint32_t n, uint32_t k, uint32_t kt_shift,
                                                              const uint32_t* __restrict__ order,
                                                              const uint32_t* __restrict__ degflag,
                                                              const float* __restrict__ c0,
                                                              const float* __restrict__ c1,
                                                              const uint32_t* __restrict__ its,
                                                              float* __restrict__ out) {
  const uint64_t t = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  const uint64_t nk = (uint64_t)n * k;
  if (t >= nk) return;
  uint32_t r, j;
  if (nk <= 0xFFFFFFFFull) {  // uniform over the launch: a 32-bit division is far cheaper
    const uint32_t t32 = (uint32_t)t;
    r = t32 / k;
    j = t32 - r * k;
  } else {
    r = (uint32_t)(t / k);
    j = (uint32_t)(t % k);
  }
  const uint32_t nj = its[j];
  const float* c = nj == 0 ? c0 : ((nj - 1) & 1) ? c0 : c1;
  const float v = c[(((uint64_t)(j >> kt_shift) * n + r) << kt_shift) + (j & ((1u << kt_shift) - 1))];
  out[(uint64_t)(order ? order[r] : r) * k + j] = ppr_score(v, degflag[r]);
}

// The same four vectors at a time, for k a multiple of 4 and 16-byte aligned scores (a wave then has
// 1 KB of them under way instead of 256 bytes: RMAT-22, k = 64: 0.93 to 0.41 ms).
__global__ __launch_bounds__(kThreads) void ppr_scores4_kernel(uint32_t n, uint32_t k4, uint32_t kt_shift,
                                                               const uint32_t* __restrict__ order,
                                                               const uint32_t* __restrict__ degflag,
                                                               const float4* __restrict__ c0,
                                                               const float4* __restrict__ c1,
                                                               const uint4* __restrict__ its,
                                                               float4* __restrict__ out) {
  const uint64_t t = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  const uint64_t nk = (uint64_t)n * k4;
  if (t >= nk) return;
  uint32_t r, j4;
  if (nk <= 0xFFFFFFFFull) {
    const uint32_t t32 = (uint32_t)t;
    r = t32 / k4;
    j4 = t32 - r * k4;
  } else {
    r = (uint32_t)(t / k4);
    j4 = (uint32_t)(t % k4);
  }
  const uint4 it = its[j4];
  auto in_c0 = [](uint32_t nj) { return nj == 0 || ((nj - 1) & 1); };
  const bool b[4] = {in_c0(it.x), in_c0(it.y), in_c0(it.z), in_c0(it.w)};
  const uint32_t ts = kt_shift - 2;
  const uint64_t at = (((uint64_t)(j4 >> ts) * n + r) << ts) + (j4 & ((1u << ts) - 1));
  const bool any0 = b[0] || b[1] || b[2] || b[3], all0 = b[0] && b[1] && b[2] && b[3];
  float4 v0, v1;
  if (any0) v0 = c0[at];
  if (!all0) v1 = c1[at];
  const uint32_t df = degflag[r];
  float4 o;
  o.x = ppr_score(b[0] ? v0.x : v1.x, df);
  o.y = ppr_score(b[1] ? v0.y : v1.y, df);
  o.z = ppr_score(b[2] ? v0.z : v1.z, df);
  o.w = ppr_score(b[3] ? v0.w : v1.w, df);
  out[(uint64_t)(order ? order[r] : r) * k4 + j4] = o;
}

inline uint32_t grid1(uint64_t m) { return (uint32_t)ceil_div(m ? m : 1, kThreads); }

__global__ __launch_bounds__(kThreads) void heavy_deg_kernel(uint32_t nh, const uint32_t* __restrict__ rows,
                                                             const uint32_t* __restrict__ rp,
                                                             uint32_t* __restrict__ deg) {
  const uint32_t h = blockIdx.x * kThreads + threadIdx.x;
  if (h < nh) deg[h] = rp[rows[h] + 1] - rp[rows[h]];
}

// heavy edge e (row h's edges at hoff[h] ..): key (slice, h), payload the source.  A row
// of at least big edges is split by source slice; a shorter one keeps its edges together
// in slice h mod nsl (pieces of its own would be mostly empty).
__global__ __launch_bounds__(kThreads) void heavy_key_kernel(uint64_t eh, uint32_t nh,
                                                             const uint32_t* __restrict__ hoff,
                                                             const uint32_t* __restrict__ rows,
                                                             const uint32_t* __restrict__ rp,
                                                             const uint32_t* __restrict__ col, uint32_t sh,
                                                             uint32_t nsl, uint32_t big,
                                                             uint64_t* __restrict__ keys,
                                                             uint32_t* __restrict__ vals) {
  const uint64_t e = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  if (e >= eh) return;
  uint32_t lo = 0, hi = nh - 1;  // last h with hoff[h] <= e
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (hoff[mid] <= e) lo = mid;
    else hi = mid - 1;
  }
  const uint32_t u = col[rp[rows[lo]] + (uint32_t)(e - hoff[lo])];
  const uint32_t x = hoff[lo + 1] - hoff[lo] >= big ? ((u >> sh) * 0x9E3779B1u >> 29) % nsl : lo % nsl;
  keys[e] = (uint64_t)x * nh + lo;
  vals[e] = u;
}

// gp[t] = first sorted position with key >= t, t in [0, ng]
__global__ __launch_bounds__(kThreads) void group_ptr_kernel(uint64_t eh, const uint64_t* __restrict__ keys,
                                                             uint64_t ng, uint32_t* __restrict__ gp) {
  const uint64_t t = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  if (t > ng) return;
  uint64_t lo = 0, hi = eh;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (keys[mid] < t) lo = mid + 1;
    else hi = mid;
  }
  gp[t] = (uint32_t)lo;
}

// group t = (slice x, heavy row h) of edges [gp[t], gp[t + 1]): its pieces
__global__ __launch_bounds__(kThreads) void piece_count_kernel(uint32_t ng, const uint32_t* __restrict__ gp,
                                                               uint32_t* __restrict__ cnt) {
  const uint32_t t = blockIdx.x * kThreads + threadIdx.x;
  if (t < ng) cnt[t] = (gp[t + 1] - gp[t] + kPiece - 1) / kPiece;
}

struct SliceOff {
  uint32_t at[kSlices + 1];    // first piece of each slice, a multiple of the groups in a workgroup
  uint32_t scan[kSlices + 1];  // and pieces of the slices before it, without padding
};

// first piece of group t of slice x
__device__ __forceinline__ uint32_t piece_at(const SliceOff& so, uint32_t x, uint32_t po) {
  return so.at[x] + (po - so.scan[x]);
}

// partials of group (x, h): one per workgroup that its pieces lie in, row by row
__global__ __launch_bounds__(kThreads) void part_count_kernel(uint32_t nh, uint32_t nsl, uint32_t groups,
                                                              const uint32_t* __restrict__ po, SliceOff so,
                                                              uint32_t* __restrict__ cnt) {
  const uint32_t q = blockIdx.x * kThreads + threadIdx.x;
  if (q >= nh * nsl) return;
  const uint32_t h = q / nsl, x = q % nsl, t = x * nh + h;
  const uint32_t c = po[t + 1] - po[t], a = piece_at(so, x, po[t]);
  cnt[q] = c ? (a + c - 1) / groups - a / groups + 1 : 0u;
}

__global__ __launch_bounds__(kThreads) void piece_fill_kernel(uint32_t nh, uint32_t nsl, uint32_t groups,
                                                              const uint32_t* __restrict__ po,
                                                              const uint32_t* __restrict__ gp,
                                                              const uint32_t* __restrict__ part, SliceOff so,
                                                              uint2* __restrict__ pieces) {
  const uint32_t q = blockIdx.x * kThreads + threadIdx.x;
  if (q >= nh * nsl) return;
  const uint32_t h = q / nsl, x = q % nsl, t = x * nh + h;
  const uint32_t c = po[t + 1] - po[t], a = piece_at(so, x, po[t]);
  for (uint32_t i = 0; i < c; ++i)
    pieces[a + i] = make_uint2(gp[t] + i * kPiece, part[q] + (a + i) / groups - a / groups);
  if (h == nh - 1) {  // the padding after the slice, and the end
    for (uint32_t p = a + c; p < so.at[x + 1]; ++p) pieces[p] = make_uint2(gp[t + 1], 0u);
    if (x == nsl - 1) pieces[so.at[nsl]] = make_uint2(gp[t + 1], 0u);
  }
}

// heavy row h's first partial
__global__ __launch_bounds__(kThreads) void part_ptr_kernel(uint32_t nh, uint32_t nsl,
                                                            const uint32_t* __restrict__ part,
                                                            uint32_t* __restrict__ ptr) {
  const uint32_t h = blockIdx.x * kThreads + threadIdx.x;
  if (h <= nh) ptr[h] = part[(uint64_t)h * nsl];
}

// light CSC: row i keeps its in-edges when in-degree <= light_max, else none
__global__ __launch_bounds__(kThreads) void light_len_kernel(uint32_t n, const uint32_t* __restrict__ rp,
                                                             uint32_t light_max, uint32_t* __restrict__ len) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n) {
    const uint32_t d = rp[i + 1] - rp[i];
    len[i] = d <= light_max ? d : 0u;
  }
}

// out[0] = one past the last row with in-edges, out[1] = most in-edges of a row.  One atomic each per workgroup.
__global__ __launch_bounds__(kThreads) void row_stats_kernel(uint32_t n, const uint32_t* __restrict__ rp,
                                                             uint32_t* __restrict__ out) {
  __shared__ uint32_t ends[kThreads / 64], mosts[kThreads / 64];
  uint32_t end = 0, most = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kThreads) {
    const uint32_t d = rp[i + 1] - rp[i];
    if (d) end = (uint32_t)i + 1;
    most = max(most, d);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    end = max(end, (uint32_t)__shfl_xor((int)end, o, 64));
    most = max(most, (uint32_t)__shfl_xor((int)most, o, 64));
  }
  if (lane_id() == 0) {
    ends[threadIdx.x / 64] = end;
    mosts[threadIdx.x / 64] = most;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicMax(out, max(max(ends[0], ends[1]), max(ends[2], ends[3])));
    atomicMax(out + 1, max(max(mosts[0], mosts[1]), max(mosts[2], mosts[3])));
  }
}

__global__ __launch_bounds__(kThreads) void light_copy_kernel(uint32_t n, const uint32_t* __restrict__ rp,
                                                              const uint32_t* __restrict__ col,
                                                              const uint32_t* __restrict__ lrp,
                                                              uint32_t* __restrict__ lcol) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const uint32_t d = lrp[i + 1] - lrp[i];
  for (uint32_t t = 0; t < d; ++t) lcol[lrp[i] + t] = col[rp[i] + t];
}

}  // namespace

// Heavy rows (in-degree >= min_deg): their in-edges regrouped by (source slice, row), the
// slice of source u being a hash of u >> sh with sh chosen so that the T-float
// contributions of one 128-byte line fall in one slice (rows of fewer than big edges
// stay whole, in slice h mod nsl).  A hash: with the lowest bits an XCD's lines would lie in some
// of its L2's channels only (RMAT-22, T = 32: 2.08 ms a sweep against 1.84).  The rows are then cut into
// pieces of at most kPiece edges, in workgroups of 1024 / tile pieces of one slice.
static void build_heavy_slices(hipStream_t s, const ActiveCsc& a, uint32_t n, uint32_t min_deg, uint32_t big,
                               uint32_t tile, uint32_t nsl, PprState& st) {
  DevBuf<uint32_t> unused_ptr, unused_row;
  uint32_t nh = 0, ns0 = 0;
  build_segments(s, a.ptr, n, min_deg, 1u << 30, st.heavy_rows, unused_ptr, unused_row, &nh, &ns0);
  const uint32_t sh = tile >= 32 ? 0u : tile == 16 ? 1u : 2u;
  const uint32_t groups = kThreads / (tile / 4);
  st.slice_off.assign(kSlices + 1, 0);
  st.n_heavy = nh;
  st.n_parts = 0;
  if (nh == 0) return;
  DevBuf<uint32_t> deg(nh), hoff((uint64_t)nh + 1);
  heavy_deg_kernel<<<grid1(nh), kThreads, 0, s>>>(nh, st.heavy_rows.p, a.ptr, deg.p);
  NWG_LAUNCH_CHECK();
  exclusive_scan_u32(s, deg.p, hoff.p, nh);
  uint32_t eh = 0;
  NWG_HIP(hipMemcpyAsync(&eh, hoff.p + nh, 4, hipMemcpyDeviceToHost, s));
  NWG_HIP(hipStreamSynchronize(s));
  st.hcol.alloc(eh);
  const uint32_t ng = nh * nsl;  // below 2^32: a heavy row has more in-edges than there are slices
  DevBuf<uint32_t> gp((uint64_t)ng + 1);
  {
    DevBuf<uint64_t> keys(eh), keys_tmp(eh);
    DevBuf<uint32_t> vals_tmp(eh);
    heavy_key_kernel<<<grid1(eh), kThreads, 0, s>>>(eh, nh, hoff.p, st.heavy_rows.p, a.ptr, a.idx, sh, nsl, big,
                                                    keys.p, st.hcol.p);
    NWG_LAUNCH_CHECK();
    int kb = 1;
    while (kb < 64 && (1ull << kb) < ng) ++kb;
    radix_sort_pairs(s, keys, keys_tmp, &st.hcol, &vals_tmp, eh, 0, kb);  // stable: sources stay ascending
    group_ptr_kernel<<<grid1((uint64_t)ng + 1), kThreads, 0, s>>>(eh, keys.p, ng, gp.p);
    NWG_LAUNCH_CHECK();
  }
  DevBuf<uint32_t> cnt(ng), po((uint64_t)ng + 1), part((uint64_t)ng + 1);
  piece_count_kernel<<<grid1(ng), kThreads, 0, s>>>(ng, gp.p, cnt.p);
  NWG_LAUNCH_CHECK();
  exclusive_scan_u32(s, cnt.p, po.p, ng);
  SliceOff so{};
  for (uint32_t x = 0; x <= nsl; ++x)
    NWG_HIP(hipMemcpyAsync(&so.scan[x], po.p + (uint64_t)x * nh, 4, hipMemcpyDeviceToHost, s));
  NWG_HIP(hipStreamSynchronize(s));
  for (uint32_t x = 0; x < nsl; ++x)
    so.at[x + 1] = so.at[x] + (uint32_t)ceil_div(so.scan[x + 1] - so.scan[x], groups) * groups;
  part_count_kernel<<<grid1(ng), kThreads, 0, s>>>(nh, nsl, groups, po.p, so, cnt.p);
  NWG_LAUNCH_CHECK();
  exclusive_scan_u32(s, cnt.p, part.p, ng);
  NWG_HIP(hipMemcpyAsync(&st.n_parts, part.p + ng, 4, hipMemcpyDeviceToHost, s));
  st.pieces.alloc((uint64_t)so.at[nsl] + 1);
  piece_fill_kernel<<<grid1(ng), kThreads, 0, s>>>(nh, nsl, groups, po.p, gp.p, part.p, so, st.pieces.p);
  NWG_LAUNCH_CHECK();
  st.part_ptr.alloc((uint64_t)nh + 1);
  part_ptr_kernel<<<grid1((uint64_t)nh + 1), kThreads, 0, s>>>(nh, nsl, part.p, st.part_ptr.p);
  NWG_LAUNCH_CHECK();
  NWG_HIP(hipStreamSynchronize(s));
  for (uint32_t x = 0; x <= nsl; ++x) st.slice_off[x] = so.at[x];
}

// The split of the rows between the two paths.  Rows of more than kLightMax in-edges are cut into pieces
// over the source slices.  Measured on MI355X (20 sweeps, ms; cut 16 / 32 / 64 / 256): RMAT 2^12 with k = 10
// 0.56 / 0.60 / 0.71 / 1.1, uniform random 20,000 with k = 33 0.77 / 0.60 / 0.60 / 0.60, RMAT-20 with k = 10
// 5.8 / 5.8 / 6.5 / 13.3 and with k = 64 7.4 / 8.0 / 9.2 / 12.5, RMAT-22 in degree order with k = 64 35.1 /
// 34.7 / 34.2 / 34.8: a lane group walks its rows in rounds of 8 gathers, and the longest light row
// decides where the graph is small or not in degree order.  Where no row stands out (most in-edges at
// most 64 + 8 times the average) light rows go up to kLightMaxWhole: the pieces would be nearly all rows
// (uniform random, ms with the cut at 32 / 256: 200,000 rows of 40, k = 64, 3.08 / 2.52, 100,000 of 200, k = 32,
// 1.96 / 1.67, 900,000 of 20, k = 40, 6.80 / 6.71, 20,000 of 16, k = 33, 0.39 / 0.37) -- but for tiles of 8,
// where a light row is two lanes' (50,000 of 100, k = 8, 0.38 / 0.40).
// Rows of fewer than kSplitMin in-edges stay in one slice (64 / 128 / 256: RMAT-20, k = 10, 5.8 / 6.5 / 8.3; all
// rows whole 10).  Denser graphs split longer rows only, so that the partial vectors take no more
// than some three times a contribution array, and a solve whose partials would take more than
// kPartBytes keeps rows whole and light up to kLightMaxWhole (at most one partial per such row and 512
// edges).
constexpr uint32_t kLightMax = 32, kLightMaxWhole = 256;
constexpr uint32_t kSplitMin = 64;
constexpr uint64_t kPartBytes = 16ull << 30;

static void build_rows(hipStream_t s, const ActiveCsc& a, uint32_t n, uint64_t nnz, uint32_t tile, bool whole,
                       PprState& st) {
  const uint32_t light_max = whole || st.even ? kLightMaxWhole : kLightMax;
  const uint32_t big = whole ? ~0u : (uint32_t)std::max<uint64_t>(kSplitMin, 4 * nnz / n);
  build_heavy_slices(s, a, n, light_max + 1, big, tile, kSlices, st);
  DevBuf<uint32_t> len(n);
  st.lrp.alloc((uint64_t)n + 1);
  light_len_kernel<<<grid1(n), kThreads, 0, s>>>(n, a.ptr, light_max, len.p);
  NWG_LAUNCH_CHECK();
  exclusive_scan_u32(s, len.p, st.lrp.p, n);
  uint32_t n_light = 0;
  NWG_HIP(hipMemcpyAsync(&n_light, st.lrp.p + n, 4, hipMemcpyDeviceToHost, s));
  NWG_HIP(hipStreamSynchronize(s));
  st.lcol.alloc(std::max<uint32_t>(n_light, 1));
  light_copy_kernel<<<grid1(n), kThreads, 0, s>>>(n, a.ptr, a.idx, st.lrp.p, st.lcol.p);
  NWG_LAUNCH_CHECK();
  NWG_HIP(hipStreamSynchronize(s));
  st.whole = whole;
  st.light_max = light_max;
}

// A lane group's light rows: 4 (their ids and old contributions loaded ahead) once that leaves the
// chip its 8192 wavefronts four times over, else 1.  RMAT-22, k = 64: 36.6 ms against 37.9 with 1; uniform
// random 300,000 with k = 24 (37,500 wavefronts with 1): 1.95 against 1.67.
constexpr uint64_t kFourRowWaves = 32768;

// Host driver; tile = k-tile width (8, 16, 32 or 64).
void ppr_run(nwg_ctx* ctx, nwg_graph* g, uint32_t k, const std::vector<uint32_t>& seed_ptr,
             const std::vector<uint32_t>& seeds, float damping, float threshold, uint64_t max_iters, uint32_t tile,
             float* scores_dev, uint64_t* iterations, nwg_pr_info* info) {
  hipStream_t s = ctx->stream;
  const uint32_t n = g->n;
  NWG_REQUIRE(k >= 1, "k must be >= 1");
  NWG_REQUIRE(tile == 8 || tile == 16 || tile == 32 || tile == 64, "k-tile must be 8, 16, 32 or 64");
  NWG_REQUIRE(max_iters < (1ull << 31), "max_iters too large");
  if (!g->plan.built) plan_build(s, g, default_plan_params());
  const Plan& pl = g->plan;
  const ActiveCsc a = g->active(pl.params.relabel != 0);
  if (!g->ppr) g->ppr.reset(new PprState());
  PprState& st = *g->ppr;
  const uint32_t kq = (uint32_t)ceil_div(k, 4);
  if (st.seg_version != g->plan_version || st.seg_tile != tile) {
    st.seg_version = 0;
    DevBuf<uint32_t> stats(2);
    uint32_t h[2] = {0, 0};
    NWG_HIP(hipMemsetAsync(stats.p, 0, 8, s));
    row_stats_kernel<<<std::min(grid1(n), 512u), kThreads, 0, s>>>(n, a.ptr, stats.p);
    NWG_LAUNCH_CHECK();
    NWG_HIP(hipMemcpyAsync(h, stats.p, 8, hipMemcpyDeviceToHost, s));
    NWG_HIP(hipStreamSynchronize(s));
    st.row_end = h[0];
    st.even = tile >= 16 && (double)h[1] <= 64.0 + 8.0 * (double)g->nnz / n;
    build_rows(s, a, n, g->nnz, tile, false, st);
    st.n_parts_split = st.n_parts;
    st.seg_version = g->plan_version;
    st.seg_tile = tile;
  }
  const bool whole = (uint64_t)st.n_parts_split * kq * 16 > kPartBytes;
  if (whole != st.whole) {
    st.seg_version = 0;
    build_rows(s, a, n, g->nnz, tile, whole, st);
    st.seg_version = g->plan_version;
  }
  const uint32_t n_heavy = st.n_heavy;
  // seed entries sorted by (row, vector); rows in the active numbering
  std::vector<std::pair<uint32_t, uint32_t>> ent;
  std::vector<float> ebase;
  for (uint32_t j = 0; j < k; ++j) {
    const uint32_t c = seed_ptr[j + 1] - seed_ptr[j];
    NWG_REQUIRE(c >= 1, "every teleport vector needs at least one seed");
    for (uint32_t q = seed_ptr[j]; q < seed_ptr[j + 1]; ++q) {
      NWG_REQUIRE(seeds[q] < n, "seed id >= n");
      ent.emplace_back(seeds[q], j);
    }
  }
  std::sort(ent.begin(), ent.end());
  for (size_t q = 1; q < ent.size(); ++q) NWG_REQUIRE(ent[q] != ent[q - 1], "duplicate seed in a teleport vector");
  const uint32_t ns = (uint32_t)ent.size();
  if (a.order) {  // map seed ids through rank (original -> relabelled) and re-sort
    std::vector<uint32_t> ids(ns);
    for (uint32_t q = 0; q < ns; ++q) ids[q] = ent[q].first;
    st.ids.ensure(ns);
    st.ids_new.ensure(ns);
    NWG_HIP(hipMemcpyAsync(st.ids.p, ids.data(), ns * 4ull, hipMemcpyHostToDevice, s));
    gather_u32_kernel<<<grid1(ns), kThreads, 0, s>>>(ns, st.ids.p, g->rl->rank.p, st.ids_new.p);
    NWG_LAUNCH_CHECK();
    NWG_HIP(hipMemcpyAsync(ids.data(), st.ids_new.p, ns * 4ull, hipMemcpyDeviceToHost, s));
    NWG_HIP(hipStreamSynchronize(s));
    for (uint32_t q = 0; q < ns; ++q) ent[q].first = ids[q];
    std::sort(ent.begin(), ent.end());
  }
  std::vector<uint32_t> erow(ns), evec(ns);
  ebase.resize(ns);
  for (size_t q = 0; q < ns; ++q) {
    erow[q] = ent[q].first;
    evec[q] = ent[q].second;
    const uint32_t c = seed_ptr[ent[q].second + 1] - seed_ptr[ent[q].second];
    const float v = 1.0f / (float)c;                                  // teleport value v_j[row]
    ebase[q] = (float)((1.0 - (double)damping) * (double)v);          // same rounding as the plain path
  }
  st.seed_row.ensure(ns);
  st.seed_vec.ensure(ns);
  st.seed_base.ensure(ns);
  st.degflag.ensure(n);
  NWG_HIP(hipMemcpyAsync(st.seed_row.p, erow.data(), ns * 4ull, hipMemcpyHostToDevice, s));
  NWG_HIP(hipMemcpyAsync(st.seed_vec.p, evec.data(), ns * 4ull, hipMemcpyHostToDevice, s));
  NWG_HIP(hipMemcpyAsync(st.seed_base.p, ebase.data(), ns * 4ull, hipMemcpyHostToDevice, s));
  ppr_degflag_kernel<<<grid1(n), kThreads, 0, s>>>(n, a.deg, st.seed_row.p, ns, st.degflag.p);
  NWG_LAUNCH_CHECK();

  const uint32_t tiles = (uint32_t)ceil_div(k, tile);
  const uint32_t kr = (uint64_t)n * tiles * tile / 1024 >= kFourRowWaves ? 4 : 1;
  const uint32_t rows_per_block = kThreads / (tile / 4) * kr;
  const uint32_t row_blocks = (uint32_t)ceil_div(n, rows_per_block);
  const uint64_t nk = (uint64_t)n * k;
  const uint64_t nc = (uint64_t)tiles * n * tile;  // tile-major contributions, last tile padded
  st.c0.ensure(nc);
  st.c1.ensure(nc);
  st.hub_part.ensure((uint64_t)std::max<uint32_t>(st.n_parts, 1) * kq * 4);
  st.blk_err.ensure((uint64_t)row_blocks * tiles * tile);
  st.acc.ensure(std::max<uint64_t>(max_iters, 1) * k);
  const uint32_t kpad = (uint32_t)ceil_div(k, 16) * 16;
  const uint64_t lane_words = 3ull * kErrLanes * kpad;
  st.lanes.ensure(lane_words);
  float* const c0p = st.c0.p;
  float* const c1p = st.c1.p;

  PprParams P{};
  P.rp = a.ptr;
  P.lrp = st.lrp.p;
  P.lcol = st.lcol.p;
  P.degflag = st.degflag.p;
  P.seed_row = st.seed_row.p;
  P.seed_vec = st.seed_vec.p;
  P.seed_base = st.seed_base.p;
  P.n_seed = ns;
  P.n = n;
  P.k = k;
  P.tiles = tiles;
  P.kt_shift = (uint32_t)__builtin_ctz(tile);
  P.damp = damping;
  P.light_max = st.light_max;
  P.row_blocks = row_blocks;
  P.n_hub_rows = n_heavy;
  P.hub_rows = st.heavy_rows.p;
  P.part_ptr = st.part_ptr.p;
  P.hub_part = st.hub_part.p;
  P.blk_err = st.blk_err.p;
  P.acc = st.acc.p;
  P.threshold = (double)threshold;
  P.hcol = st.hcol.p;
  P.pieces = st.pieces.p;
  P.lanes = st.lanes.p;
  P.kpad = kpad;
  P.kq = kq;
  uint32_t max_slice = 0;
  for (uint32_t x = 0; x <= kSlices; ++x) P.slice_off[x] = st.slice_off[x];
  for (uint32_t x = 0; x < kSlices; ++x) max_slice = std::max(max_slice, st.slice_off[x + 1] - st.slice_off[x]);
  const uint32_t slice_blocks = max_slice / (kThreads / (tile / 4));
  P.heavy_blocks = slice_blocks * kSlices;
  // Rows without in-edges reach their fixed point (1-d) v_j in one sweep and hold it, and the
  // next sweep writes the same contribution into the other buffer: from the third sweep on
  // only the row workgroups up to the last row with in-edges run (degree ordering puts
  // every row without in-edges last, half of RMAT-22's rows).
  const uint32_t live_row_blocks = (uint32_t)std::min<uint64_t>(ceil_div(st.row_end, rows_per_block), row_blocks);

  const float init = (float)(1.0 / n);
  NWG_HIP(hipEventRecord(ctx->ev0, s));
  {
    const uint64_t per_tile = (uint64_t)n << P.kt_shift;
    NWG_REQUIRE(ceil_div(per_tile, kThreads) < (1ull << 31) && P.tiles < 65536u, "batched solve too large for one launch");
    ppr_init_kernel<<<dim3((uint32_t)ceil_div(per_tile / 4, kThreads), P.tiles), kThreads, 0, s>>>(
        n, P.kt_shift, a.deg, init, reinterpret_cast<float4*>(c0p));
  }
  NWG_LAUNCH_CHECK();
  ppr_zero_acc_kernel<<<grid1(lane_words), kThreads, 0, s>>>(st.lanes.p, lane_words);
  NWG_LAUNCH_CHECK();
  const uint64_t grid64 = ((uint64_t)P.heavy_blocks + ceil_div(row_blocks, 8) * 8) * tiles;
  NWG_REQUIRE(grid64 < (1ull << 31), "batched solve too large for one launch");
  const uint64_t fin_a = ceil_div((uint64_t)n_heavy * kq, kThreads), fin_b = ceil_div(row_blocks, kFoldRows);
  const uint32_t fin = (uint32_t)std::max<uint64_t>(std::max(fin_a, fin_b), 1);
  NWG_REQUIRE(std::max(fin_a, fin_b) < (1ull << 31), "batched solve too large for one launch");
  P.fold_rows = std::min<uint32_t>(kFoldRows, std::max<uint32_t>((uint32_t)ceil_div(row_blocks, fin), 1));
  for (uint64_t it = 0; it < max_iters; ++it) {
    P.iter = (uint32_t)it;
    P.cin = (it & 1) ? c1p : c0p;
    P.cout = (it & 1) ? c0p : c1p;
    P.row_blocks_run = it >= 2 ? live_row_blocks : row_blocks;
    P.tile_blocks = P.heavy_blocks + (uint32_t)ceil_div(P.row_blocks_run, 8) * 8;
    const uint32_t grid = P.tile_blocks * tiles;  // 0 only for a graph without edges
    auto sweep = [&](auto t) {
      constexpr int T = decltype(t)::value;
      if (grid && !st.even && kr == 4) ppr_sweep_kernel<T, 4, false><<<grid, kThreads, 0, s>>>(P);
      else if (grid && !st.even) ppr_sweep_kernel<T, 1, false><<<grid, kThreads, 0, s>>>(P);
      else if (grid && kr == 4) ppr_sweep_kernel<T, 4, true><<<grid, kThreads, 0, s>>>(P);
      else if (grid) ppr_sweep_kernel<T, 1, true><<<grid, kThreads, 0, s>>>(P);
      ppr_finish_kernel<T><<<fin, kThreads, 0, s>>>(P, tiles);
    };
    if (tile == 8) sweep(std::integral_constant<int, 8>());
    else if (tile == 16) sweep(std::integral_constant<int, 16>());
    else if (tile == 32) sweep(std::integral_constant<int, 32>());
    else sweep(std::integral_constant<int, 64>());
    NWG_LAUNCH_CHECK();
  }
  NWG_HIP(hipEventRecord(ctx->ev1, s));
  st.its.ensure(k);
  ppr_its_kernel<<<grid1(k), kThreads, 0, s>>>(k, st.lanes.p, kpad, st.acc.p, max_iters, (double)threshold, st.its.p);
  if (k % 4 == 0 && (uintptr_t)scores_dev % 16 == 0)
    ppr_scores4_kernel<<<grid1(nk / 4), kThreads, 0, s>>>(
        n, k / 4, P.kt_shift, a.order, st.degflag.p, reinterpret_cast<const float4*>(c0p),
        reinterpret_cast<const float4*>(c1p), reinterpret_cast<const uint4*>(st.its.p),
        reinterpret_cast<float4*>(scores_dev));
  else
    ppr_scores_kernel<<<grid1(nk), kThreads, 0, s>>>(n, k, P.kt_shift, a.order, st.degflag.p, c0p, c1p, st.its.p,
                                                     scores_dev);
  NWG_LAUNCH_CHECK();
  std::vector<unsigned long long> h_acc(std::max<uint64_t>(max_iters, 1) * k);
  NWG_HIP(hipMemcpyAsync(h_acc.data(), st.acc.p, max_iters * k * 8ull, hipMemcpyDeviceToHost, s));
  NWG_HIP(hipStreamSynchronize(s));
  float ms = 0.f;
  NWG_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
  uint64_t max_it = 0;
  for (uint32_t j = 0; j < k; ++j) {
    uint64_t itj = max_iters;
    for (uint64_t t = 0; t < max_iters; ++t)
      if (fixed_to_err(h_acc[t * k + j]) < (double)threshold) {
        itj = t + 1;
        break;
      }
    if (iterations) iterations[j] = itj;
    max_it = std::max(max_it, itj);
  }
  if (info) {
    info->iterations = max_it;
    info->final_error = 0.0;
    for (uint32_t j = 0; j < k && max_it; ++j) info->final_error += fixed_to_err(h_acc[(max_it - 1) * k + j]);
    info->ms_total = ms;
    info->ms_per_iter = max_it ? ms / (double)max_it : 0.0;
    info->sweep_ms_avg = 0.0;
  }
}

}  // namespace nwg
