// small.hpp -- whole solves of small graphs, one workgroup each (small.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nwg {

// A teleport vector's sum, and whether some entry is no value of [0, 1].
struct TeleCheck {
  double sum;
  double bad;
};
// rounding slack allowed above 1 in the sum of a teleport vector
constexpr double kTeleportSlack = 1e-4;
__host__ __device__ __forceinline__ bool teleport_ok(const TeleCheck& c) {
  return c.bad == 0.0 && c.sum <= 1.0 + kTeleportSlack;
}

// One graph, or many in one block-diagonal CSC (a workgroup per graph).
struct SmallParams {
  const uint32_t* rp;
  const uint32_t* col;
  const uint32_t* deg;
  const uint32_t* voff;   // many graphs: first row of each, ngraphs + 1; null: one graph of n rows
  uint32_t n;
  uint32_t ngraphs;
  const float* basev;     // base per row, or null
  float base;
  float damp;
  float* x;               // scores; with k0 > 0 those of sweep k0 - 1
  float* out;             // nullable: out[order ? order[i] : i] = x[i], unless tele (nullable) failed
  const uint32_t* order;
  const TeleCheck* tele;
  const uint32_t* bad;       // nullable: two flags that say the graph is not to be looked at; in bad_mail too
  unsigned long long* bad_mail;
  unsigned long long* acc;   // [k * ngraphs + graph]: L1 change of sweep k, fixed point; 0 once stopped
  unsigned long long* mail;  // nullable, one graph: acc[k] there too
  unsigned long long* cut;   // set to 1 when fixed point cut bits off some contribution
  double threshold;
};

// One weighted solve y <- fma(d, sum w y, b), whose scales are made on the device (WItemParams).
struct SmallWeighted {
  const uint32_t* rp;
  const uint32_t* col;
  const float* w;         // in the order of col
  const float* base;
  const float* y0;        // first iterate; null: uniform
  float uniform;
  float damp;
  uint32_t n;
  float* state;           // the iterate between launches
  float* out;             // the last iterate
  const int* qshift;
  double* err;            // [k]: L1 change of sweep k; 0 once stopped
  unsigned long long* mail;         // nullable: the scales' two words, then err
  unsigned long long* cut;          // set to 1 when fixed point cut bits off some product
  const unsigned long long* scale;
  double threshold;
  const double* thr_scale;  // nullable: the stop compares with threshold * *thr_scale
};

// A solve that reports a cut is no answer: the item sweep is, which adds rows up once more where it shows.

// Sweeps per launch: a solve of any length is cut into launches of bounded time.
constexpr uint64_t kSmallSweeps = 1024;

// whether a graph of n rows and nnz edges (many: every graph of at most that) is solved by one workgroup
bool small_fits(uint64_t n, uint64_t nnz, bool many);
// sweeps [k0, k1) of the solve; n and nnz: the largest graph's
void small_enqueue(hipStream_t s, const SmallParams& P, uint64_t n, uint64_t nnz, uint64_t k0, uint64_t k1);
void small_weighted_enqueue(hipStream_t s, const SmallWeighted& P, uint64_t nnz, uint64_t k0, uint64_t k1);

}  // namespace nwg
