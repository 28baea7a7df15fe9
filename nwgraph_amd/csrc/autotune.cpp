// autotune.cpp -- picks the sweep plan (degree-bin cutoffs, hub split, cache hints)
// of a graph by timing candidate plans on the device with HIP events.
//
// Search: coordinate descent over the pull sweep's parameters from the default plan (the item
// sweep; cutoffs of its own ask for the row classes, and only those have cache hints), one
// parameter at a time, each candidate timed over a few sweeps (launched one by one, each
// bracketed by events); then the binned sweep in both numberings, with its cache hints and
// bin size, which is named throughout (left open, the plan may run the item sweep); then the best pull
// plan and the best binned plan timed again as whole captured 20-sweep solves (median of 7), and
// the faster one kept.
// Results are cached per (log2 in-degree histogram, n, nnz, device) for the process
// and, if NWG_TUNE_CACHE names a file, appended there and reloaded by later processes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <map>
#include <mutex>
#include <sstream>
#include <string>
#include <vector>

#include "nwg_internal.hpp"

namespace nwg {

namespace {

std::mutex g_cache_mu;
std::map<std::string, nwg_plan_params> g_cache;
bool g_file_loaded = false;

std::string params_to_string(const nwg_plan_params& p) {
  std::ostringstream o;
  o << p.short_max << ' ' << p.group_max << ' ' << p.hub_min << ' ' << p.hub_segment << ' ' << p.slice_min
    << ' ' << p.stream_hints << ' ' << p.ppr_tile << ' ' << p.relabel << ' ' << p.binned << ' ' << p.bin_bits;
  return o.str();
}

bool params_from_stream(std::istream& in, nwg_plan_params* p) {
  nwg_plan_params q{};
  if (!(in >> q.short_max >> q.group_max >> q.hub_min >> q.hub_segment >> q.slice_min >> q.stream_hints >>
        q.ppr_tile >> q.relabel >> q.binned))
    return false;
  if (!(in >> q.bin_bits)) q.bin_bits = 0;  // entries written before the field existed
  *p = q;
  return true;
}

void load_file_cache() {
  if (g_file_loaded) return;
  g_file_loaded = true;
  const char* path = std::getenv("NWG_TUNE_CACHE");
  if (!path) return;
  std::ifstream in(path);
  std::string line;
  while (std::getline(in, line)) {
    std::istringstream ls(line);
    std::string key;
    nwg_plan_params p{};
    if (ls >> key && params_from_stream(ls, &p)) g_cache[key] = p;
  }
}

void store_file_cache(const std::string& key, const nwg_plan_params& p) {
  const char* path = std::getenv("NWG_TUNE_CACHE");
  if (!path) return;
  std::ofstream out(path, std::ios::app);
  out << key << ' ' << params_to_string(p) << '\n';
}

// in-degree histogram of the CSC, log2 buckets, as a cache key
std::string graph_key(hipStream_t s, const nwg_graph* g) {
  std::vector<uint32_t> rp((size_t)g->n + 1);
  NWG_HIP(hipMemcpyAsync(rp.data(), g->csc_ptr.p, rp.size() * 4, hipMemcpyDeviceToHost, s));
  NWG_HIP(hipStreamSynchronize(s));
  uint64_t hist[33] = {};
  for (uint32_t i = 0; i < g->n; ++i) {
    const uint32_t d = rp[i + 1] - rp[i];
    int b = 0;
    while (b < 32 && (1u << b) <= d) ++b;
    hist[b]++;
  }
  int dev = 0;
  NWG_HIP(hipGetDevice(&dev));
  hipDeviceProp_t prop{};
  NWG_HIP(hipGetDeviceProperties(&prop, dev));
  uint64_t h = 1469598103934665603ull;  // FNV-1a over the histogram
  for (uint64_t v : hist) {
    for (int q = 0; q < 8; ++q) {
      h ^= (v >> (8 * q)) & 0xFF;
      h *= 1099511628211ull;
    }
  }
  std::ostringstream o;
  o << prop.gcnArchName << ':' << prop.multiProcessorCount << ":n" << g->n << ":e" << g->nnz << ":h" << std::hex
    << h;
  std::string k = o.str();
  for (auto& c : k)
    if (c == ' ') c = '_';
  return k;
}

}  // namespace

double time_plan_sweeps(nwg_ctx* ctx, nwg_graph* g, uint64_t iters) {
  nwg_pr_info info{};
  info.flags = NWG_INFO_KERNEL_TIMING;
  DevBuf<float> out(g->n);
  pagerank_run(ctx, g, nullptr, 0.85f, -1.0f, iters, &info, out.p);
  return info.sweep_ms_avg;
}

// Median device time per sweep of whole solves (the captured HIP graph of `iters` sweeps,
// as a caller runs it), after one solve whose launches go out one by one and one that captures them.
// Small graphs are launch-bound, where per-sweep event timing of one-by-one launches is
// noisy and measures launch gaps the captured loop does not have.
static double time_plan_solve(nwg_ctx* ctx, nwg_graph* g, uint64_t iters, int reps) {
  nwg_pr_info info{};
  DevBuf<float> out(g->n);
  for (int r = 0; r < 2; ++r) pagerank_run(ctx, g, nullptr, 0.85f, -1.0f, iters, &info, out.p);
  std::vector<double> t;
  for (int r = 0; r < reps; ++r) {
    pagerank_run(ctx, g, nullptr, 0.85f, -1.0f, iters, &info, out.p);
    t.push_back(info.ms_total / (double)iters);
  }
  std::sort(t.begin(), t.end());
  return t[t.size() / 2];
}

nwg_plan_params autotune_plan(nwg_ctx* ctx, nwg_graph* g) {
  hipStream_t s = ctx->stream;
  const std::string key = graph_key(s, g);
  {
    std::lock_guard<std::mutex> lk(g_cache_mu);
    load_file_cache();
    auto it = g_cache.find(key);
    if (it != g_cache.end()) {
      plan_build(s, g, it->second);
      return it->second;
    }
  }
  auto eval_n = [&](const nwg_plan_params& p, int reps, uint64_t sweeps) -> double {
    try {
      plan_build(s, g, p);
    } catch (const Error&) {
      return 1e30;  // invalid combination
    }
    double best = 1e30;
    for (int r = 0; r < reps; ++r) best = std::min(best, time_plan_sweeps(ctx, g, sweeps));
    return best;
  };
  auto eval = [&](const nwg_plan_params& p) -> double { return eval_n(p, 2, 4); };
  nwg_plan_params best = default_plan_params();  // the pull sweep, original numbering
  double best_ms = eval(best);
  auto try_field = [&](uint32_t nwg_plan_params::*field, std::initializer_list<uint32_t> values) {
    for (uint32_t v : values) {
      nwg_plan_params c = best;
      c.*field = v;
      if (c.*field == best.*field) continue;
      const double ms = eval(c);
      if (ms < best_ms) {
        best_ms = ms;
        best = c;
      }
    }
  };
  // the pull sweep: numbering, then its row-class cutoffs, hub split and slicing, and the row
  // classes' hints
  try_field(&nwg_plan_params::relabel, {0, 1});
  try_field(&nwg_plan_params::short_max, {0, 2, 4, 8, 16, 32});
  try_field(&nwg_plan_params::group_max, {16, 32, 64, 128, 256, 512, 1024});
  try_field(&nwg_plan_params::hub_min, {2048, 4096, 8192, 16384, 32768, 65536, 262144});
  try_field(&nwg_plan_params::hub_segment, {1024, 2048, 4096, 8192, 16384});
  try_field(&nwg_plan_params::slice_min, {0, 33, 65, 129, 257, 1025});
  try_field(&nwg_plan_params::short_max, {0, 2, 4, 8, 16, 32});
  if (!plan_takes_items(best, g)) try_field(&nwg_plan_params::stream_hints, {0, 1, 2});
  const nwg_plan_params pull = best;
  // the binned sweep ignores the row-class cutoffs; only the numbering matters
  nwg_plan_params binned = pull, b0 = pull;
  binned.binned = b0.binned = 1;
  binned.bin_bits = b0.bin_bits = 13;
  binned.relabel = 1;
  b0.relabel = 0;
  if (eval(b0) < eval(binned)) binned = b0;
  // and its cache hints (non-temporal loads / stores of the once-read streams)
  {
    double bt = 1e30;
    nwg_plan_params bh = binned;
    for (uint32_t h : {0u, 1u, 2u}) {
      nwg_plan_params c = binned;
      c.stream_hints = h;
      const double ms = eval(c);
      if (ms < bt) {
        bt = ms;
        bh = c;
      }
    }
    binned = bh;
  }
  // and its bin size (2^14-row bins: fewer pairs, one bin-pass workgroup per CU)
  {
    nwg_plan_params c = binned;
    const double b13 = eval(c);
    c.bin_bits = 14;
    if (eval(c) < b13) binned = c;
  }
  // the two winners, timed again as whole captured solves (median of 7)
  plan_build(s, g, pull);
  const double t_pull = time_plan_solve(ctx, g, 20, 7);
  plan_build(s, g, binned);
  const double t_binned = time_plan_solve(ctx, g, 20, 7);
  best = t_binned <= t_pull ? binned : pull;
  plan_build(s, g, best);
  {
    std::lock_guard<std::mutex> lk(g_cache_mu);
    g_cache[key] = best;
    store_file_cache(key, best);
  }
  return best;
}

}  // namespace nwg
