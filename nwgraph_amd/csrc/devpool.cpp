// devpool.cpp -- the free lists of devpool.hpp.
#include "devpool.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <new>
#include <vector>

#include "nwg_internal.hpp"

namespace nwg {

namespace {

thread_local std::shared_ptr<DevPool> t_pool;

// every pool, for trim_all (never destroyed: a context may outlive this file's statics)
std::mutex g_pools_mu;
std::vector<DevPool*>& pools() {
  static auto* all = new std::vector<DevPool*>();
  return *all;
}

// below 1 MiB powers of two, from there whole MiB: few sizes, little waste
size_t block_size(size_t bytes) {
  constexpr size_t kMiB = 1u << 20;
  if (bytes >= kMiB) return (bytes + kMiB - 1) / kMiB * kMiB;
  size_t s = 512;
  while (s < bytes) s <<= 1;
  return s;
}

}  // namespace

const std::shared_ptr<DevPool>& current_pool() { return t_pool; }
PoolScope::PoolScope(std::shared_ptr<DevPool> p) : prev_(std::move(t_pool)) { t_pool = std::move(p); }
PoolScope::~PoolScope() { t_pool = std::move(prev_); }

DevPool::DevPool(int device, size_t limit) : device_(device), limit_(limit) {
  std::lock_guard<std::mutex> lk(g_pools_mu);
  pools().push_back(this);
}

DevPool::~DevPool() {
  {
    std::lock_guard<std::mutex> lk(g_pools_mu);
    pools().erase(std::find(pools().begin(), pools().end(), this));
  }
  close();
}

// hipFree waits for the device, which must not happen while another thread records a graph
void DevPool::trim_all(int device) {
  std::lock_guard<std::mutex> recording(capture_mutex());
  std::lock_guard<std::mutex> lk(g_pools_mu);
  for (DevPool* p : pools()) {
    if (p->device_ != device) continue;
    std::lock_guard<std::mutex> own(p->mu_);
    p->trim_locked();
  }
}

void DevPool::trim_locked() noexcept {
  for (auto& b : free_) (void)hipFree(b.second.p);
  free_.clear();
  held_ = 0;
}

void* DevPool::take(size_t bytes, size_t* size) {
  const size_t want = block_size(bytes);
  *size = want;
  {
    std::lock_guard<std::mutex> lk(mu_);
    const auto it = free_.lower_bound(want);
    if (it != free_.end() && it->first <= want + want / 2) {  // the smallest that does, if not much too large
      void* p = it->second.p;
      *size = it->first;
      held_ -= it->first;
      free_.erase(it);
      return p;
    }
  }
  void* p = nullptr;
  if (hipMalloc(&p, want) == hipSuccess) return p;
  (void)hipGetLastError();
  trim_all(device_);
  const hipError_t e = hipMalloc(&p, want);
  if (e == hipSuccess) return p;
  (void)hipGetLastError();  // reported here; a caller may go on without the block
  throw Error(e == hipErrorOutOfMemory ? NWG_ENOMEM : NWG_EHIP,
              "hipMalloc of " + std::to_string(want) + " bytes failed: " + hipGetErrorString(e));
}

void DevPool::give(void* p, size_t size) noexcept {
  {
    std::lock_guard<std::mutex> lk(mu_);
    if (size <= limit_) {
      while (held_ + size > limit_) {
        const auto it = std::min_element(free_.begin(), free_.end(), [](const auto& a, const auto& b) {
          return a.second.given < b.second.given;
        });
        (void)hipFree(it->second.p);
        held_ -= it->first;
        free_.erase(it);
      }
      try {
        free_.emplace(size, Free{p, ++gifts_});
        held_ += size;
        return;
      } catch (const std::bad_alloc&) {
      }
    }
  }
  (void)hipFree(p);
}

void DevPool::close() noexcept {
  std::lock_guard<std::mutex> lk(mu_);
  trim_locked();
  limit_ = 0;
}

void* dev_alloc(const std::shared_ptr<DevPool>& pool, size_t bytes, size_t* size) {
  if (pool) return pool->take(bytes, size);
  void* p = nullptr;
  NWG_HIP(hipMalloc(&p, bytes));
  *size = bytes;
  return p;
}

void dev_free(const std::shared_ptr<DevPool>& pool, void* p, size_t size) noexcept {
  if (pool) pool->give(p, size);
  else (void)hipFree(p);
}

}  // namespace nwg
