// devpool.hpp -- device memory kept by a context between calls.
//
// hipMalloc and hipFree of large blocks are slow (on MI355X 270 us for 256 MB and more, and once
// a program has freed as much as the card holds, every new block waits until freed memory is
// cleared: building a graph of 67 M edges, which took 2.5 GB in 16 blocks, went from 13 to
// 100 ms a call).  A context therefore keeps the blocks its calls release and hands them out
// again.
//
// Safe reuse: a block goes back to the pool of the context whose call allocated it and only to
// calls of that context, whose device work is ordered by the context's stream; calls wait for
// their work before they return (also when they fail: guarded()), so a block that comes back
// after the stream was changed has no work left on it.  Objects that outlive a call are
// destroyed after the device is idle.  The lists are locked: objects are destroyed outside a call's
// turn on its context.
//
// Bounds: the pool keeps at most 1/64 of the device's memory in free blocks, of which those
// given back longest ago make room for new ones (the largest first instead: once a program has solved
// graphs of many sizes, every build of the 67 M-edge graph gave its own blocks away, 27 ms against 4),
// gives all of them back when an allocation of any context on the device fails or its own is destroyed,
// and keeps nothing after that.
#pragma once

#include <cstddef>
#include <cstdint>
#include <map>
#include <memory>
#include <mutex>

namespace nwg {

class DevPool {
 public:
  DevPool(int device, size_t limit);
  ~DevPool();
  DevPool(const DevPool&) = delete;
  DevPool& operator=(const DevPool&) = delete;
  // a block of at least bytes (> 0) on the current device; *size receives its size.  Throws Error.
  void* take(size_t bytes, size_t* size);
  void give(void* p, size_t size) noexcept;
  // frees every free block and keeps none from now on
  void close() noexcept;

 private:
  void trim_locked() noexcept;
  static void trim_all(int device);
  std::mutex mu_;
  const int device_;
  struct Free {
    void* p;
    uint64_t given;  // when: blocks given back longest ago go first
  };
  std::multimap<size_t, Free> free_;  // by size
  uint64_t gifts_ = 0;
  size_t held_ = 0, limit_;
};

// The pool that allocations of this thread use while a call on a context runs (null: none).
const std::shared_ptr<DevPool>& current_pool();
class PoolScope {
 public:
  explicit PoolScope(std::shared_ptr<DevPool> p);
  ~PoolScope();
  PoolScope(const PoolScope&) = delete;
  PoolScope& operator=(const PoolScope&) = delete;

 private:
  std::shared_ptr<DevPool> prev_;
};

// allocation and release of a DevBuf: from pool when given, else hipMalloc / hipFree
void* dev_alloc(const std::shared_ptr<DevPool>& pool, size_t bytes, size_t* size);
void dev_free(const std::shared_ptr<DevPool>& pool, void* p, size_t size) noexcept;

}  // namespace nwg
