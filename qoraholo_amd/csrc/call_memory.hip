#include "call_memory.hpp"

#include <algorithm>
#include <mutex>

#include "runtime.hpp"
#include "thread_end.hpp"

namespace qh {

namespace {

struct Entry {
  void* p;
  std::size_t bytes;
  int device;
  unsigned call;  // number of the call that gave it back
};

class Pool {
 public:
  void* get(std::size_t bytes, int device, std::size_t& got) {
    std::lock_guard<std::mutex> lock(mu_);
    auto best = entries_.end();
    for (auto it = entries_.begin(); it != entries_.end(); ++it) {
      // No block of more than twice the size: a small buffer would keep a large one from the
      // allocation that it fits.
      if (it->device == device && it->bytes >= bytes &&
          it->bytes <= std::max<std::size_t>(2 * bytes, 1 << 16) &&
          (best == entries_.end() || it->bytes < best->bytes)) {
        best = it;
      }
    }
    if (best == entries_.end()) return nullptr;
    void* const p = best->p;
    got = best->bytes;
    total_ -= best->bytes;
    entries_.erase(best);
    return p;
  }

  // The blocks of a call that has ended; those beyond the bounds are freed, oldest first.
  void put(std::vector<Entry>& blocks) {
    std::vector<void*> drop;
    {
      std::lock_guard<std::mutex> lock(mu_);
      ++call_;
      for (Entry& e : blocks) {
        e.call = call_;
        entries_.push_back(e);
        total_ += e.bytes;
      }
      while (!entries_.empty() &&
             (total_ > kPoolBytes || call_ - entries_.front().call > kPoolCalls)) {
        drop.push_back(entries_.front().p);
        total_ -= entries_.front().bytes;
        entries_.erase(entries_.begin());
      }
    }
    for (void* p : drop) (void)hipFree(p);
  }

  void trim() {
    std::vector<Entry> all;
    {
      std::lock_guard<std::mutex> lock(mu_);
      all.swap(entries_);
      total_ = 0;
    }
    for (const Entry& e : all) (void)hipFree(e.p);
  }

  std::size_t bytes(int device) {
    std::lock_guard<std::mutex> lock(mu_);
    std::size_t b = 0;
    for (const Entry& e : entries_) b += e.device == device ? e.bytes : 0;
    return b;
  }

  void enter() {
    std::lock_guard<std::mutex> lock(mu_);
    ++threads_;
  }
  void leave() {
    bool last = false;
    {
      std::lock_guard<std::mutex> lock(mu_);
      last = --threads_ == 0;
    }
    if (last) trim();
  }

 private:
  std::mutex mu_;
  std::vector<Entry> entries_;  // in the order they were given back
  std::size_t total_ = 0;
  unsigned call_ = 0;
  int threads_ = 0;
};

// Never destroyed: threads may end after the static objects.
Pool& pool() {
  static Pool* const p = new Pool;
  return *p;
}

struct ThreadMark {
  ThreadMark() { pool().enter(); }
  ~ThreadMark() { pool().leave(); }
};

CallMemory*& current_call() {
  thread_local CallMemory* c = nullptr;
  return c;
}

int current_device() {
  int d = 0;
  check(hipGetDevice(&d), "hipGetDevice");
  return d;
}

// Sizes of pooled blocks: calls of nearly the same size share them.
std::size_t rounded(std::size_t bytes) {
  const std::size_t step = bytes < (std::size_t(16) << 20) ? std::size_t(1) << 16 : std::size_t(2) << 20;
  return (bytes + step - 1) / step * step;
}

}  // namespace

void* device_alloc(std::size_t bytes) {
  void* p = nullptr;
  hipError_t e = hipMalloc(&p, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    pool().trim();
    e = hipMalloc(&p, bytes);
  }
  check(e, "hipMalloc");
  return p;
}

std::size_t device_bytes_free() {
  std::size_t free_bytes = 0, total_bytes = 0;
  check(hipMemGetInfo(&free_bytes, &total_bytes), "hipMemGetInfo");
  return free_bytes + pool().bytes(current_device());
}

CallMemory::CallMemory(hipStream_t s) : s_(s), device_(current_device()), outer_(current_call()) {
  thread_local PerThread<ThreadMark> mark;
  mark.get();
  current_call() = this;
}

CallMemory::~CallMemory() {
  current_call() = outer_;
  // A stream that failed may still use the blocks: hipFree waits for the device.
  const bool done = hipStreamSynchronize(s_) == hipSuccess;
  if (!done) {
    for (const Block& b : blocks_) (void)hipFree(b.p);
    return;
  }
  try {
    std::vector<Entry> entries;
    entries.reserve(blocks_.size());
    for (const Block& b : blocks_) entries.push_back({b.p, b.bytes, device_, 0});
    pool().put(entries);
  } catch (...) {
    // Out of host memory: what put() has not taken stays allocated.
  }
}

CallMemory* CallMemory::current() { return current_call(); }

void* CallMemory::take(std::size_t bytes) {
  blocks_.reserve(blocks_.size() + 1);
  std::size_t got = rounded(bytes);
  void* p = pool().get(got, device_, got);
  if (p == nullptr) {
    hipError_t e = hipMalloc(&p, got);
    if (e == hipErrorOutOfMemory) {
      // What earlier steps of the call have given up, the pool, and no rounding.
      (void)hipGetLastError();
      check(hipStreamSynchronize(s_), "hipStreamSynchronize");
      const auto spent = std::partition(blocks_.begin(), blocks_.end(), [](const Block& b) { return b.live; });
      for (auto it = spent; it != blocks_.end(); ++it) (void)hipFree(it->p);
      blocks_.erase(spent, blocks_.end());
      got = bytes;
      p = device_alloc(got);
    } else {
      check(e, "hipMalloc");
    }
  }
  blocks_.push_back({p, got, true});
  return p;
}

void CallMemory::give(void* p) {
  for (Block& b : blocks_) {
    if (b.p == p) b.live = false;
  }
}

CallMemory::Outside::Outside() : saved_(current_call()) { current_call() = nullptr; }
CallMemory::Outside::~Outside() { current_call() = saved_; }

}  // namespace qh
