// Host ingest and egress (see hostio.hpp).
#include "hostio.hpp"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <bit>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

#include "runtime.hpp"
#include "thread_end.hpp"

namespace qh {

namespace {

// Staging slots: two that transfers in several chunks take in turn, either way, and four in turn for
// the single chunks of each direction.
constexpr int kPair = 2;
constexpr int kRing = 4;
constexpr int kSlots = kPair + 2 * kRing;
// Chunks of transfers that take several. A DMA of 4 MB leaves a gap of a seventh
// of its time to the next one (128 / 256 MB in and out: 7.0 / 13.0 ms in chunks of 4 MB, 5.5 / 10.7 of
// 8, 5.4 / 10.4 of 16), and the first and last host copy of a smaller transfer wait for less in
// smaller chunks (24 MB: 1.21 ms of 8, 1.27 to 1.33 of 16).
constexpr std::size_t kLarge = std::size_t(128) << 20;
constexpr std::size_t kLargeChunk = std::size_t(16) << 20;
constexpr std::size_t chunk_of(std::size_t bytes) {
  return bytes > kLarge ? kLargeChunk : kStagingSlot;
}
// Host copies are split over threads, into parts of at least kMinPart, from where that pays for waking
// them (calls that move 1 / 1.25 / 1.5 MB in and out: 162 / 180 / 180 us by two threads, 137 / 158 /
// 200 us by one).
constexpr std::size_t kMinPart = std::size_t(1) << 19;
constexpr std::size_t kMinSplit = 3 * kMinPart;

int usable_cpus() {
  cpu_set_t set;
  CPU_ZERO(&set);
  if (sched_getaffinity(0, sizeof set, &set) == 0) return std::max(1, CPU_COUNT(&set));
  return std::max(1u, std::thread::hardware_concurrency());
}

// A fixed set of copy threads. A job is a number of parts; the submitting thread works on its
// own job too, so a job always finishes even when every pool thread is busy with other jobs.
class CopyPool {
 public:
  explicit CopyPool(int threads) {
    for (int i = 0; i < threads; ++i) workers_.emplace_back([this] { loop(); });
  }
  ~CopyPool() {
    {
      std::lock_guard<std::mutex> lock(mu_);
      stop_ = true;
    }
    cv_.notify_all();
    for (auto& t : workers_) t.join();
  }
  CopyPool(const CopyPool&) = delete;
  CopyPool& operator=(const CopyPool&) = delete;

  void run(int parts, const std::function<void(int)>& part) {
    auto job = std::make_shared<Job>();
    job->parts = parts;
    job->part = &part;
    {
      std::lock_guard<std::mutex> lock(mu_);
      jobs_.push_back(job);
    }
    cv_.notify_all();
    work(*job);
    retire(job);
    std::unique_lock<std::mutex> lock(job->mu);
    job->done_cv.wait(lock, [&] { return job->done == job->parts; });
  }

 private:
  struct Job {
    int parts = 0;
    const std::function<void(int)>* part = nullptr;
    std::atomic<int> next{0};
    int done = 0;  // guarded by mu
    std::mutex mu;
    std::condition_variable done_cv;
  };

  static void work(Job& job) {
    for (;;) {
      const int i = job.next.fetch_add(1);
      if (i >= job.parts) return;
      (*job.part)(i);
      std::lock_guard<std::mutex> lock(job.mu);
      if (++job.done == job.parts) job.done_cv.notify_all();
    }
  }

  // Takes a job off the queue once all its parts are claimed (work() has returned for it).
  void retire(const std::shared_ptr<Job>& job) {
    std::lock_guard<std::mutex> lock(mu_);
    const auto it = std::find(jobs_.begin(), jobs_.end(), job);
    if (it != jobs_.end()) jobs_.erase(it);
  }

  void loop() {
    for (;;) {
      std::shared_ptr<Job> job;
      {
        std::unique_lock<std::mutex> lock(mu_);
        for (;;) {
          cv_.wait(lock, [&] { return stop_ || !jobs_.empty(); });
          if (stop_) return;
          job = jobs_.front();
          if (job->next.load() < job->parts) break;
          jobs_.pop_front();  // every part is claimed already
        }
      }
      work(*job);
      retire(job);
    }
  }

  std::vector<std::thread> workers_;
  std::mutex mu_;
  std::condition_variable cv_;
  std::deque<std::shared_ptr<Job>> jobs_;
  bool stop_ = false;
};

CopyPool& pool() {
  static CopyPool p(host_copy_threads() - 1);
  return p;
}

// The calling thread's pinned slots and what marks their last DMA. A slot grows to what it is used
// for, so that a thread's small calls pin little. Transfers of one slot on the thread's own stream, or
// on that of a StagedStream, are marked by the stream alone (an event after each is 10 us of a small
// call); several in a row, and all on other streams, which may be destroyed before the slot is used
// again, by the slot's event.
struct Staging {
  std::unique_ptr<Stream> own;   // call_stream()
  hipStream_t staged = nullptr;  // of the thread's StagedStream
  PinnedBuffer<char> memory[kSlots];
  Event done[kSlots]{Event(false), Event(false), Event(false), Event(false), Event(false),
                     Event(false), Event(false), Event(false), Event(false), Event(false)};
  enum class Mark { none, event, stream };
  Mark mark[kSlots] = {};
  hipStream_t stream[kSlots] = {};
  int pair = 0;
  int up = 0;
  int down = 0;

  // An error is reported once: the slot is free after it.
  void wait(int i) {
    const Mark m = std::exchange(mark[i], Mark::none);
    if (m == Mark::event) check(hipEventSynchronize(done[i].get()), "hipEventSynchronize");
    if (m == Mark::stream) check(hipStreamSynchronize(stream[i]), "hipStreamSynchronize");
  }
  // Slot i, its last DMA over, with room for `bytes`.
  char* slot(int i, std::size_t bytes) {
    wait(i);
    if (memory[i].size() < bytes) {
      memory[i] = PinnedBuffer<char>();
      memory[i] = PinnedBuffer<char>(std::max(std::bit_ceil(bytes), std::size_t(1) << 16));
    }
    return memory[i].get();
  }
  void queued(int i, hipStream_t s, bool alone) {
    const bool by_stream = alone && ((own && s == own->get()) || (staged && s == staged));
    if (!by_stream) done[i].record(s);
    mark[i] = by_stream ? Mark::stream : Mark::event;
    stream[i] = s;
  }
  // The slot of the next chunk.
  int next(bool several, bool download) {
    if (several) return std::exchange(pair, (pair + 1) % kPair);
    int& at = download ? down : up;
    return kPair + (download ? kRing : 0) + std::exchange(at, (at + 1) % kRing);
  }
  // s has been waited for.
  void settled(hipStream_t s) {
    for (int i = 0; i < kSlots; ++i) {
      if (mark[i] == Mark::stream && stream[i] == s) mark[i] = Mark::none;
    }
  }
};

Staging& staging() {
  thread_local PerThread<Staging> s;
  return s.get();
}

}  // namespace

int host_copy_threads() {
  static const int n = std::clamp(usable_cpus() / 2, 1, 8);
  return n;
}

void host_copy(void* dst, const void* src, std::size_t bytes) {
  const int threads = host_copy_threads();
  if (bytes < kMinSplit || threads == 1) {
    std::memcpy(dst, src, bytes);
    return;
  }
  const int parts = static_cast<int>(std::min<std::size_t>(threads, bytes / kMinPart));
  // Part boundaries on 4 KiB pages.
  const std::size_t step = ((bytes / parts) + 4095) & ~std::size_t(4095);
  auto* d = static_cast<char*>(dst);
  const auto* s = static_cast<const char*>(src);
  pool().run(parts, [&](int i) {
    const std::size_t a = std::min(bytes, i * step);
    const std::size_t b = std::min(bytes, a + step);
    if (b > a) std::memcpy(d + a, s + a, b - a);
  });
}

void parallel_for(int parts, const std::function<void(int)>& part) {
  if (parts <= 1) {
    if (parts == 1) part(0);
    return;
  }
  pool().run(parts, part);
}

hipStream_t call_stream() {
  Staging& st = staging();
  if (!st.own) st.own = std::make_unique<Stream>();
  return st.own->get();
}

StagedStream::StagedStream(hipStream_t s) : s_(s), outer_(std::exchange(staging().staged, s)) {}
StagedStream::~StagedStream() {
  // Settled also after an error: the stream does not run on past it.
  (void)hipStreamSynchronize(s_);
  Staging& st = staging();
  if (!(st.own && s_ == st.own->get())) st.settled(s_);
  st.staged = outer_;
}

void upload(void* dst, const void* src, std::size_t bytes, hipStream_t s) {
  Staging& st = staging();
  auto* d = static_cast<char*>(dst);
  const auto* h = static_cast<const char*>(src);
  const std::size_t chunk = chunk_of(bytes);
  for (std::size_t off = 0; off < bytes; off += chunk) {
    const std::size_t len = std::min(chunk, bytes - off);
    const int i = st.next(bytes > chunk, false);
    char* const slot = st.slot(i, len);
    host_copy(slot, h + off, len);
    check(hipMemcpyAsync(d + off, slot, len, hipMemcpyHostToDevice, s), "upload");
    st.queued(i, s, bytes <= chunk);
  }
}

void Downloads::add(void* dst, const void* src, std::size_t bytes, hipStream_t s, bool alone) {
  Staging& st = staging();
  auto* h = static_cast<char*>(dst);
  const auto* d = static_cast<const char*>(src);
  const std::size_t chunk = chunk_of(bytes);
  for (std::size_t off = 0; off < bytes; off += chunk) {
    const std::size_t len = std::min(chunk, bytes - off);
    const int i = st.next(bytes > chunk, true);
    while (std::any_of(parts_.begin(), parts_.end(), [&](const Part& p) { return p.slot == i; })) {
      retire();
    }
    check(hipMemcpyAsync(st.slot(i, len), d + off, len, hipMemcpyDeviceToHost, s), "download");
    st.queued(i, s, alone);
    parts_.push_back({i, h + off, len});
  }
}

void Downloads::retire() {
  Staging& st = staging();
  const Part p = parts_.front();
  parts_.pop_front();
  host_copy(p.dst, st.slot(p.slot, p.bytes), p.bytes);
}

void Downloads::finish() {
  while (!parts_.empty()) retire();
}

void download(void* dst, const void* src, std::size_t bytes, hipStream_t s) {
  Downloads d;
  d.add(dst, src, bytes, s, bytes <= kStagingSlot);
  d.finish();
}

}  // namespace qh
