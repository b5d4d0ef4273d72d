// Host ingest and egress. Copies between pageable host memory (numpy arrays, callers' buffers)
// and the device go through rings of pinned staging slots of the calling thread, chunk by chunk:
// the host side of each chunk is spread over a small pool of copy threads and overlaps the DMA
// of the neighbouring chunk. A plain hipMemcpy from pageable memory stages through the
// runtime's own buffers with one host thread: 25.7 MB take 754 us in and 1560 us out that way,
// 1 MB 46 and 65 us; the DMA alone 476 and 27 us, the host copy 190 and 14 us.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <deque>
#include <functional>

namespace qh {

// Transfers up to this size go through one staging slot: a copy into it takes about half the time of
// its DMA, so that the first chunk's copy is all the DMA of a larger transfer waits for and the last
// chunk's all that follows it.
inline constexpr std::size_t kStagingSlot = std::size_t(8) << 20;

// Threads a host copy is spread over (the caller included): half the CPUs this process may
// run on, at most 8.
int host_copy_threads();

// dst[0, bytes) = src[0, bytes), split over host_copy_threads() threads.
void host_copy(void* dst, const void* src, std::size_t bytes);

// part(0) .. part(parts - 1) on the copy threads and the calling thread; returns when all are
// done.
void parallel_for(int parts, const std::function<void(int)>& part);

// Per-thread stream of the per-call entry points, so calls from different host threads run
// independently. It lives as long as the thread's staging slots.
hipStream_t call_stream();

// While it lives, small transfers of the calling thread on s are waited for with the stream, as on
// call_stream(), instead of an event each. It waits for s when it ends, so that the staging keeps
// nothing of a stream that may be destroyed then.
class StagedStream {
 public:
  explicit StagedStream(hipStream_t s);
  ~StagedStream();
  StagedStream(const StagedStream&) = delete;
  StagedStream& operator=(const StagedStream&) = delete;

 private:
  hipStream_t s_;
  hipStream_t outer_;
};

// Device dst <- pageable host src. Returns once src may be reused; the DMA of the last chunks
// may still be in flight on s, ahead of any later work on s.
void upload(void* dst, const void* src, std::size_t bytes, hipStream_t s);

// Pageable host dst <- device src, after the work already queued on s. Returns with dst
// complete.
void download(void* dst, const void* src, std::size_t bytes, hipStream_t s);

// Several downloads whose DMAs queue up behind each other: add() returns with the copies queued
// as far as the staging slots go, finish() with every dst complete.
class Downloads {
 public:
  // alone: next to nothing is queued behind it on s before finish(), so that on call_stream() and
  // a StagedStream it is waited for with the stream and needs no event.
  void add(void* dst, const void* src, std::size_t bytes, hipStream_t s, bool alone = false);
  void finish();

 private:
  void retire();
  struct Part {
    int slot;
    char* dst;
    std::size_t bytes;
  };
  std::deque<Part> parts_;
};

}  // namespace qh
