// Device memory of the per-call entry points.
//
// A call allocates its buffers, works on one stream and returns when the stream is done. The
// blocks go back to a pool of the process instead of the driver: an allocation and free of 4 MB or
// more takes 23 us, and each free waits for the device (rytov of 49 x 256^2 spent about 0.4 of its
// 2.0 ms outside its transfers and kernels; reconstruct of 25 x 64^2 about 0.1 of 0.33 ms).
//
// The pool keeps at most kPoolBytes per process, frees blocks that kPoolCalls calls in a row did
// not take, and is freed when an allocation of the library runs out of memory and when the last
// thread that made calls ends before the process does. Blocks are handed over only after the stream
// that used them has been waited for, so any thread and stream may take them. Other allocators of the
// process do not see the pool: one that runs out (torch's, say) finds up to kPoolBytes less than
// before.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <vector>

namespace qh {

inline constexpr std::size_t kPoolBytes = std::size_t(1) << 30;
inline constexpr unsigned kPoolCalls = 64;

// hipMalloc, with the pool freed and one more attempt when memory runs out.
void* device_alloc(std::size_t bytes);
// Device memory an allocation could get: what is free and what the pool would give back.
std::size_t device_bytes_free();

// The device allocations of the calling thread (DeviceBuffer) come from the pool while this
// object lives, and go back to it, after the stream has been waited for, when it ends. It is
// declared before the buffers it serves; what outlives the call is allocated under Outside.
class CallMemory {
 public:
  explicit CallMemory(hipStream_t s);
  ~CallMemory();
  CallMemory(const CallMemory&) = delete;
  CallMemory& operator=(const CallMemory&) = delete;

  static CallMemory* current();
  void* take(std::size_t bytes);
  // The block is not used again within the call: memory may still be read by queued work.
  void give(void* p);

  class Outside {
   public:
    Outside();
    ~Outside();
    Outside(const Outside&) = delete;
    Outside& operator=(const Outside&) = delete;

   private:
    CallMemory* saved_;
  };

 private:
  struct Block {
    void* p;
    std::size_t bytes;
    bool live;
  };
  hipStream_t s_;
  int device_ = 0;
  CallMemory* outer_;
  std::vector<Block> blocks_;
};

}  // namespace qh
