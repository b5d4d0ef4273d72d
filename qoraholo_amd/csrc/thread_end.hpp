// What a thread keeps of the device, released when the thread ends, but not while the process does.
//
// The thread_local objects of a thread end with the operating system's thread, which may be after
// whoever joined it goes on (a Python thread counts as joined once its interpreter state is gone). A
// process that exits right after its last calls would have such a thread call into the HIP runtime
// while exit() takes the runtime down. So the objects of ended threads are released under a lock which
// an exit handler takes as well: it waits for a release that is under way, and those that come later
// leave their objects to the end of the process. Handlers run in reverse order of their registration,
// so it is registered after the runtime has been initialised.
#pragma once

#include <functional>

namespace qh {

// Registers the exit handler, once. The HIP runtime has been used.
void watch_exit();
// f(), unless the process is exiting.
void at_thread_end(const std::function<void()>& f);

// A thread's T, built on first use (which uses the device) and deleted at the end of the thread.
template <class T>
class PerThread {
 public:
  PerThread() = default;
  ~PerThread() {
    if (p_) at_thread_end([this] { delete p_; });
  }
  PerThread(const PerThread&) = delete;
  PerThread& operator=(const PerThread&) = delete;
  T& get() {
    if (!p_) {
      p_ = new T;
      watch_exit();
    }
    return *p_;
  }

 private:
  T* p_ = nullptr;
};

}  // namespace qh
