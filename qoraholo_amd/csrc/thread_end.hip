// Release of threads' device objects against the end of the process (see thread_end.hpp).
#include "thread_end.hpp"

#include <cstdlib>
#include <mutex>

namespace qh {

namespace {

// Never destroyed: threads may end after the static objects.
struct Exit {
  std::mutex mu;
  std::once_flag once;
  bool exiting = false;
};
Exit& process_exit() {
  static Exit* const e = new Exit;
  return *e;
}

}  // namespace

void watch_exit() {
  std::call_once(process_exit().once, [] {
    std::atexit([] {
      std::lock_guard<std::mutex> lock(process_exit().mu);
      process_exit().exiting = true;
    });
  });
}

void at_thread_end(const std::function<void()>& f) {
  std::lock_guard<std::mutex> lock(process_exit().mu);
  if (!process_exit().exiting) f();
}

}  // namespace qh
