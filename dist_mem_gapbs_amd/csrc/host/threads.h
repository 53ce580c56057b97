// Threads that a call can do without: an entry point with a C interface lets
// no exception out, and a started thread is always joined.
#ifndef DMM_HOST_THREADS_H_
#define DMM_HOST_THREADS_H_

#include <exception>
#include <thread>
#include <utility>

namespace dmm {

// Runs f on a thread of its own.  False, with nothing started, where none is
// to be had: no thread (std::system_error) or no memory for its state
// (std::bad_alloc).
template <typename F>
bool start_thread(std::thread* t, F f) noexcept {
  try {
    *t = std::thread(std::move(f));
    return true;
  } catch (const std::exception&) {
    return false;
  }
}

}  // namespace dmm

#endif  // DMM_HOST_THREADS_H_
