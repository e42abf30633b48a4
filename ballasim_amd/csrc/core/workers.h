// A call's work spread over a few threads that are joined before it returns.
#pragma once

#include <stddef.h>

#include <exception>
#include <thread>
#include <vector>

namespace bsx {

// work(0) .. work(n - 1), each once: work(0) on the calling thread, the others on a thread each, or on the calling
// one too where no thread (or no memory for one) is to be had. work must not throw.
template <class F>
void run_workers(size_t n, const F& work) {
  static_assert(noexcept(work(size_t{0})), "a thrown exception would end the process with threads to join");
  if (n == 0) return;
  std::vector<std::thread> pool;
  size_t started = 1;
  try {
    pool.reserve(n - 1);  // (a growth that fails would destroy threads that run)
    for (; started < n; ++started) pool.emplace_back([&work, started] { work(started); });
  } catch (const std::exception&) {  // no thread (system_error), or no memory for its state (bad_alloc)
  }
  for (size_t k = started; k < n; ++k) work(k);
  work(0);
  for (std::thread& t : pool) t.join();
}

}  // namespace bsx
