// run_workers when memory runs out: the allocations after the first argv[1] fail (up to argv[2] of them), and each
// piece of work must still be done exactly once. Prints how often each was done.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>

#include "workers.h"

static std::atomic<long> budget{1 << 30}, failures{0};

void* operator new(size_t n) {
  if (budget.fetch_sub(1) <= 0 && failures.fetch_sub(1) > 0) throw std::bad_alloc();
  void* p = std::malloc(n);
  if (p == nullptr) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

int main(int argc, char** argv) {
  constexpr size_t kN = 6;
  std::atomic<int> done[kN] = {};
  failures = argc > 2 ? std::atol(argv[2]) : 0;
  budget = argc > 1 ? std::atol(argv[1]) : 1 << 30;
  bsx::run_workers(kN, [&](size_t k) noexcept { done[k].fetch_add(1); });
  budget = 1 << 30;
  bool ok = true;
  for (std::atomic<int>& d : done) {
    std::printf("%d ", d.load());
    ok = ok && d.load() == 1;
  }
  std::printf("\n");
  return ok ? 0 : 1;
}
