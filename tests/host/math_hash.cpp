// math_hash FN FIRST LAST STRIDE: the sum of math_hash(FN, u) over u = FIRST, FIRST + STRIDE, ... <= LAST, with
// the host's plain divisions (core/math_check.h).
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

#include "math_check.h"

int main(int argc, char** argv) {
  if (argc != 5) return 2;
  const int fn = std::atoi(argv[1]);
  const uint64_t first = std::strtoull(argv[2], nullptr, 10), last = std::strtoull(argv[3], nullptr, 10),
                 stride = std::strtoull(argv[4], nullptr, 10);
  constexpr int kThreads = 8;
  std::vector<uint64_t> part(kThreads, 0);
  std::vector<std::thread> pool;
  for (int w = 0; w < kThreads; ++w)
    pool.emplace_back([&, w] {
      uint64_t h = 0;
      for (uint64_t u = first + w * stride; u <= last; u += kThreads * stride)
        h += bsx::math_hash(fn, static_cast<uint32_t>(u));
      part[w] = h;
    });
  for (std::thread& t : pool) t.join();
  uint64_t h = 0;
  for (const uint64_t p : part) h += p;
  std::printf("%llu\n", static_cast<unsigned long long>(h));
  return 0;
}
