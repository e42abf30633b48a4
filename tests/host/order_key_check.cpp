// The output stage's one-integer order on the host.
//   order TRIALS SEED: over random readouts (quanta, delays, phases, drifts of either sign, early and late times) and
//     events that crowd a few reports, pixels and times, the order of the keys is the lexicographic order
//     (t_reported, x, y, t_cross), and keys are equal only where all four are.
//   fill N WIDTH HEIGHT QUANTUM_NS DRIFT_PPM: the largest bucket of N events spread evenly over the frame and a
//     window of 2^23 ns.
// Exit status 1 on any difference.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <tuple>
#include <vector>

#include "order_key.h"

using bsx::OrderKey;
using bsx::Readout;

struct Event {
  int64_t rep;
  uint32_t x, y;
  int64_t cross;
  auto tie() const { return std::tie(rep, x, y, cross); }
};

static int bits_for(uint32_t v) {
  int b = 1;
  while ((uint64_t{1} << b) < v) ++b;
  return b;
}

static OrderKey key_of(const Readout& r, const std::vector<Event>& ev, uint32_t w, uint32_t h) {
  int64_t r0 = INT64_MAX, r1 = INT64_MIN, l0 = INT64_MAX, l1 = INT64_MIN;
  for (const Event& e : ev) {
    r0 = std::min(r0, e.rep), r1 = std::max(r1, e.rep);
    l0 = std::min(l0, e.cross - e.rep), l1 = std::max(l1, e.cross - e.rep);
  }
  return bsx::order_key_of(r, r0, r1, l0, l1, bits_for(w), bits_for(h));
}

static int order(int trials, unsigned long long seed) {
  std::mt19937_64 rng(seed);
  const auto below = [&](uint64_t n) { return rng() % n; };
  const double drifts[] = {0.0, 35.0, -35.0, -4000.0, 250000.0, -999999.0, -1000000.0, -2500000.0, 3e6};
  const int64_t quanta[] = {0, 1, 2, 3, 8, 250, 1000, 6001, 20000, 1000000, 33333333, 1000000000};
  long long used = 0, shifted = 0, wide = 0, bad = 0;
  for (int k = 0; k < trials; ++k) {
    Readout r{};
    r.quantum_ns = quanta[below(12)];
    r.delay_ns = r.quantum_ns + static_cast<int64_t>(below(2) * below(1000000));
    r.phase_ns = r.quantum_ns > 0 ? static_cast<int64_t>(below(static_cast<uint64_t>(r.quantum_ns))) : 0;
    r.clock_offset_ns = static_cast<int64_t>(below(3)) * 12345 - 12345;
    r.clock_drift_ppm = drifts[below(9)];
    const int64_t origin = below(3) == 0 ? int64_t{1} << (30 + below(31)) : 0;
    const int64_t span = int64_t{1} << (1 + below(30));
    const uint32_t w = 1 + static_cast<uint32_t>(below(below(2) ? 8 : 4096)), h = 1 + static_cast<uint32_t>(below(below(2) ? 4 : 2048));
    std::vector<Event> ev(300);
    for (Event& e : ev) {
      e.cross = origin + static_cast<int64_t>(below(static_cast<uint64_t>(span)));
      e.rep = bsx::reported_time(r, e.cross);
      e.x = static_cast<uint32_t>(below(w));
      e.y = static_cast<uint32_t>(below(h));
    }
    const OrderKey q = key_of(r, ev, w, h);
    if (q.bits() > 64) {
      ++wide;
      continue;
    }
    ++used;
    shifted += q.rep_shift > 0;
    std::sort(ev.begin(), ev.end(), [](const Event& a, const Event& b) { return a.tie() < b.tie(); });
    const auto key = [&](const Event& e) { return bsx::order_key(q, e.rep, e.x, e.y, e.cross); };
    for (size_t i = 1; i < ev.size(); ++i) {
      const uint64_t a = key(ev[i - 1]), b = key(ev[i]);
      const bool equal = ev[i - 1].tie() == ev[i].tie();
      if (equal ? a != b : a >= b) {
        if (bad++ < 5)
          std::printf("quantum %lld drift %g: %lld %u %u %lld -> %llx, then %lld %u %u %lld -> %llx\n",
                      (long long)r.quantum_ns, r.clock_drift_ppm, (long long)ev[i - 1].rep, ev[i - 1].x, ev[i - 1].y,
                      (long long)ev[i - 1].cross, (unsigned long long)a, (long long)ev[i].rep, ev[i].x, ev[i].y,
                      (long long)ev[i].cross, (unsigned long long)b);
      }
    }
  }
  std::printf("trials %lld shifted %lld wide %lld differences %lld\n", used, shifted, wide, bad);
  return bad != 0;
}

static int fill(size_t n, uint32_t w, uint32_t h, int64_t quantum, double drift) {
  std::mt19937_64 rng(n);
  Readout r{};
  r.quantum_ns = r.delay_ns = quantum;
  r.phase_ns = quantum / 3;
  r.clock_drift_ppm = drift;
  std::vector<Event> ev(n);
  for (Event& e : ev) {
    e.cross = static_cast<int64_t>(rng() % (1 << 23));
    e.rep = bsx::reported_time(r, e.cross);
    e.x = static_cast<uint32_t>(rng() % w);
    e.y = static_cast<uint32_t>(rng() % h);
  }
  const OrderKey q = key_of(r, ev, w, h);
  int64_t r0 = INT64_MAX, r1 = INT64_MIN;
  for (const Event& e : ev) r0 = std::min(r0, e.rep), r1 = std::max(r1, e.rep);
  const int bb = bsx::out_bucket_bits(n, q, bsx::report_count(r, r0, r1), w, h);
  if (bb < 0) {
    std::printf("too many\n");
    return 0;
  }
  const int shift = std::max(0, q.bits() - bb);
  std::vector<uint32_t> count(size_t{1} << bb);
  for (const Event& e : ev) ++count[bsx::bucket_of(bsx::order_key(q, e.rep, e.x, e.y, e.cross), shift, 1u << bb)];
  std::printf("key bits %d buckets %d largest %u cap %d\n", q.bits(), 1 << bb, *std::max_element(count.begin(), count.end()),
              bsx::kBucketCap);
  return 0;
}

int main(int argc, char** argv) {
  if (argc >= 4 && std::strcmp(argv[1], "order") == 0) return order(std::atoi(argv[2]), std::strtoull(argv[3], nullptr, 10));
  if (argc >= 7 && std::strcmp(argv[1], "fill") == 0) {
    return fill(std::strtoull(argv[2], nullptr, 10), std::atoi(argv[3]), std::atoi(argv[4]), std::atoll(argv[5]),
                std::atof(argv[6]));
  }
  return 2;
}
