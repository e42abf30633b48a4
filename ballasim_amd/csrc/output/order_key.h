// The output order (t_reported, x, y, t_cross) as the order of one integer, and how its leading bits part the
// events into buckets.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "../core/hd.h"
#include "../sensor/readout.h"

namespace bsx {

// t_reported - rep_min without its rep_shift low bits, x, y and the lag t_cross - t_reported less lag_min, from the
// leading bits down.
struct OrderKey {
  int64_t rep_min, lag_min;
  int32_t rep_shift, rep_bits, x_bits, y_bits, lag_bits;
  BSX_HD int bits() const { return rep_bits + x_bits + y_bits + lag_bits; }
};

BSX_HD BSX_INLINE uint64_t order_key(const OrderKey& k, int64_t t_reported, uint32_t x, uint32_t y, int64_t t_cross) {
  const uint64_t rep = static_cast<uint64_t>(t_reported - k.rep_min) >> k.rep_shift;
  return (((((rep << k.x_bits) | x) << k.y_bits) | y) << k.lag_bits) |
         static_cast<uint64_t>((t_cross - t_reported) - k.lag_min);
}

inline int bit_length(uint64_t v) {
  int b = 0;
  while (v != 0) {
    ++b;
    v >>= 1;
  }
  return b;
}

// The low bits of a reported time's distance to the earliest one that the order does not need: a quantum leaves
// different reports at least `gap` apart (the drift stretches the quantum and rounds each of them once, after a double
// product off by at most 2^12 |drift| ns for any 64-bit time), so those whose quotients by 2^shift <= gap are equal
// are equal. With the raw nanoseconds as the key's leading bits a quantum of 20 us put a window's 2.9 M events into
// 1 of 40 buckets, each past what a block sorts, and the digit sort ran after all (a window and its flush to a stream
// 2.26 ms, 0.98 this way, 1.52 by the digit sort alone; at 1 ms 1.46, 1.27 and 1.51).
inline int report_shift(const Readout& r) {
  if (r.quantum_ns <= 1) return 0;
  const double drift = r.clock_drift_ppm * 1e-6;
  const double gap = drift == 0.0 ? static_cast<double>(r.quantum_ns)
                                  : fabs(1.0 + drift) * static_cast<double>(r.quantum_ns) - 2.0 - 4096.0 * fabs(drift);
  int s = 0;
  while (s < 62 && static_cast<double>(int64_t{2} << s) <= gap) ++s;
  return s;
}

// The key of events whose reported times and lags lie in the given ranges.
inline OrderKey order_key_of(const Readout& r, int64_t rep_min, int64_t rep_max, int64_t lag_min, int64_t lag_max,
                             int x_bits, int y_bits) {
  const int shift = report_shift(r);
  return OrderKey{rep_min,
                  lag_min,
                  shift,
                  bit_length((static_cast<uint64_t>(rep_max) - static_cast<uint64_t>(rep_min)) >> shift),
                  x_bits,
                  y_bits,
                  bit_length(static_cast<uint64_t>(lag_max) - static_cast<uint64_t>(lag_min))};
}

// Events a block sorts at once, and the most buckets.
inline constexpr int kBucketCap = 2048, kMaxBucketBits = 14;

// The reports that a window's range of reported times can hold.
inline double report_count(const Readout& r, int64_t rep_min, int64_t rep_max) {
  const double range = static_cast<double>(static_cast<uint64_t>(rep_max) - static_cast<uint64_t>(rep_min));
  return (r.quantum_ns > 1 ? range / static_cast<double>(r.quantum_ns) : range) + 1.0;
}

// The buckets of n events (as a power of two; 0: one block takes them all): as many as leave 512 to each bucket that
// events of `reports` reported times and a crop of width x height pixels can reach. (Of a field that the bucket's bits
// touch only the values in use are reached: of 2,048 buckets that 900,000 events over 1280x720 and nine reports were
// parted into, 360.) -1: more events than blocks could sort if they were spread evenly, the digit sort's (20 M events
// over 8 ms and 2048x1536 pixels took 10.4 ms with the bucket passes in vain, 7.2 without).
inline int out_bucket_bits(size_t n, const OrderKey& k, double reports, uint32_t width, uint32_t height) {
  if (n <= kBucketCap) return 0;
  const auto share = [](double values, int bits) {
    return bits >= 63 ? 1.0 : vmin(1.0, values / static_cast<double>(int64_t{1} << bits));
  };
  for (int b = 1; b <= kMaxBucketBits; ++b) {
    double reached = static_cast<double>(1 << b);
    reached *= share(reports, k.rep_bits);
    if (b > k.rep_bits) reached *= share(width, k.x_bits);
    if (b > k.rep_bits + k.x_bits) reached *= share(height, k.y_bits);
    if (static_cast<double>(n) <= 512.0 * reached) return b;
    if (b == kMaxBucketBits && static_cast<double>(n) > static_cast<double>(kBucketCap) * reached) return -1;
  }
  return kMaxBucketBits;
}

// (clamped: an event outside the frame has a key past the others')
BSX_HD BSX_INLINE uint32_t bucket_of(uint64_t key, int shift, uint32_t buckets) {
  const uint64_t b = key >> shift;
  return b < buckets ? static_cast<uint32_t>(b) : buckets - 1;
}

}  // namespace bsx
