// The output stage's host side: window and flush orchestration over output.hip's kernels.
#include "output.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <stdexcept>
#include <string>

#include "../core/workers.h"
#include "output_kernels.h"

namespace bsx {

void OutputColumns::resize(size_t n) {
  x.resize(n);
  y.resize(n);
  p.resize(n);
  t_us.resize(n);
  t_ns_rem.resize(n);
  t_reported.resize(n);
  t_cross.resize(n);
  label.resize(n);
  flags.resize(n);
}

OutputStage::OutputStage(uint32_t width, uint32_t height, const Readout& readout, const CropBox* crop,
                         int64_t t_offset_us)
    : width_(width), height_(height), readout_(readout), crop_on_(crop != nullptr), t_offset_us_(t_offset_us) {
  if (width == 0 || height == 0) throw std::invalid_argument("OutputStage: empty camera");
  if (crop != nullptr) {
    if (!(crop->x0 >= 0 && crop->y0 >= 0 && crop->x0 < crop->x1 && crop->y0 < crop->y1 &&
          crop->x1 <= static_cast<int32_t>(width) && crop->y1 <= static_cast<int32_t>(height))) {
      throw std::invalid_argument("OutputStage: the crop must lie inside the frame and be non-empty");
    }
    crop_ = *crop;
  }
  y_bits_ = 1;
  while ((uint64_t{1} << y_bits_) < height) ++y_bits_;
  x_bits_ = 1;
  while ((uint64_t{1} << x_bits_) < width) ++x_bits_;
  scratch_.ensure(kOutScratch * 8);
  hip_check(hipHostMalloc(reinterpret_cast<void**>(&h_scratch_), kOutScratch * 8, hipHostMallocDefault), "scratch");
}

OutputStage::~OutputStage() {
  if (h_scratch_ != nullptr) (void)hipHostFree(h_scratch_);
  if (staging_ != nullptr) (void)hipHostFree(staging_);
}

void OutputStage::read_scratch(hipStream_t stream) {
  hip_check(hipMemcpyAsync(h_scratch_, scratch_.get(), kOutScratch * 8, hipMemcpyDeviceToHost, stream),
            "read scratch");
  hip_check(hipStreamSynchronize(stream), "output stage");
}

size_t OutputStage::take(const RawEventDev* raw, size_t n, hipStream_t stream) {
  if (n > 0 && raw == nullptr) throw std::invalid_argument("OutputStage.window: null events");
  const size_t n_max = n_held_ + n;
  if (n_max > 0xffffffffull) throw std::invalid_argument("OutputStage.window: at most 2^32 - 1 events");
  released_ = 0;
  // The held events stay at the front of held_; the window's kept events are appended after them.
  if (held_.bytes() < std::max<size_t>(n_max, 1) * sizeof(OutEventDev)) {
    DeviceBuffer grown;
    grown.ensure(std::max<size_t>(n_max + n_max / 2, 1024) * sizeof(OutEventDev));
    if (n_held_ > 0) {
      hip_check(hipMemcpyAsync(grown.get(), held_.get(), n_held_ * sizeof(OutEventDev), hipMemcpyDeviceToDevice,
                               stream),
                "grow held");
    }
    hip_check(hipStreamSynchronize(stream), "grow held");
    held_.swap(grown);
  }
  hip_check(launch_out_build(raw, n, width_, readout_, crop_on_, crop_, held_.as<OutEventDev>(), n_held_,
                             scratch_.as<unsigned long long>(), stream),
            "build events");
  read_scratch(stream);
  return n_held_ + static_cast<size_t>(h_scratch_[kOutKept]);
}

const OutputColumns& OutputStage::window(const RawEventDev* raw, size_t n, int64_t t_w, hipStream_t stream) {
  const OutEventDev* ev = nullptr;
  return download(window_device(raw, n, t_w, stream, &ev), stream);
}

const OutputColumns& OutputStage::flush(hipStream_t stream) {
  const OutEventDev* ev = nullptr;
  return download(flush_device(stream, &ev), stream);
}

size_t OutputStage::window_device(const RawEventDev* raw, size_t n, int64_t t_w, hipStream_t stream,
                                  const OutEventDev** released) {
  const size_t m = release_sorted(take(raw, n, stream), output_cut(readout_, t_w + kPlainSegmentNs), stream);
  *released = sorted_.as<const OutEventDev>();
  return m;
}

size_t OutputStage::flush_device(hipStream_t stream, const OutEventDev** released) {
  const size_t m = release_sorted(take(nullptr, 0, stream), INT64_MAX, stream);
  *released = sorted_.as<const OutEventDev>();
  return m;
}

size_t OutputStage::release_sorted(size_t total, int64_t cut, hipStream_t stream) {
  if (total == 0) {
    n_held_ = 0;
    return 0;
  }
  const uint64_t bias = uint64_t{1} << 63;
  const auto unbias = [&](int k) { return static_cast<int64_t>(h_scratch_[k] ^ bias); };
  const int64_t tr_min = unbias(kOutRepMin), tr_max = unbias(kOutRepMax);
  const int64_t lag_min = unbias(kOutLagMin), lag_max = unbias(kOutLagMax);
  const OutEventDev* ev = held_.as<const OutEventDev>();
  sorted_.ensure(total * sizeof(OutEventDev));
  const OrderKey key = order_key_of(readout_, tr_min, tr_max, lag_min, lag_max, x_bits_, y_bits_);
  const int bb = key.bits() > 64 ? -1
                                 : out_bucket_bits(total, key, report_count(readout_, tr_min, tr_max),
                                                   crop_on_ ? static_cast<uint32_t>(crop_.x1 - crop_.x0) : width_,
                                                   crop_on_ ? static_cast<uint32_t>(crop_.y1 - crop_.y0) : height_);
  bool done = false;
  if (bb >= 0) {
    if (bb > 0) {
      keys_.ensure(total * 8);
      perm_.ensure(total * 4);
      buckets_.ensure((size_t{3} << bb) * 4);
    }
    hip_check(launch_out_buckets(ev, total, key, bb, cut, buckets_.as<uint32_t>(), keys_.as<uint64_t>(),
                                 perm_.as<uint32_t>(), sorted_.as<OutEventDev>(), scratch_.as<unsigned long long>(),
                                 stream),
              "bucket sort");
    read_scratch(stream);
    done = h_scratch_[kOutMostBucket] <= kBucketCap;
  }
  if (!done) {
    sort_digits(total, cut, tr_min, tr_max, tr_min + lag_min, tr_max + lag_max, stream);
    read_scratch(stream);
  }
  const size_t m = static_cast<size_t>(h_scratch_[kOutReady]);
  // The unreleased rest, in output order, becomes the held buffer.
  n_held_ = total - m;
  if (n_held_ > 0) {
    hip_check(hipMemcpyAsync(held_.get(), sorted_.as<OutEventDev>() + m, n_held_ * sizeof(OutEventDev),
                             hipMemcpyDeviceToDevice, stream),
              "hold");
  }
  released_ = m;
  return m;
}

void OutputStage::sort_digits(size_t total, int64_t cut, int64_t tr_min, int64_t tr_max, int64_t tc_min, int64_t tc_max,
                              hipStream_t stream) {
  const OutEventDev* ev = held_.as<const OutEventDev>();
  keys_.ensure(total * 8);
  keys_alt_.ensure(total * 8);
  perm_.ensure(total * 4);
  perm_alt_.ensure(total * 4);
  hip_check(launch_out_reset_ready(scratch_.as<unsigned long long>(), stream), "reset");
  // Three stable passes, least significant first: t_cross, (x, y), t_reported.
  const int bits[3] = {std::max(1, bit_length(static_cast<uint64_t>(tc_max - tc_min))), 16 + y_bits_,
                       std::max(1, bit_length(static_cast<uint64_t>(tr_max - tr_min)))};
  for (int pass = 0; pass < 3; ++pass) {
    hip_check(launch_out_keys(ev, pass == 0 ? nullptr : perm_.as<const uint32_t>(),
                              pass == 0 ? perm_.as<uint32_t>() : nullptr, total, pass, y_bits_, tc_min, tr_min,
                              keys_.as<uint64_t>(), stream),
              "sort keys");
    hip_check(launch_out_sort(keys_.as<uint64_t>(), keys_alt_.as<uint64_t>(), perm_.as<uint32_t>(),
                              perm_alt_.as<uint32_t>(), total, bits[pass], temp_, stream),
              "radix sort");
    perm_.swap(perm_alt_);
  }
  hip_check(launch_out_gather(ev, perm_.as<const uint32_t>(), total, cut, sorted_.as<OutEventDev>(),
                              scratch_.as<unsigned long long>(), stream),
            "gather");
}

namespace {

constexpr size_t kCopyBytes = size_t{1} << 20;  // of a staging slot
constexpr int kCopyThreads = 6;                 // of a large copy, two slots each
constexpr int kCopySlots = 2 * kCopyThreads;

}  // namespace

// A device-to-host copy into ordinary memory goes through the runtime's own staging on one thread, and fresh
// pages fault in as it writes (2.9 M events, 98 MB of columns: 13-17 ms with a second copy by the caller). Here
// each of a few threads copies its chunks to pinned slots of its own and from there to their places, the next
// chunk's transfer under way meanwhile, so that the transfers, the copies and the page faults overlap. Up to two
// slots' bytes the calling thread does it alone, and so it does where the caller names its stream by
// hipStreamPerThread: that handle is another stream in each thread, on which a transfer would not wait for the columns.
void OutputStage::copy_out(const char* from, const std::vector<Piece>& dst, size_t bytes, hipStream_t stream) {
  const size_t chunks = (bytes + kCopyBytes - 1) / kCopyBytes;
  const bool alone = chunks <= 2 || stream == hipStreamPerThread;
  const int slots = alone ? 2 : kCopySlots;
  if (slots > staging_slots_) {
    if (staging_ != nullptr) hip_check(hipHostFree(staging_), "staging");
    staging_ = nullptr;
    staging_slots_ = 0;
    hip_check(hipHostMalloc(reinterpret_cast<void**>(&staging_), slots * kCopyBytes, hipHostMallocDefault), "staging");
    staging_slots_ = slots;
  }
  const auto place = [&](size_t at, const char* src, size_t n) {  // bytes [at, at + n) of the copy to their places
    size_t start = 0;
    for (const Piece& p : dst) {
      const size_t lo = std::max(at, start), hi = std::min(at + n, start + p.bytes);
      if (lo < hi) std::memcpy(p.to + (lo - start), src + (lo - at), hi - lo);
      start += p.bytes;
    }
  };
  if (chunks == 1) {
    hip_check(hipMemcpyAsync(staging_, from, bytes, hipMemcpyDeviceToHost, stream), "download columns");
    hip_check(hipStreamSynchronize(stream), "download columns");
    place(0, staging_, bytes);
    return;
  }
  const auto run = [&](size_t first, size_t step, char* slots) {
    hipEvent_t landed[2] = {nullptr, nullptr};
    hipError_t e = hipEventCreateWithFlags(&landed[0], hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&landed[1], hipEventDisableTiming);
    const auto size_of = [&](size_t c) { return std::min(kCopyBytes, bytes - c * kCopyBytes); };
    const auto start = [&](size_t c, int s) {
      if (e == hipSuccess) {
        e = hipMemcpyAsync(slots + s * kCopyBytes, from + c * kCopyBytes, size_of(c), hipMemcpyDeviceToHost, stream);
      }
      if (e == hipSuccess) e = hipEventRecord(landed[s], stream);
    };
    int s = 0;
    if (first < chunks) start(first, s);
    for (size_t c = first; c < chunks && e == hipSuccess; c += step, s ^= 1) {
      if (c + step < chunks) start(c + step, s ^ 1);
      if (e == hipSuccess) e = hipEventSynchronize(landed[s]);
      if (e == hipSuccess) place(c * kCopyBytes, slots + s * kCopyBytes, size_of(c));
    }
    // (after an error a transfer may still be writing the slots)
    if (e != hipSuccess) (void)hipStreamSynchronize(stream);
    for (hipEvent_t& ev : landed)
      if (ev != nullptr) (void)hipEventDestroy(ev);
    return e;
  };
  if (alone) {
    hip_check(run(0, 1, staging_), "download columns");
    return;
  }
  int device = 0;
  hip_check(hipGetDevice(&device), "device");
  const size_t n_threads = std::min<size_t>(kCopyThreads, (chunks + 1) / 2);
  std::atomic<int> error{hipSuccess};
  run_workers(n_threads, [&](size_t k) noexcept {
    hipError_t e = hipSetDevice(device);
    if (e == hipSuccess) e = run(k, n_threads, staging_ + 2 * k * kCopyBytes);
    if (e != hipSuccess) error.store(e);
  });
  hip_check(static_cast<hipError_t>(error.load()), "download columns");
}

void OutputStage::fetch(const OutputColumnsDst& d, hipStream_t stream) {
  const size_t m = released_;
  if (m == 0) return;
  // The columns one after another, the widest first (each is then aligned for its type).
  columns_.ensure(m * 34);
  char* b = static_cast<char*>(columns_.get());
  char* const first = b;
  std::vector<Piece> pieces;
  const auto column = [&](auto* to) {
    if (to == nullptr) throw std::invalid_argument("OutputStage.fetch: null column");
    using T = std::remove_pointer_t<decltype(to)>;
    T* at = reinterpret_cast<T*>(b);
    b += m * sizeof(T);
    pieces.push_back(Piece{reinterpret_cast<char*>(to), m * sizeof(T)});
    return at;
  };
  int64_t *t_us = column(d.t_us), *t_rep = column(d.t_reported), *t_cross = column(d.t_cross);
  uint16_t *x = column(d.x), *y = column(d.y), *rem = column(d.t_ns_rem), *flags = column(d.flags);
  uint8_t *p = column(d.p), *label = column(d.label);
  hip_check(launch_out_columns(sorted_.as<const OutEventDev>(), m, t_offset_us_, x, y, p, t_us, rem, t_rep, t_cross,
                               label, flags, stream),
            "columns");
  copy_out(first, pieces, static_cast<size_t>(b - first), stream);
}

const OutputColumns& OutputStage::download(size_t m, hipStream_t stream) {
  out_.resize(m);
  fetch(OutputColumnsDst{out_.x.data(), out_.y.data(), out_.p.data(), out_.t_us.data(), out_.t_ns_rem.data(),
                         out_.t_reported.data(), out_.t_cross.data(), out_.label.data(), out_.flags.data()},
        stream);
  return out_;
}

}  // namespace bsx
