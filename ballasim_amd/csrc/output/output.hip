// Kernels of the output stage: event build with crop and readout, key passes, a stable LSD radix sort,
// gather with the window cut, and the C4 columns.
#include <hip/hip_runtime.h>

#include "output_kernels.h"

namespace bsx {

// Exclusive scan of int32 counts into int64 offsets (defined with the scene kernels).
size_t scan_scratch_count(size_t n);
hipError_t launch_exclusive_scan(const int32_t* counts, size_t n, int64_t* out, int64_t* scratch, hipStream_t stream);

namespace {

// S1 class of a sensor label's two class bits (signal 0, noise 2, leak 3, hot 4; reference: label_s1,
// src/sensor/output_order.h:23-26).
__device__ __forceinline__ uint8_t label_s1(uint8_t c) {
  const uint8_t c3 = c & 3;
  return c3 == 0 ? 0 : static_cast<uint8_t>(c3 + 1);
}

constexpr uint64_t kBias = uint64_t{1} << 63;
constexpr int kOutBlock = 256;  // threads per block of the per-event kernels

// Raw events a block takes at once: one atomic on the kept count and one set on the extremes per 2,048 events
// (per 256 the atomics on one address set the time: 143 us and a separate 40-us pass over 2.9 M events).
constexpr int kBuildItems = 8;

__global__ void reset_kernel(unsigned long long* scratch) {
  if (threadIdx.x < kOutScratch)
    scratch[threadIdx.x] = threadIdx.x == kOutRepMin || threadIdx.x == kOutLagMin ? ~0ull : 0ull;
}

// The extremes of the reported times and of the lags t_cross - t_reported (biased to unsigned order) of a
// block's threads into scratch. Called by every thread of the block.
__device__ __forceinline__ void fold_extremes(unsigned long long a, unsigned long long b, unsigned long long c,
                                              unsigned long long d, unsigned long long* scratch) {
  __shared__ unsigned long long part[4][kOutBlock / 64];
  for (int off = 32; off > 0; off >>= 1) {
    a = min(a, static_cast<unsigned long long>(__shfl_xor(a, off)));
    b = max(b, static_cast<unsigned long long>(__shfl_xor(b, off)));
    c = min(c, static_cast<unsigned long long>(__shfl_xor(c, off)));
    d = max(d, static_cast<unsigned long long>(__shfl_xor(d, off)));
  }
  const int wave = threadIdx.x >> 6;
  if (__lane_id() == 0) {
    part[0][wave] = a;
    part[1][wave] = b;
    part[2][wave] = c;
    part[3][wave] = d;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < static_cast<int>(blockDim.x >> 6); ++w) {
      a = min(a, part[0][w]);
      b = max(b, part[1][w]);
      c = min(c, part[2][w]);
      d = max(d, part[3][w]);
    }
    if (a != ~0ull) {
      atomicMin(scratch + kOutRepMin, a);
      atomicMax(scratch + kOutRepMax, b);
      atomicMin(scratch + kOutLagMin, c);
      atomicMax(scratch + kOutLagMax, d);
    }
  }
}

// Appends the kept raw events at held[n_held ..] and folds the extremes of the new and the held events.
__global__ __launch_bounds__(kOutBlock) void build_kernel(const RawEventDev* raw, size_t n, uint32_t width, Readout r,
                                                          int crop, CropBox box, OutEventDev* held, size_t n_held,
                                                          unsigned long long* scratch) {
  unsigned long long a = ~0ull, b = 0ull, c = ~0ull, d = 0ull;
  const auto fold = [&](const OutEventDev& o) {
    const unsigned long long tr = static_cast<uint64_t>(o.t_reported) ^ kBias;
    const unsigned long long lag = static_cast<uint64_t>(o.t_cross - o.t_reported) ^ kBias;
    a = min(a, tr);
    b = max(b, tr);
    c = min(c, lag);
    d = max(d, lag);
  };
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n_held;
       i += static_cast<size_t>(gridDim.x) * blockDim.x)
    fold(held[i]);
  __shared__ unsigned int kept[kBuildItems * (kOutBlock / 64)];
  __shared__ unsigned long long block_base;
  const int lane = __lane_id(), wave = threadIdx.x >> 6;
  OutEventDev ev[kBuildItems];
  unsigned long long mask[kBuildItems];
  for (int k = 0; k < kBuildItems; ++k) {
    const size_t i = (static_cast<size_t>(blockIdx.x) * kBuildItems + k) * kOutBlock + threadIdx.x;
    bool keep = false;
    OutEventDev o{};
    if (i < n) {
      const RawEventDev e = raw[i];
      const int32_t x = static_cast<int32_t>(e.pixel % width), y = static_cast<int32_t>(e.pixel / width);
      keep = !crop || (x >= box.x0 && x < box.x1 && y >= box.y0 && y < box.y1);
      o.t_cross = e.t_cross;
      o.t_reported = reported_time(r, e.t_cross);
      o.x = static_cast<uint16_t>(x);
      o.y = static_cast<uint16_t>(y);
      o.flags = e.flags;
      o.p = e.polarity;
      o.label = label_s1(e.label);
      if (keep) fold(o);
    }
    ev[k] = o;
    mask[k] = __ballot(keep);
    if (lane == 0) kept[k * (kOutBlock / 64) + wave] = static_cast<unsigned int>(__popcll(mask[k]));
  }
  __syncthreads();
  // (the order of the kept events does not matter: the output key is unique)
  if (threadIdx.x == 0) {
    unsigned int total = 0;
    for (int q = 0; q < kBuildItems * (kOutBlock / 64); ++q) {
      const unsigned int w = kept[q];
      kept[q] = total;
      total += w;
    }
    block_base = total != 0 ? atomicAdd(scratch + kOutKept, static_cast<unsigned long long>(total)) : 0;
  }
  __syncthreads();
  for (int k = 0; k < kBuildItems; ++k) {
    if ((mask[k] >> lane) & 1ull)
      held[n_held + block_base + kept[k * (kOutBlock / 64) + wave] + __popcll(mask[k] & ((1ull << lane) - 1ull))] = ev[k];
  }
  fold_extremes(a, b, c, d, scratch);
}

// ---- The bucket sort -----------------------------------------------------------------------------
// The output order is the order of one integer key (OrderKey: t_reported, x, y and the lag t_cross -
// t_reported), unique per event. Its leading bits part the events into buckets of a few
// hundred (reported times spread over the window), counted and filled, and one block
// per bucket sorts its keys in LDS and writes the events in order: four short passes whatever the key's
// length, where the digit sort below makes ten of five kernels each (2.9 M events: 0.58 ms of kernels, and
// 50 launches in a window of any size). Keys of more than 64 bits, and a bucket of more than kBucketCap events
// (bursts; nothing is filled or sorted then), are left to the digit sort.
__device__ __forceinline__ uint64_t order_key(const OrderKey& k, const OutEventDev& o) {
  return order_key(k, o.t_reported, o.x, o.y, o.t_cross);
}

// Counted in LDS first, one global atomic per block and bucket: a flash that puts most of a window into a few buckets
// made an atomic per event on their few addresses (2.9 M events, all but 1 % in
// 10 us: a window and its flush 20.1 ms, 1.10 this way; spread over 8 ms 0.84 and 0.70).
__global__ __launch_bounds__(1024) void bucket_count_kernel(const OutEventDev* ev, size_t n, OrderKey k, int shift,
                                                            uint32_t buckets, uint32_t* counts) {
  extern __shared__ uint32_t hist[];  // [buckets]
  for (uint32_t b = threadIdx.x; b < buckets; b += blockDim.x) hist[b] = 0;
  __syncthreads();
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<size_t>(gridDim.x) * blockDim.x)
    atomicAdd(hist + bucket_of(order_key(k, ev[i]), shift, buckets), 1u);
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < buckets; b += blockDim.x) {
    const uint32_t c = hist[b];
    if (c != 0) atomicAdd(counts + b, c);
  }
}

// base[b] = cursor[b] = the events of the buckets before b; the largest bucket in scratch (one block).
__global__ __launch_bounds__(1024) void bucket_scan_kernel(const uint32_t* counts, int buckets, uint32_t* base,
                                                           uint32_t* cursor, unsigned long long* scratch) {
  __shared__ uint32_t wave_sum[16];
  __shared__ uint32_t carry;
  if (threadIdx.x == 0) carry = 0;
  uint32_t most = 0;
  for (int b0 = 0; b0 < buckets; b0 += 1024) {
    __syncthreads();
    const int b = b0 + threadIdx.x, lane = __lane_id(), wave = threadIdx.x >> 6;
    const uint32_t v = b < buckets ? counts[b] : 0;
    most = max(most, v);
    uint32_t inc = v;
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t o = __shfl_up(inc, off);
      if (lane >= off) inc += o;
    }
    if (lane == 63) wave_sum[wave] = inc;
    __syncthreads();
    uint32_t before = carry;
    for (int w = 0; w < wave; ++w) before += wave_sum[w];
    if (b < buckets) {
      base[b] = before + inc - v;
      cursor[b] = before + inc - v;
    }
    __syncthreads();
    if (threadIdx.x == 1023) carry = before + inc;
  }
  for (int off = 32; off > 0; off >>= 1) most = max(most, static_cast<uint32_t>(__shfl_xor(most, off)));
  if (__lane_id() == 0) atomicMax(scratch + kOutMostBucket, static_cast<unsigned long long>(most));
}

__global__ __launch_bounds__(256) void bucket_fill_kernel(const OutEventDev* ev, size_t n, OrderKey k, int shift,
                                                          uint32_t buckets, uint32_t* cursor, uint64_t* keys,
                                                          uint32_t* perm, const unsigned long long* scratch) {
  if (scratch[kOutMostBucket] > kBucketCap) return;  // left to the digit sort
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t key = order_key(k, ev[i]);
  const uint32_t slot = atomicAdd(cursor + bucket_of(key, shift, buckets), 1u);
  keys[slot] = key;
  perm[slot] = static_cast<uint32_t>(i);
}

// One block per bucket: its keys sorted in LDS (bitonic, padded to a power of two with the largest key), its
// events written in order and those reported before cut counted. With base null the events are one bucket,
// whose keys the block forms itself. With a bucket past kBucketCap nothing is sorted (the host sees the largest).
__global__ __launch_bounds__(256) void bucket_sort_kernel(const OutEventDev* ev, size_t n, OrderKey k,
                                                          const uint32_t* counts, const uint32_t* base,
                                                          const uint64_t* keys, const uint32_t* perm, int64_t cut,
                                                          OutEventDev* sorted, unsigned long long* scratch) {
  __shared__ uint64_t key[kBucketCap];
  __shared__ uint32_t idx[kBucketCap];
  __shared__ uint32_t ready;
  const uint32_t c = base != nullptr ? counts[blockIdx.x] : static_cast<uint32_t>(n);
  const uint32_t first = base != nullptr ? base[blockIdx.x] : 0;
  if (c == 0 || c > kBucketCap || scratch[kOutMostBucket] > kBucketCap) return;
  uint32_t size = 64;
  while (size < c) size <<= 1;
  if (threadIdx.x == 0) ready = 0;
  for (uint32_t i = threadIdx.x; i < size; i += 256) {
    const bool real = i < c;
    const uint32_t e = !real ? 0u : base != nullptr ? perm[first + i] : i;
    key[i] = !real ? ~0ull : base != nullptr ? keys[first + i] : order_key(k, ev[e]);
    idx[i] = real ? e : 0xffffffffu;  // (a real key of all ones sorts before the padding)
  }
  __syncthreads();
  for (uint32_t span = 2; span <= size; span <<= 1) {
    for (uint32_t step = span >> 1; step > 0; step >>= 1) {
      for (uint32_t q = threadIdx.x; q < size / 2; q += 256) {
        const uint32_t lo = 2 * q - (q & (step - 1)), hi = lo + step;
        const bool up = (lo & span) == 0;
        const uint64_t ka = key[lo], kb = key[hi];
        const uint32_t ia = idx[lo], ib = idx[hi];
        const bool above = ka > kb || (ka == kb && ia > ib);
        if (above == up) {
          key[lo] = kb;
          key[hi] = ka;
          idx[lo] = ib;
          idx[hi] = ia;
        }
      }
      __syncthreads();
    }
  }
  uint32_t mine = 0;
  for (uint32_t i = threadIdx.x; i < c; i += 256) {
    const OutEventDev o = ev[idx[i]];
    sorted[first + i] = o;
    mine += o.t_reported < cut ? 1u : 0u;
  }
  for (int off = 32; off > 0; off >>= 1) mine += __shfl_xor(mine, off);
  if (__lane_id() == 0 && mine != 0) atomicAdd(&ready, mine);
  __syncthreads();
  if (threadIdx.x == 0 && ready != 0) atomicAdd(scratch + kOutReady, static_cast<unsigned long long>(ready));
}

__global__ void fill_counts_kernel(uint32_t* counts, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) counts[i] = 0;
}

__global__ void keys_kernel(const OutEventDev* ev, const uint32_t* perm, uint32_t* perm_init, size_t n, int pass,
                            int y_bits, int64_t tc_min, int64_t tr_min, uint64_t* keys) {
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t e = static_cast<uint32_t>(i);
  if (perm != nullptr) e = perm[i];
  else if (perm_init != nullptr) perm_init[i] = e;
  const OutEventDev o = ev[e];
  keys[i] = pass == 0   ? static_cast<uint64_t>(o.t_cross - tc_min)
            : pass == 1 ? (static_cast<uint64_t>(o.x) << y_bits) | o.y
                        : static_cast<uint64_t>(o.t_reported - tr_min);
}

__global__ void gather_kernel(const OutEventDev* ev, const uint32_t* perm, size_t n, int64_t cut, OutEventDev* sorted,
                              unsigned long long* scratch) {
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  bool ready = false;
  if (i < n) {
    const OutEventDev o = ev[perm[i]];
    sorted[i] = o;
    ready = o.t_reported < cut;
  }
  __shared__ unsigned int wave_ready[kOutBlock / 64];
  const unsigned long long m = __ballot(ready);
  if (__lane_id() == 0) wave_ready[threadIdx.x >> 6] = static_cast<unsigned int>(__popcll(m));
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long total = 0;
    for (int w = 0; w < static_cast<int>(blockDim.x >> 6); ++w) total += wave_ready[w];
    if (total != 0) atomicAdd(scratch + kOutReady, total);
  }
}

__global__ void columns_kernel(const OutEventDev* ev, size_t n, int64_t t_offset_us, uint16_t* x, uint16_t* y,
                               uint8_t* p, int64_t* t_us, uint16_t* t_ns_rem, int64_t* t_rep, int64_t* t_cross,
                               uint8_t* label, uint16_t* flags) {
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const OutEventDev o = ev[i];
  const int64_t us = floor_div64(o.t_reported, 1000);
  x[i] = o.x;
  y[i] = o.y;
  p[i] = o.p;
  t_us[i] = us - t_offset_us;
  t_ns_rem[i] = static_cast<uint16_t>(o.t_reported - 1000 * us);
  t_rep[i] = o.t_reported;
  t_cross[i] = o.t_cross;
  label[i] = o.label;
  flags[i] = o.flags;
}

// The compact 16-byte records of ev[0 .. n) (one thread per event; 16-byte stores).
__global__ void pack_kernel(const OutEventDev* ev, size_t n, StreamEventDev* dst) {
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const OutEventDev o = ev[i];
  dst[i] = StreamEventDev{o.t_reported, o.x, o.y, o.p, o.label, o.flags};
}

// The radix sort: 8-bit digits, least significant first. A block owns a tile of kSortTile consecutive
// items (kSortItems per thread, item k * 256 + thread of the tile at step k, so that the block walks its
// tile in order). Per digit: every tile's digit histogram, written digit-major (hist[d * tiles + tile]);
// the exclusive scan of that array, which gives each (digit, tile) its first output slot with every
// smaller digit, and every earlier tile's equal digits, before it; then the scatter, in which each tile
// ranks its items stably (the wave's equal digits by an 8-ballot match, the earlier waves' through LDS
// counts) and writes them from its slots on.
constexpr int kSortBits = 8;
constexpr int kSortBins = 1 << kSortBits;
constexpr int kSortItems = 8;
constexpr int kSortTile = 256 * kSortItems;

__global__ __launch_bounds__(256) void digit_hist_kernel(const uint64_t* keys, size_t n, int shift, size_t tiles,
                                                         int32_t* hist) {
  __shared__ uint32_t h[kSortBins];
  h[threadIdx.x] = 0;
  __syncthreads();
  const size_t base = static_cast<size_t>(blockIdx.x) * kSortTile;
  for (int k = 0; k < kSortItems; ++k) {
    const size_t i = base + static_cast<size_t>(k) * 256 + threadIdx.x;
    if (i < n) atomicAdd(&h[(keys[i] >> shift) & (kSortBins - 1)], 1u);
  }
  __syncthreads();
  hist[static_cast<size_t>(threadIdx.x) * tiles + blockIdx.x] = static_cast<int32_t>(h[threadIdx.x]);
}

__global__ __launch_bounds__(256) void digit_scatter_kernel(const uint64_t* keys, const uint32_t* vals, size_t n,
                                                            int shift, size_t tiles, const int64_t* offsets,
                                                            uint64_t* keys_out, uint32_t* vals_out) {
  __shared__ uint32_t base[kSortBins];          // this tile's next free slot of each digit
  __shared__ uint32_t wave_count[4][kSortBins];  // the current step's items of each digit, per wave
  const int lane = __lane_id(), wave = threadIdx.x >> 6;
  base[threadIdx.x] = static_cast<uint32_t>(offsets[static_cast<size_t>(threadIdx.x) * tiles + blockIdx.x]);
  for (int w = 0; w < 4; ++w) wave_count[w][threadIdx.x] = 0;
  __syncthreads();
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  const size_t tile = static_cast<size_t>(blockIdx.x) * kSortTile;
  for (int k = 0; k < kSortItems; ++k) {
    const size_t i = tile + static_cast<size_t>(k) * 256 + threadIdx.x;
    const bool valid = i < n;
    uint64_t key = 0;
    uint32_t val = 0, d = 0;
    if (valid) {
      key = keys[i];
      val = vals[i];
      d = static_cast<uint32_t>((key >> shift) & (kSortBins - 1));
    }
    uint64_t peers = __ballot(valid);
    for (int b = 0; b < kSortBits; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t set = __ballot(bit);
      peers &= bit ? set : ~set;
    }
    const uint32_t rank = static_cast<uint32_t>(__popcll(peers & below));
    const bool leader = valid && rank == 0;
    if (leader) wave_count[wave][d] = static_cast<uint32_t>(__popcll(peers));
    __syncthreads();
    if (valid) {
      uint32_t slot = base[d] + rank;
      for (int w = 0; w < wave; ++w) slot += wave_count[w][d];
      keys_out[slot] = key;
      vals_out[slot] = val;
    }
    __syncthreads();
    base[threadIdx.x] += wave_count[0][threadIdx.x] + wave_count[1][threadIdx.x] + wave_count[2][threadIdx.x] +
                         wave_count[3][threadIdx.x];
    __syncthreads();
    if (leader) wave_count[wave][d] = 0;
  }
}

inline unsigned grid(size_t n) { return static_cast<unsigned>((n + kOutBlock - 1) / kOutBlock); }

}  // namespace

hipError_t launch_out_build(const RawEventDev* raw, size_t n, uint32_t width, const Readout& r, bool crop,
                            const CropBox& box, OutEventDev* held, size_t n_held, unsigned long long* scratch,
                            hipStream_t stream) {
  reset_kernel<<<1, 64, 0, stream>>>(scratch);
  if (n + n_held > 0) {
    const size_t tile = static_cast<size_t>(kOutBlock) * kBuildItems;
    // (blocks past the new events, up to a bound, stride over the held ones)
    const unsigned blocks = vmax(static_cast<unsigned>((n + tile - 1) / tile), vmin(grid(n_held), 512u));
    build_kernel<<<blocks, kOutBlock, 0, stream>>>(raw, n, width, r, crop ? 1 : 0, box, held, n_held, scratch);
  }
  return hipGetLastError();
}

hipError_t launch_out_buckets(const OutEventDev* ev, size_t n, const OrderKey& k, int bucket_bits, int64_t cut,
                              uint32_t* words, uint64_t* keys, uint32_t* perm, OutEventDev* sorted,
                              unsigned long long* scratch, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  if (bucket_bits == 0) {
    if (n > kBucketCap) return hipErrorInvalidValue;
    bucket_sort_kernel<<<1, 256, 0, stream>>>(ev, n, k, nullptr, nullptr, nullptr, nullptr, cut, sorted, scratch);
    return hipGetLastError();
  }
  const int buckets = 1 << bucket_bits;
  const int shift = vmax(0, k.bits() - bucket_bits);
  uint32_t *counts = words, *base = words + buckets, *cursor = words + 2 * buckets;
  fill_counts_kernel<<<(buckets + 255) / 256, 256, 0, stream>>>(counts, buckets);
  const unsigned count_blocks = static_cast<unsigned>(vmin<size_t>((n + 4095) / 4096, 512));  // two a compute unit
  bucket_count_kernel<<<count_blocks, 1024, buckets * sizeof(uint32_t), stream>>>(ev, n, k, shift,
                                                                                  static_cast<uint32_t>(buckets), counts);
  bucket_scan_kernel<<<1, 1024, 0, stream>>>(counts, buckets, base, cursor, scratch);
  bucket_fill_kernel<<<grid(n), 256, 0, stream>>>(ev, n, k, shift, static_cast<uint32_t>(buckets), cursor, keys, perm,
                                                  scratch);
  bucket_sort_kernel<<<buckets, 256, 0, stream>>>(ev, n, k, counts, base, keys, perm, cut, sorted, scratch);
  return hipGetLastError();
}

hipError_t launch_out_reset_ready(unsigned long long* scratch, hipStream_t stream) {
  fill_counts_kernel<<<1, 64, 0, stream>>>(reinterpret_cast<uint32_t*>(scratch + kOutReady), 2);
  return hipGetLastError();
}

hipError_t launch_out_keys(const OutEventDev* ev, const uint32_t* perm, uint32_t* perm_init, size_t n, int pass,
                           int y_bits, int64_t tc_min, int64_t tr_min, uint64_t* keys, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  keys_kernel<<<grid(n), 256, 0, stream>>>(ev, perm, perm_init, n, pass, y_bits, tc_min, tr_min, keys);
  return hipGetLastError();
}

hipError_t launch_out_sort(uint64_t* keys, uint64_t* keys_out, uint32_t* perm, uint32_t* perm_out, size_t n, int bits,
                           DeviceBuffer& temp, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  if (n >= (size_t{1} << 32) || bits < 1 || bits > 64) return hipErrorInvalidValue;
  const size_t tiles = (n + kSortTile - 1) / kSortTile;
  const size_t cells = tiles * kSortBins;
  const size_t scan_words = scan_scratch_count(cells);
  uint8_t* t = static_cast<uint8_t*>(temp.ensure(cells * 4 + cells * 8 + scan_words * 8));
  int32_t* hist = reinterpret_cast<int32_t*>(t);
  int64_t* offsets = reinterpret_cast<int64_t*>(t + cells * 4);
  int64_t* scan = reinterpret_cast<int64_t*>(t + cells * 12);
  uint64_t* k_src = keys;
  uint64_t* k_dst = keys_out;
  uint32_t* v_src = perm;
  uint32_t* v_dst = perm_out;
  for (int shift = 0; shift < bits; shift += kSortBits) {
    digit_hist_kernel<<<static_cast<unsigned>(tiles), 256, 0, stream>>>(k_src, n, shift, tiles, hist);
    hipError_t e = launch_exclusive_scan(hist, cells, offsets, scan, stream);
    if (e != hipSuccess) return e;
    digit_scatter_kernel<<<static_cast<unsigned>(tiles), 256, 0, stream>>>(k_src, v_src, n, shift, tiles, offsets,
                                                                           k_dst, v_dst);
    std::swap(k_src, k_dst);
    std::swap(v_src, v_dst);
  }
  if (v_src != perm_out) {  // an even number of digits: the sorted pairs are in the input buffers
    hipError_t e = hipMemcpyAsync(keys_out, keys, n * sizeof(uint64_t), hipMemcpyDeviceToDevice, stream);
    if (e == hipSuccess) e = hipMemcpyAsync(perm_out, perm, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, stream);
    if (e != hipSuccess) return e;
  }
  return hipGetLastError();
}

hipError_t launch_out_gather(const OutEventDev* ev, const uint32_t* perm, size_t n, int64_t cut, OutEventDev* sorted,
                             unsigned long long* scratch, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  gather_kernel<<<grid(n), kOutBlock, 0, stream>>>(ev, perm, n, cut, sorted, scratch);
  return hipGetLastError();
}

hipError_t launch_out_columns(const OutEventDev* ev, size_t n, int64_t t_offset_us, uint16_t* x, uint16_t* y,
                              uint8_t* p, int64_t* t_us, uint16_t* t_ns_rem, int64_t* t_rep, int64_t* t_cross,
                              uint8_t* label, uint16_t* flags, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  columns_kernel<<<grid(n), 256, 0, stream>>>(ev, n, t_offset_us, x, y, p, t_us, t_ns_rem, t_rep, t_cross, label,
                                              flags);
  return hipGetLastError();
}

hipError_t launch_out_pack(const OutEventDev* ev, size_t n, StreamEventDev* dst, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  pack_kernel<<<grid(n), 256, 0, stream>>>(ev, n, dst);
  return hipGetLastError();
}

}  // namespace bsx
