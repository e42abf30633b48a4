// Launch wrappers of the output stage's kernels (output.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "order_key.h"
#include "output.h"

namespace bsx {

// scratch words: the kept new events, the extremes of t_reported and of the lag t_cross - t_reported over the
// held and new events (biased to unsigned order), the released events, the largest bucket.
enum OutScratch : int { kOutKept, kOutRepMin, kOutRepMax, kOutLagMin, kOutLagMax, kOutReady, kOutMostBucket, kOutScratch };

// Resets scratch, appends the kept raw events as OutEventDev at held[n_held ..] and folds the extremes.
hipError_t launch_out_build(const RawEventDev* raw, size_t n, uint32_t width, const Readout& r, bool crop,
                            const CropBox& box, OutEventDev* held, size_t n_held, unsigned long long* scratch,
                            hipStream_t stream);
// The bucket sort of ev[0 .. n) into sorted by a key of at most 64 bits, the events reported before cut counted:
// 2^bucket_bits buckets (0: n events fit one block), words holds 3 << bucket_bits. Complete
// when the largest bucket (scratch) is at most kBucketCap.
hipError_t launch_out_buckets(const OutEventDev* ev, size_t n, const OrderKey& k, int bucket_bits, int64_t cut,
                              uint32_t* words, uint64_t* keys, uint32_t* perm, OutEventDev* sorted,
                              unsigned long long* scratch, hipStream_t stream);
hipError_t launch_out_reset_ready(unsigned long long* scratch, hipStream_t stream);
// keys[i] of pass (0: t_cross - tc_min, 1: (x << y_bits) | y, 2: t_reported - tr_min) of ev[perm[i]] (perm
// null: identity, perm_init filled with it).
hipError_t launch_out_keys(const OutEventDev* ev, const uint32_t* perm, uint32_t* perm_init, size_t n, int pass,
                           int y_bits, int64_t tc_min, int64_t tr_min, uint64_t* keys, hipStream_t stream);
// Stable radix sort of (keys, perm) by the key's low `bits` bits (n < 2^32); the sorted copies land in keys_out /
// perm_out, and keys / perm are overwritten.
hipError_t launch_out_sort(uint64_t* keys, uint64_t* keys_out, uint32_t* perm, uint32_t* perm_out, size_t n, int bits,
                           DeviceBuffer& temp, hipStream_t stream);
// sorted[i] = ev[perm[i]], counting those reported before cut into scratch.
hipError_t launch_out_gather(const OutEventDev* ev, const uint32_t* perm, size_t n, int64_t cut, OutEventDev* sorted,
                             unsigned long long* scratch, hipStream_t stream);
// The C4 columns of ev[0 .. n).
hipError_t launch_out_columns(const OutEventDev* ev, size_t n, int64_t t_offset_us, uint16_t* x, uint16_t* y,
                              uint8_t* p, int64_t* t_us, uint16_t* t_ns_rem, int64_t* t_rep, int64_t* t_cross,
                              uint8_t* label, uint16_t* flags, hipStream_t stream);

// The compact stream records of ev[0 .. n) at dst.
hipError_t launch_out_pack(const OutEventDev* ev, size_t n, StreamEventDev* dst, hipStream_t stream);

}  // namespace bsx
