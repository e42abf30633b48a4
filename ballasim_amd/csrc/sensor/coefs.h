// How much device memory a camera's segment coefficients may take.
#pragma once

#include <stddef.h>

namespace bsx {

// Bytes to hold for a call that needs `need`, of which `have` are held, with `free` bytes of device memory free: up to
// 32 GiB and up to a quarter of the memory that is free without the buffer, the rest being the caller's to use; when it
// grows, a quarter more than needed as far as that goes, so that windows that differ a little in size do not each free
// and allocate gigabytes. 0: the call goes without coefficients, and the walk forms them itself (the same values).
inline size_t coef_bytes(size_t need, size_t have, size_t free) {
  constexpr size_t kMost = size_t{32} << 30;
  if (need <= have) return have;
  const size_t share = (free + have) / 4, limit = share < kMost ? share : kMost;
  if (need > limit) return 0;
  const size_t roomy = need + need / 4;
  return roomy < limit ? roomy : limit;
}

}  // namespace bsx
