// The fp32 functions of pmath.h by number, and an order-independent hash of their results over a range
// of bit patterns: the device's forms (divisions by reciprocal and remainder, hardware splitting and
// scaling) are compared with the host's plain ones this way.
#pragma once

#include "pmath.h"

namespace bsx {

inline constexpr int kMathFunctions = 12;

BSX_HD inline float math_function(int fn, float x) {
  switch (fn) {
    case 0: return pm::log(x);
    case 1: return pm::exp(x);
    case 2: return pm::erfcx(x);
    case 3: return pm::dawson(x);
    case 4: return pm::resid_exp<1>(x);
    case 5: return pm::resid_exp<2>(x);
    case 6: return pm::resid_exp<3>(x);
    case 7: return pm::resid_exp<4>(x);
    case 8: return pm::recip_any(x);
    case 9: return pm::div_by_any<3>(x);
    case 10: return pm::div_by_any<6>(x);
    default: return pm::div_by_any<384>(x);
  }
}

// (every NaN hashes alike)
BSX_HD inline uint64_t math_hash(int fn, uint32_t u) {
  const float y = math_function(fn, float_of(u));
  uint64_t z = (static_cast<uint64_t>(u) << 32) | (y == y ? bits_of(y) : 0x7fc00000u);
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

}  // namespace bsx
