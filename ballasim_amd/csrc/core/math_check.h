// The fp32 functions of pmath.h by number (of one argument, and div_with on drawn pairs), and an
// order-independent hash of their results over a range of bit patterns: the device's forms (divisions by reciprocal and remainder, hardware splitting and
// scaling) are compared with the host's plain ones this way.
#pragma once

#include "pmath.h"

namespace bsx {

inline constexpr int kMathFunctions = 14;

// div_with on a pair (a, b) drawn from u: any mantissas, exponents in [-60, 60], among them all-ones and zero mantissas,
// exact quotients and their neighbours, and zeros, infinities and NaNs.
BSX_HD inline float div_with_drawn(uint32_t u) {
  uint64_t z = (static_cast<uint64_t>(u) + 1) * 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z ^= z >> 27;
  const uint32_t ma = static_cast<uint32_t>(z) & 0x7fffffu, mb = static_cast<uint32_t>(z >> 23) & 0x7fffffu;
  const uint32_t ea = 67 + static_cast<uint32_t>(z >> 46) % 121, eb = 67 + static_cast<uint32_t>(z >> 53) % 121;
  uint32_t a = (static_cast<uint32_t>(z >> 62) << 31) | (ea << 23) | ma, b = (static_cast<uint32_t>(z >> 63) << 31) | (eb << 23) | mb;
  const uint32_t special[8] = {0u, 0x80000000u, 0x7f800000u, 0xff800000u, 0x7fc00000u, 0x3f800000u, 0xbf800000u, 0x40400000u};
  switch (u & 15) {
    case 0: b |= 0x7fffffu; break;
    case 1: a |= 0x7fffffu; break;
    case 2: a &= 0xff800000u; break;
    case 3: b &= 0xff800000u; break;
    case 4: a = bits_of(float_of(b & 0xfffff000u) * static_cast<float>(ma & 0xfffu)), b &= 0xfffff000u; break;  // exact
    case 5: a = bits_of(float_of(b) * static_cast<float>(1 + (ma & 0xffu))) + 1; break;  // beside one
    case 6: a = special[ma & 7]; break;
    case 7: a = special[ma & 7], b = special[(ma >> 3) & 7]; break;
    default: break;
  }
  return pm::div_with(float_of(a), float_of(b), pm::recip(float_of(b)));
}

BSX_HD inline float math_function(int fn, uint32_t u) {
  const float x = float_of(u);
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
    case 11: return pm::div_by_any<384>(x);
    case 12: return pm::recip(x);
    default: return div_with_drawn(u);
  }
}

// (every NaN hashes alike)
BSX_HD inline uint64_t math_hash(int fn, uint32_t u) {
  const float y = math_function(fn, u);
  uint64_t z = (static_cast<uint64_t>(u) << 32) | (y == y ? bits_of(y) : 0x7fc00000u);
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

}  // namespace bsx
