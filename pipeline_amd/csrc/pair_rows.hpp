// Rows of sixteen small values as bytes, and the comparison of a whole row with
// one value: what the radix tree's search for the nearest smaller common
// prefix (k_radix_tree.hip) is made of.
#pragma once

#include "ocp_internal.hpp"

namespace ocp {

typedef int32_t v4i __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint16_t v2h __attribute__((ext_vector_type(2)));

// Bit p of the result: byte p of the row is below t, where key = t + 127 in
// every byte (bytes and t at most 31, so no byte borrows from its neighbour).
__device__ __forceinline__ uint32_t below16(const v4u w, uint32_t key) {
  const uint32_t hi = 0x80808080u;
  const uint32_t a = __builtin_amdgcn_udot4(
      (key - w.y) & hi, 0x80402010u,
      __builtin_amdgcn_udot4((key - w.x) & hi, 0x08040201u, 0u, false), false);
  const uint32_t b = __builtin_amdgcn_udot4(
      (key - w.w) & hi, 0x80402010u,
      __builtin_amdgcn_udot4((key - w.z) & hi, 0x08040201u, 0u, false), false);
  return (a >> 7) | (b << 1);
}
__device__ __forceinline__ v2h as_halves(uint32_t x) { return __builtin_bit_cast(v2h, x); }
__device__ __forceinline__ uint32_t min16(const v4u w) {
  v2h m = as_halves(w.x & 0x00ff00ffu);
  m = __builtin_elementwise_min(m, as_halves((w.x >> 8) & 0x00ff00ffu));
  m = __builtin_elementwise_min(m, as_halves(w.y & 0x00ff00ffu));
  m = __builtin_elementwise_min(m, as_halves((w.y >> 8) & 0x00ff00ffu));
  m = __builtin_elementwise_min(m, as_halves(w.z & 0x00ff00ffu));
  m = __builtin_elementwise_min(m, as_halves((w.z >> 8) & 0x00ff00ffu));
  m = __builtin_elementwise_min(m, as_halves(w.w & 0x00ff00ffu));
  m = __builtin_elementwise_min(m, as_halves((w.w >> 8) & 0x00ff00ffu));
  return min(static_cast<uint32_t>(m.x), static_cast<uint32_t>(m.y));
}

}  // namespace ocp
