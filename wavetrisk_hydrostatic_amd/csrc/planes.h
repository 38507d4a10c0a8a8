// Planes of an array as buffer loads address them.
#pragma once
#include <cstdint>

namespace wtg {

struct PlaneAt {
  int64_t first;  // doubles from the array to the base of the descriptor
  uint32_t byte;  // byte offset of the plane from that base
};

// Plane p of an array of planes of nc doubles.  A load adds the cell's byte
// offset to the plane's in 32 bits, and three planes of the largest grid (level
// 12: 1.34 GB each) still lie within 4 GiB of their base; a fourth does not.
constexpr PlaneAt plane_at(int p, int64_t nc) { return {p / 3 * 3 * nc, (uint32_t)(p % 3 * nc * 8)}; }

}  // namespace wtg
