// How the workgroups of a dense map are launched (densify.hip).
#pragma once
#include <cstdint>

namespace d3d {

// pieces = 0: the grid is (tiles of a plane, planes, channel chunks).  Otherwise it is one-dimensional, x workgroups of which the
// first `pieces` in XCD order have one to do.
struct DensifyGrid {
  uint32_t x, y, z, pieces;
};

// A launch takes fewer than 2^32 threads in a dimension: 2^24 workgroups of 256.  Three dimensions hold more.
inline DensifyGrid densifyGrid(int64_t tiles, int64_t planes, int64_t chunks, int xcdShift) {
  constexpr int64_t kMostWorkgroups = (int64_t(1) << 24) - 1, kLarge = (int64_t(64) << 20) / (64 * 128);
  const int64_t pieces = tiles * planes * chunks, xcds = int64_t(1) << xcdShift;
  const int64_t whole = (pieces + xcds - 1) / xcds * xcds;
  if (pieces >= kLarge && whole <= kMostWorkgroups) return {static_cast<uint32_t>(whole), 1, 1, static_cast<uint32_t>(pieces)};
  return {static_cast<uint32_t>(tiles), static_cast<uint32_t>(planes), static_cast<uint32_t>(chunks), 0};
}

}  // namespace d3d
