// How the workgroups of a dense map are launched (densify.hip).
#pragma once
#include <cstdint>

namespace d3d {

// pieces = 0: the grid is (tiles of a plane, planes, channel chunks).  Otherwise it is one-dimensional, x workgroups of which the
// first `pieces` in XCD order have one to do.
struct DensifyGrid {
  uint32_t x, y, z, pieces;
};

constexpr int kDzTile = 64;          // cells per workgroup, consecutive in y*X + x
constexpr int kDzChunkBytes = 128;   // bytes of a feature row handled by one workgroup

// Where planes are no multiple of what a tile writes per channel (64 cells, at most a line of 128 bytes), every tile but a plane's
// first begins and ends inside a line, which the tile beside it completes.  Two XCDs each write their part of it; in XCD order the
// line is whole in one L2.  us in three dimensions / by XCD, one output written again and again: int8 [1, 512, 180, 181] 12.8 / 9.8,
// [1, 512, 301, 316] 26.6 / 20.6, fp16 [2, 512, 200, 201] (82 MB) 27.4 / 25.3, fp32 [1, 512, 330, 332] 101 / 89; four outputs in
// turn (more than the caches behind the L2s hold): fp16 82 MB 40.1 / 26.4, int8 93 MB 63.9 / 31.4, fp32 257 MB 120 / 93.
// Planes of whole lines gain nothing and pay for the divisions: fp16 [1, 512, 300, 320] 98 MB 26.2 / 28.1, int8 with 66 MB 20.6 /
// 21.5, fp32 with 98 MB 26.8 / 29.0.  Nor do narrow types' maps of fewer elements than the line below by more than a microsecond,
// or fp32 ones at all: fp32 of 30 and 41 MB 12.9 / 13.8 and 15.9 / 16.9, 67 MB 22.0 / 22.5, 82 MB 24.7 / 25.6 in one output and
// 34.9 / 27.4 in four; fp16 of 32 channels, 46 MB 22.9 / 23.1, 56 MB 25.9 / 26.1.
// A launch takes fewer than 2^32 threads in a dimension: 2^24 workgroups of 256.  Three dimensions hold more.
inline DensifyGrid densifyGrid(int64_t yx, int64_t planes, int64_t channels, int elemBytes, int xcdShift) {
  constexpr int64_t kMostWorkgroups = (int64_t(1) << 24) - 1, kLargeMap = int64_t(1) << 24;  // elements
  const int64_t tiles = (yx + kDzTile - 1) / kDzTile, chunks = (channels * elemBytes + kDzChunkBytes - 1) / kDzChunkBytes;
  const int64_t pieces = tiles * planes * chunks, xcds = int64_t(1) << xcdShift;
  const int64_t whole = (pieces + xcds - 1) / xcds * xcds;
  const int64_t boundary = elemBytes == 1 ? kDzTile : 128;
  if (yx * elemBytes % boundary != 0 && yx * planes * channels >= kLargeMap && whole <= kMostWorkgroups)
    return {static_cast<uint32_t>(whole), 1, 1, static_cast<uint32_t>(pieces)};
  return {static_cast<uint32_t>(tiles), static_cast<uint32_t>(planes), static_cast<uint32_t>(chunks), 0};
}

}  // namespace d3d
