// Host check of how work is cut into workgroups: arithmetic of csrc headers that needs no GPU.
#include <cstdio>

#include "densify_grid.h"

#define CHECK(cond)                                                                 \
  do {                                                                              \
    if (!(cond)) {                                                                  \
      std::fprintf(stderr, "dispatch_check: %s failed (line %d)\n", #cond, __LINE__); \
      return 1;                                                                     \
    }                                                                               \
  } while (0)

namespace {

// Dense maps: every piece has a workgroup, and no dimension of a launch has 2^32 threads or more.
int denseMaps() {
  const int64_t k24 = int64_t(1) << 24;
  // 2^30 cells of four int8 channels in 64 planes, and sizes around 2^24 workgroups
  const int64_t shapes[][3] = {{262144, 64, 1}, {k24 - 1, 1, 1}, {k24 / 8 - 1, 8, 1}, {k24 / 8, 8, 1}, {k24 / 16, 4, 4}, {k24 / 8 + 1, 8, 1},
                               {8191, 1, 1}, {8192, 1, 1}, {1, 1, 1}, {507, 2, 2}, {2704, 2, 2}, {3, 65535, 65535}};
  for (const auto& s : shapes)
    for (int xcdShift = 0; xcdShift <= 3; ++xcdShift) {
      const d3d::DensifyGrid g = d3d::densifyGrid(s[0], s[1], s[2], xcdShift);
      CHECK(static_cast<uint64_t>(g.x) * 256 < (uint64_t(1) << 32) && g.y <= 65535 && g.z <= 65535);
      const int64_t pieces = s[0] * s[1] * s[2];
      if (g.pieces) {
        CHECK(g.pieces == pieces && g.y == 1 && g.z == 1 && g.x >= pieces && g.x < pieces + (1 << xcdShift) && g.x % (1 << xcdShift) == 0);
      } else {
        CHECK(g.x == s[0] && g.y == s[1] && g.z == s[2]);
      }
    }
  return 0;
}

}  // namespace

int main() {
  if (denseMaps()) return 1;
  std::puts("dispatch_check ok");
  return 0;
}
