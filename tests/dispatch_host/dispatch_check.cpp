// Host check of how work is cut into workgroups: arithmetic of csrc headers that needs no GPU.
#include <cstdio>
#include <vector>

#include "deal.h"
#include "densify_grid.h"

#define CHECK(cond)                                                                 \
  do {                                                                              \
    if (!(cond)) {                                                                  \
      std::fprintf(stderr, "dispatch_check: %s failed (line %d)\n", #cond, __LINE__); \
      return 1;                                                                     \
    }                                                                               \
  } while (0)

namespace {

// Dense maps: every piece has a workgroup, no dimension of a launch has 2^32 threads or more, and what counts for the line is the
// map itself, not the bytes that whole chunks would have.
int denseMaps() {
  struct Shape {
    int64_t yx, planes, channels;
    int elemBytes;
    bool byXcd;
  };
  const int64_t k24 = int64_t(1) << 24;
  const Shape shapes[] = {
      {int64_t(4096) * 4096, 64, 4, 1, false},   // 2^24 workgroups, 4.3 GB
      {int64_t(4095) * 4095, 64, 4, 1, true},    // fewer, planes off the tiles
      {int64_t(4097) * 4095, 64, 4, 1, false},   // more
      {k24 * 8 - 63, 8, 2, 2, false},            // 2^24 workgroups exactly, 2^24 - 8 below
      {(k24 / 8 - 1) * 64 - 1, 8, 2, 2, true},
      {int64_t(300) * 320, 2, 256, 2, false},    // planes of whole lines
      {int64_t(300) * 301, 4, 128, 2, true},
      {int64_t(200) * 200, 4, 256, 1, false},    // planes of whole int8 tiles
      {int64_t(300) * 300, 4, 256, 4, true},     // a line off by half
      {int64_t(300) * 301, 2, 32, 1, false},     // 5.8 MB: 16 MB in whole chunks
      {int64_t(300) * 301, 8, 32, 1, true},
      {int64_t(180) * 181, 2, 256, 1, false},
      {int64_t(181) * 182, 2, 256, 1, true},
      {1, 1, 1, 4, false},
      {129, 65535, 1, 1, false},
  };
  for (const Shape& s : shapes)
    for (int xcdShift = 0; xcdShift <= 3; ++xcdShift) {
      const d3d::DensifyGrid g = d3d::densifyGrid(s.yx, s.planes, s.channels, s.elemBytes, xcdShift);
      CHECK(static_cast<uint64_t>(g.x) * 256 < (uint64_t(1) << 32) && g.y <= 65535 && g.z <= 65535);
      CHECK((g.pieces != 0) == s.byXcd);
      const int64_t tiles = (s.yx + 63) / 64, chunks = (s.channels * s.elemBytes + 127) / 128, pieces = tiles * s.planes * chunks;
      if (g.pieces) {
        CHECK(g.pieces == pieces && g.y == 1 && g.z == 1 && g.x >= pieces && g.x < pieces + (1 << xcdShift) && g.x % (1 << xcdShift) == 0);
      } else {
        CHECK(g.x == tiles && g.y == s.planes && g.z == chunks);
      }
    }
  return 0;
}

// Dealt tiles: ranked in batches of 256, each goes to one workgroup; a workgroup's turns follow one another without a gap and no
// workgroup has two tiles more than another.
int dealtTiles() {
  for (int per : {1, 2, 3, 31, 32, 48, 64, 95, 96, 192})
    for (int tiles : {1, 100, 255, 256, 257, 700, 1024, 1537, 32 * per}) {
      std::vector<int> has(static_cast<size_t>(per), 0);
      std::vector<std::vector<bool>> turns(static_cast<size_t>(per), std::vector<bool>(static_cast<size_t>(tiles / per) + 1));
      for (int from = 0; from < tiles; from += 256)
        for (int rank = 0; rank < 256 && from + rank < tiles; ++rank) {
          const d3d::DealtTile to = d3d::dealTile(from, rank, per);
          CHECK(to.workgroup >= 0 && to.workgroup < per && to.turn >= 0 && to.turn <= tiles / per);
          CHECK(!turns[to.workgroup][to.turn]);
          turns[to.workgroup][to.turn] = true;
          ++has[to.workgroup];
        }
      int least = tiles, most = 0;
      for (int w = 0; w < per; ++w) {
        for (int t = 0; t < has[w]; ++t) CHECK(turns[w][t]);
        least = has[w] < least ? has[w] : least;
        most = has[w] > most ? has[w] : most;
      }
      CHECK(most - least <= 1);
    }
  return 0;
}

}  // namespace

int main() {
  if (denseMaps() || dealtTiles()) return 1;
  std::puts("dispatch_check ok");
  return 0;
}
