// Which workgroup takes a ranked tile (TileDeal, conv_pipe.h).
#pragma once
#include <hip/hip_runtime.h>

namespace d3d {

struct DealtTile {
  int turn, workgroup;
};

// Tiles are dealt to `per` workgroups in turns, forth and back.  They are ranked in batches; `rank` is a tile's place in the batch that
// begins behind `before` tiles.  Turns run on from batch to batch, so that a workgroup has one tile of every turn and no two of them
// differ by more than one tile.  (With turns that began anew in every batch of 256, 96 workgroups had three or two tiles of each, and
// always the same 64 had three.  64 -> 64 in fp32, 300 000 rows 434 -> 425 us, 600 000 843 -> 829; 128 -> 128 in fp16, 313 000 rows
// 212 -> 209.  Ranking every other batch lightest first, so that its lightest follow those of the one before: no change.)
__host__ __device__ inline DealtTile dealTile(int before, int rank, int per) {
  const int at = before + rank, turn = at / per, place = at - turn * per;
  return {turn, turn & 1 ? per - 1 - place : place};
}

}  // namespace d3d
