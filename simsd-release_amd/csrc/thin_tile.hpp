// Tile kernel of the linear layers above 8 tokens (thin_tile.hip): its plan
// and its launch.
#pragma once

#include "thin_common.hpp"

namespace simsd {

struct TilePlan {
  int cfg;                   // index into the tile table
  int bm, bn;                // tokens and weight rows of a tile
  int waves;
  int split;                 // workgroups along K
  int64_t tiles_n, tiles_m;
  int steps, steps_per_split;   // in stages of 128 bytes of every row
};

// The tile and, for split_k <= 0, the split along K of a call over `rows`
// weight rows (gated: both halves); partials: the caller's next launch sums them.
TilePlan thin_tile_plan(int64_t M, int64_t rows, int64_t K, bool partials, int split_k);

// Whether the operands fit the kernel's 32-bit offsets for any of its tiles.
bool thin_tile_fits(int64_t M, int64_t N, int64_t K, int64_t sxm, int64_t swn, int64_t sw2n, int64_t sym, int64_t srm);

// bf16 / fp16; partials to a.part where `part` is set, else outputs.
void launch_thin_tile(const TilePlan& p, ThinArgs a, int dtype, bool glu, bool part, hipStream_t stream);

}  // namespace simsd
