// Products of many activation rows with a gated activation behind them (tile_linear.h's kernel, compiled beside the plain ones).
#include "tile_linear.h"

namespace xgm {
int tile_launch_gated(const TileArgs& a, int fm, int fn, int cus, hipStream_t st) { return tile_launch_size<true>(a, fm, fn, cus, st); }
}  // namespace xgm
