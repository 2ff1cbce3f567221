// Products of the experts' sorted rows (tile_linear.h's kernel, its grouped form).
#include "tile_linear.h"

namespace xgm {
template <int FM, int FN, int RA, int RW, int OCC = 1, bool SHORT = false>
static void tile_launch_grouped(const TileArgs& a, int cus, hipStream_t st) {
  const int64_t tiles = (int64_t)(a.M / (32 * FM) + a.E) * ((a.N + 32 * FN - 1) / (32 * FN));   // at most
  const int grid = SHORT || tiles < cus * OCC ? (int)tiles : cus * OCC;
  if (a.pairs) tile_linear_kernel<FM, FN, RA, RW, OCC, true, true, SHORT><<<grid, 256, 0, st>>>(a);
  else tile_linear_kernel<FM, FN, RA, RW, OCC, false, true, SHORT><<<grid, 256, 0, st>>>(a);
}

// Products of the experts' sorted rows (moe_align, moe_ff.hip) with their expert's weights w [E, N, K]: gated (act >= kTileGlu) `out`
// [M, N / 2] bf16 of w's rows [gate | up], or fp32 `y` [M, N]. rows[p] / top is row p's row of x (nullptr: p), x_rows of them. Rows of
// no expert are not written; a segment's pads (rows below 0) hold something finite.
int tile_grouped(const void* x, int64_t ld_x, int x_rows, const int32_t* rows, const int32_t* offs, int E, int top, const void* w,
                 float* y, void* out, int M, int N, int K, int act, float p0, float p1, int fm, int fn, int cus, hipStream_t st) {
  const bool gated = act >= kTileGlu;
  if (M < 1 || E < 1 || top < 1 || x_rows < 1 || N < 8 || N % 8 || K < 64 || K % 64 || ld_x < K || ld_x % 8 || !offs || cus < 1 ||
      (gated ? !out || y || !xgk::glu_known(act - kTileGlu) : !y || out || act != kTileNone) || (!rows && x_rows < M) ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y | (uintptr_t)out) & 15) || (int64_t)N * K * 2 >= (1LL << 32) ||
      N >= kTileColumns || x_rows * ld_x * 2 >= (1LL << 32))
    return -1;
  TileArgs a = {(const bf16*)x, (const bf16*)w, nullptr, y, (bf16*)out, ld_x, M, N, K, 1, act, gated ? kPairHalves : kPairNone, p0, p1,
                false, rows, offs, E, top, (int64_t)N * K, M <= (int64_t)kRotateRows * E ? 32 * fn : 0};
#define XGM_TILE(FM, FN, RA, RW)                                                \
  else if (fm == FM && fn == FN) {                                              \
    if (K / 64 > RA) tile_launch_grouped<FM, FN, RA, RW>(a, cus, st);           \
    else if (K / 64 > 2) tile_launch_grouped<4, 4, 2, 3, 2>(a, cus, st);        \
    else tile_launch_grouped<4, 4, 2, 2, 2, true>(a, cus, st);                  \
  }
  if (false) {}
  XGM_TILE(8, 8, 2, 3)
  XGM_TILE(7, 8, 2, 3)
  XGM_TILE(6, 8, 2, 3)
  XGM_TILE(4, 8, 3, 3)
  XGM_TILE(6, 4, 4, 4)
  XGM_TILE(4, 4, 5, 5)
  XGM_TILE(3, 4, 5, 5)
  else return -1;
#undef XGM_TILE
  return 0;
}
}  // namespace xgm
