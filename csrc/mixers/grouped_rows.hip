// Products of sorted rows with their experts' weights (moe_ff.hip: grouped_gemm) where an expert has up to a few dozen
// rows, so that reading the weights carries the time: a workgroup owns one layout tile of 16 MT rows and WV waves of 16 NW
// weight rows of its expert. Chunks of the (gathered) rows and of the weights come in by LDS-DMA through a ring of NS
// slots, as in rows_linear.hip; the products are 16x16x32 MFMAs with fp32 sums over the whole K, so nothing has to meet.
// Rows of the tile that hold no pair read some other row and are not stored: a row only enters its own results.
//
// Measured on 8 experts of 2 x 3584 x 4096 (gated) and 4096 x 3584, cold weights, us, against fragments read straight from
// global memory by four waves with a quarter of K each:
//   64 tokens, top 2 (tiles of 32)    73.7 + 39.2 against 140.7 + 70.9   (6.4 and 6.0 TB/s of weights; in a step, between other
//                                     launches, 78.8 + 45.7 against 152 + 82: 6.0 and 5.1)
//   150 tokens (64)                   79.3 + 47.6 against 175.8 + 105.6 (its 32-row tiles)
//   4 tokens, 1 token (16)            53.7 + 28.5, 22.1 + 12.1 against 88.3 + 40.7, 68.7 + 34.0
// and against tiles of 64 x 128 (gated) and 64 x 256 columns staged in LDS, which had the experts of 64 rows and more; sorting
// and both products:
//   64 / 80 / 95 rows on average, gated               202 / 248 / 246 against 367 / 397 / 557
//   64 / 95 / 112 / 127 rows, one weight block        165 / 194 / 195 / 233 against 318 / 357 / 380 / 405
//   32 experts of 1024 x 2048, 64 / 95 rows           141 / 169 against 193 / 228 (gated), 114 / 138 against 163 / 177
// Two to four workgroups share a compute unit (40 KB of LDS in the gated form for 16 rows, 48 to 61 for 32, 64 and 72 for 64), which
// hides that the grid seldom is a multiple of 256: one workgroup of 144 KB per unit took 88.6 for the first.
#include "attention_common.h"
#include "glds.h"
#include "glu.h"

namespace xgm {
using xgk::as_frag;
using xgk::f32x4_t;
using xgk::glu;
using xgk::mfma16x16x32;

struct GroupedArgs {
  const bf16 *A, *w;
  const int32_t *rows, *tile_expert;
  void* out;
  const float* row_scale;   // [pairs] or nullptr (MODE 2)
  int64_t lda;
  int top, N, K, kind;
  float limit, alpha;
};

// MODE 0: A rows as they lie -> fp32; 1: gathered rows, weights [gate | up] -> bf16 glu; 2: gathered rows -> bf16
// max(scale z, 0)^2. N: output columns.
template <int MODE, int MT, int NW, int WV, int KC, int NS>
__global__ __launch_bounds__(64 * WV, 1) void grouped_rows_kernel(const GroupedArgs a) {
  constexpr bool GATED = MODE == 1, FIRST = MODE != 0;
  constexpr int RB = KC * 2, GPR = KC / 8, RPI = 1024 / RB;   // bytes and granules per staged row, rows per DMA instruction
  constexpr int XROWS = 16 * MT, WROWS = 16 * NW, OUT = GATED ? 8 * NW : 16 * NW;   // OUT: output columns of a wave
  constexpr int XI = XROWS / RPI / WV, WI = WROWS / RPI, G = XI + WI;
  constexpr int SLOT = (XROWS + WROWS * WV) * RB;
  static_assert(XI >= 1 && WI >= 1 && XROWS % (RPI * WV) == 0 && NS * SLOT <= 160 * 1024 && (!GATED || NW % 2 == 0),
                "grouped_rows geometry");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[NS * SLOT];
  const int tile = blockIdx.y, e = a.tile_expert[tile];
  if (e < 0) return;
  const int lane = threadIdx.x & 63, g4 = lane >> 4, l16 = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = (blockIdx.x * WV + wv) * OUT, rbase = tile * XROWS, nch = a.K / KC;
  const bf16* We = a.w + (int64_t)e * (GATED ? 2 : 1) * a.N * a.K;
  const int dr = lane / GPR, dj = lane % GPR;
  const bf16 *ws[WI], *xs[XI];
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int r = RPI * i + dr, c = GATED ? r % OUT : r;
    const int64_t n = min(n0 + c, a.N - 1) + (GATED && r >= OUT ? a.N : 0);
    ws[i] = We + n * a.K + 8 * (dj ^ (r & (GPR - 1)));
  }
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int r = RPI * (wv * XI + i) + dr;
    const int64_t src = FIRST ? max(a.rows[rbase + r], 0) / a.top : rbase + r;
    xs[i] = a.A + src * a.lda + 8 * (dj ^ (r & (GPR - 1)));
  }
  // (see rows_linear.hip: the tiles of a launch start at different chunks)
  const int rot = (int)((unsigned)blockIdx.x * 37u % (unsigned)nch);
  auto issue = [&](int c) {
    uint8_t* slot = lds + (c % NS) * SLOT;
    int cc = min(c, nch - 1) + rot;
    cc = cc >= nch ? cc - nch : cc;
#pragma unroll
    for (int i = 0; i < XI; ++i) xgk::glds16(xs[i] + cc * KC, slot + RPI * (wv * XI + i) * RB);
#pragma unroll
    for (int i = 0; i < WI; ++i) xgk::glds16_nt(ws[i] + cc * KC, slot + (XROWS + WROWS * wv) * RB + i * 1024);
  };
  // lane of a product: weight row 4 g4 + r, row l16 of the tile
  f32x4_t acc[NW][MT];
#pragma unroll
  for (int n = 0; n < NW; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < NS - 1; ++c) issue(c);
  for (int c = 0; c < nch; ++c) {
    xgk::wait_vmcnt<(NS - 2) * G>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    xgk::raw_barrier();
    issue(c + NS - 1);
    const uint8_t* xl = lds + (c % NS) * SLOT;
    const uint8_t* wl = xl + (XROWS + WROWS * wv) * RB;
#pragma unroll
    for (int t = 0; t < KC / 32; ++t) {
      const int ph = ((4 * t + g4) ^ (l16 & (GPR - 1))) * 16;
      uint4 b[MT], w[NW];
#pragma unroll
      for (int m = 0; m < MT; ++m) b[m] = *reinterpret_cast<const uint4*>(xl + (16 * m + l16) * RB + ph);
#pragma unroll
      for (int n = 0; n < NW; ++n) w[n] = *reinterpret_cast<const uint4*>(wl + (16 * n + l16) * RB + ph);
#pragma unroll
      for (int n = 0; n < NW; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[n][m] = mfma16x16x32(as_frag(w[n]), as_frag(b[m]), acc[n][m]);
    }
  }
  xgk::wait_vmcnt<0>();
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int r = rbase + 16 * m + l16, pr = a.rows[r];
    if (pr < 0) continue;
#pragma unroll
    for (int n = 0; n < (GATED ? NW / 2 : NW); ++n) {
      const int col = n0 + 16 * n + 4 * g4;
      if (col >= a.N) continue;
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = acc[n][m][j];
        if (MODE == 1) v[j] = glu(a.kind, v[j], acc[(GATED ? NW / 2 : 0) + n][m][j], a.limit, a.alpha);
        if (MODE == 2) v[j] = relu2f(v[j] * (a.row_scale ? a.row_scale[pr] : 1.f));
      }
      if (FIRST) st4((bf16*)a.out + (int64_t)r * a.N + col, v);
      else st4((float*)a.out + (int64_t)r * a.N + col, v);
    }
  }
}
// Returns 0, or -1 for sizes that it does not take: tm (rows per layout tile) 16, 32 or 64, K % 64 == 0, N % 4 == 0,
// 16-byte aligned rows and weights. The caller has checked the layout (moe_align).
int grouped_rows(const void* A, int64_t lda, const void* w, const int32_t* rows, const int32_t* tile_expert, int cap, int tm,
                 int top, int N, int K, int mode, void* out, int kind, float limit, float alpha, const float* row_scale,
                 hipStream_t st) {
  if ((tm != 16 && tm != 32 && tm != 64) || cap % tm || K < 64 || K % 64 || N < 4 || N % 4 || lda % 8 ||
      (((uintptr_t)A | (uintptr_t)w | (uintptr_t)out) & 15))
    return -1;
  const GroupedArgs a = {(const bf16*)A, (const bf16*)w, rows, tile_expert, out, row_scale, lda, top, N, K, kind, limit, alpha};
#define XGM_GR(MODE, MT, NW, WV, NS)                                                                       \
  {                                                                                                        \
    constexpr int cols = (MODE == 1 ? 8 : 16) * NW * WV;                                                   \
    grouped_rows_kernel<MODE, MT, NW, WV, 64, NS><<<dim3((N + cols - 1) / cols, cap / tm), 64 * WV, 0, st>>>(a); \
  }
#define XGM_GR_ONE(MODE)                        \
  if (tm == 16) XGM_GR(MODE, 1, 1, 2, 8)        \
  else if (tm == 32) XGM_GR(MODE, 2, 1, 4, 4)   \
  else XGM_GR(MODE, 4, 1, 4, 4)
  if (mode == 1) {
    if (tm == 16) XGM_GR(1, 1, 2, 2, 4)
    else if (tm == 32) XGM_GR(1, 2, 2, 4, 3)
    else XGM_GR(1, 4, 2, 4, 3)
  } else if (mode == 2) {
    XGM_GR_ONE(2)
  } else {
    XGM_GR_ONE(0)
  }
#undef XGM_GR_ONE
#undef XGM_GR
  return 0;
}
}  // namespace xgm
