// Products of a few activation rows (decode steps, T <= 64) with a weight matrix, and what follows them:
//
//   rows_linear         out [T, N] = act(x [T, K] . w [N, K]^T + bias), or glu(gate, up) of w's two halves
//
// The weights are read once and carry the time: 2 N K bytes against T <= 64 rows. A workgroup owns COLS weight rows and
// one of S equal parts of K; its chunks of x and w come in by LDS-DMA through a ring of NS slots (NS - 1 chunks in
// flight, so that a CU keeps 40 to 100 KB on the way), every weight row a full 128- or 256-byte line, and the products
// are 16x16x32 MFMAs with fp32 sums. Rows are staged with their 16-byte granules permuted by the row number, so the
// fragment reads of 16 rows fall on all banks.
//
// S parts of K: the parts of a column tile write fp32 slabs (write-through) and take a ticket; the one that draws the
// last adds the slabs in order and finishes the tile, so a narrow product still puts a workgroup on every CU and needs
// no second launch. The tickets are words that are zero before the launch and zero again after it. Without tickets the
// slabs are the result: the next kernel adds them as it reads them (row_update.hip, postnorm.hip), which saves the wait
// for the last part.
//
// That meeting costs 1.5 us at one row and 3.5 to 5 at 64: store, ticket, reads back, one behind the other. rows_whole_kernel
// takes narrower tiles over the whole K instead. A CU has about 105 requests of 128 bytes under way, each for some 1000
// clocks where it goes to memory (w) and 400 where it hits L2 (x, which every workgroup reads), so a workgroup costs about
// (0.4 rows + columns) K whatever the ring holds, and the caller takes the form that costs less (ops.seqmix._rows_cols). Its
// waves divide K, not the columns: each byte is read from LDS once, where four waves over the columns read x four times, which at
// 64 rows was 670 clocks for every 64 of K. us, cold weights, T = 1 / 17 / 40 / 64, parts with tickets (or whole tiles of 64) before:
//   1088 x 2048    5.1 /  6.8 /  7.6 /  8.6 -> 3.9 / 4.8 / 6.3 / 7.3     16384 x 2048, gated  16.2 / 19.2 / 18.8 / 20.4 -> 12.7 / 13.2 / 14.6 / 15.1
//   3072 x 768     4.1 /  4.9 /  6.0 /  6.4 -> 3.2 / 3.6 / 4.2 / 4.8     7168 x 4096, gated   13.9 / 17.2 / 18.0 / 21.1 -> 11.0 / 12.8 / 15.6 / 18.2
//   6176 x 4096   11.5 / 13.3 / 16.7 / 20.5 -> 10.0 / 12.3 / 15.3 / 17.8  10768 x 4096, 64 rows 24.9 -> 22.4; 8192 x 2048, 64 rows 13.3 -> 10.7
//
// Measured against the library's product without what follows it, each in the form it runs in, cold weights, us (T = 1 / 17 / 64):
//   2048 x 2048    4.3 /  5.2 /  7.6 against 11.0 / 11.0 / 11.8      18560 x 4096   30 / 30 / 38 against 67 / 36 / 40
//   2048 x 8192    9.6 / 11.0 / 13.7 against 12.9 / 13.7 / 22.6      28672 x 4096   39 / 38 / 41 against 64 / 55 / 56
//   10272 x 2048   8.7 /  9.4 / 13.0 against 16.3 / 14.6 / 15.9      4096 x 14336   22 / 23 / 28 against 26 / 28 / 39
// (5.8 TB/s of weights at the largest; 2048 x 8192, 18560 x 4096 and 4096 x 14336 in parts or tiles of 128, the small ones over the whole K.)
#include "attention_common.h"
#include "glds.h"
#include "glu.h"

namespace xgm {
using xgk::as_frag;
using xgk::f32x4_t;
using xgk::glu;
using xgk::mfma16x16x32;

enum { kActNone = 0, kActXielu = 1, kActRelu2 = 2, kActGlu = 3 };   // kActGlu + kind: glu.h

struct RowsArgs {
  const bf16 *x, *w;
  const void* bias;        // [N] fp32 or bf16, or nullptr
  float* part;             // S > 1: [S, T, N] fp32
  bf16* out;               // [T, N], or [T, N / 2] for the gated activations
  int* tickets;            // one zero word per column tile (S > 1), or nullptr: the slabs are the result
  int64_t ld_x;
  int T, N, K, act;
  float p0, p1;
  bool bias_f32;
};

// act(v + bias) of four neighbouring columns
__device__ __forceinline__ void rows_finish(const RowsArgs& a, int tok, int col, float (&v)[4]) {
  if (a.bias) {
    float b[4];
    if (a.bias_f32) ld4((const float*)a.bias + col, b);
    else ld4((const bf16*)a.bias + col, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += b[e];
  }
  if (a.act == kActXielu) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = xieluf(v[e], a.p0, a.p1);
  } else if (a.act == kActRelu2) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = relu2f(v[e]);
  }
  st4(a.out + (int64_t)tok * a.N + col, v);
}

__device__ __forceinline__ void rows_finish_glu(const RowsArgs& a, int tok, int f, const float (&g)[4], const float (&u)[4]) {
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = glu(a.act - kActGlu, g[e], u[e], a.p0, a.p1);
  st4(a.out + (int64_t)tok * (a.N / 2) + f, v);
}

// sum of the S slabs at `at` (every read comes from another XCD's workgroup: all S are in flight before the first add)
template <int S>
__device__ __forceinline__ void slab_sum(const float* __restrict__ at, int64_t slab, float (&v)[4]) {
  float p[S][4];
#pragma unroll
  for (int s = 0; s < S; ++s) ld4(at + s * slab, p[s]);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = p[0][e];
#pragma unroll
    for (int s = 1; s < S; ++s) v[e] += p[s][e];
  }
}

// the last part of a column tile: columns [c0, c0 + NC) (gated: and as many of the second half) of every row
template <int NC, int NTHR, int S>
__device__ __forceinline__ void rows_tail(const RowsArgs& a, int c0, bool gated) {
  const int64_t slab = (int64_t)a.T * a.N;
  const int half = a.N / 2;
#pragma unroll 2
  for (int i = threadIdx.x; i < a.T * (NC / 4); i += NTHR) {
    const int tok = i / (NC / 4), col = c0 + 4 * (i % (NC / 4));
    const float* at = a.part + (int64_t)tok * a.N + col;
    float v[4];
    if (gated) {
      if (col >= half) continue;
      float u[4];
      slab_sum<S>(at, slab, v);
      slab_sum<S>(at + half, slab, u);
      rows_finish_glu(a, tok, col, v, u);
    } else {
      if (col >= a.N) continue;
      slab_sum<S>(at, slab, v);
      rows_finish(a, tok, col, v);
    }
  }
}

// Workgroup (tile, part of K): WV waves of NW 16-row weight tiles each, MT 16-row x tiles. A gated launch (NW = 2)
// gives each wave the same 16 rows of w's first and second half.
template <int MT, int NW, int WV, int KC, int NS>
__global__ __launch_bounds__(64 * WV, 1) void rows_linear_kernel(const RowsArgs a) {
  constexpr int RB = KC * 2, GPR = KC / 8, RPI = 1024 / RB;   // bytes and granules per staged row, rows per DMA instruction
  constexpr int XROWS = 16 * MT, COLS = 16 * NW * WV;
  constexpr int XI = XROWS / RPI / WV, WI = 16 * NW / RPI, G = XI + WI;
  constexpr int SLOT = (XROWS + COLS) * RB;
  static_assert(XI >= 1 && WI >= 1 && XROWS % (RPI * WV) == 0 && NS * SLOT <= 160 * 1024, "rows_linear geometry");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[NS * SLOT];
  const int lane = threadIdx.x & 63, g4 = lane >> 4, l16 = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int S = gridDim.y, part = blockIdx.y, bx = blockIdx.x;
  const bool gated = NW == 2 && a.act >= kActGlu;
  const int half = a.N / 2;
  const int chunks = a.K / KC, c_lo = part * chunks / S, nch = (part + 1) * chunks / S - c_lo;
  const int n0 = gated ? bx * (COLS / 2) + 16 * wv : bx * COLS + 16 * NW * wv;
  const int dr = lane / GPR, dj = lane % GPR;
  const bf16 *ws[WI], *xs[XI];
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int r = RPI * i + dr;
    const int n = gated ? (r < 16 ? min(n0 + r, half - 1) : half + min(n0 + r - 16, half - 1)) : min(n0 + r, a.N - 1);
    ws[i] = a.w + (int64_t)n * a.K + c_lo * KC + 8 * (dj ^ (r & (GPR - 1)));
  }
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int r = RPI * (wv * XI + i) + dr;
    xs[i] = a.x + min(r, a.T - 1) * a.ld_x + c_lo * KC + 8 * (dj ^ (r & (GPR - 1)));
  }
  // few parts: neighbouring tiles start at different chunks, or all of them would ask for the same column of weight rows
  // 2 K bytes apart (few memory channels) at the same time
  const int rot = S <= 2 ? (int)((unsigned)bx * 37u % (unsigned)nch) : 0;
  auto issue = [&](int c) {   // (past the end: the last chunk again, into a slot that nobody reads)
    uint8_t* slot = lds + (c % NS) * SLOT;
    int cc = min(c, nch - 1) + rot;
    cc = cc >= nch ? cc - nch : cc;
#pragma unroll
    for (int i = 0; i < XI; ++i) xgk::glds16(xs[i] + cc * KC, slot + RPI * (wv * XI + i) * RB);
#pragma unroll
    for (int i = 0; i < WI; ++i) xgk::glds16_nt(ws[i] + cc * KC, slot + (XROWS + 16 * NW * wv) * RB + i * 1024);
  };
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
    const uint8_t* wl = xl + (XROWS + 16 * NW * wv) * RB;
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
  // lane: weight row 4 g4 + r of the tile, token l16
  if (S == 1) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int tok = 16 * m + l16;
      if (tok >= a.T) continue;
      if (gated) {
        const int f = n0 + 4 * g4;
        if (f >= half) continue;
        const float g[4] = {acc[0][m][0], acc[0][m][1], acc[0][m][2], acc[0][m][3]};
        const float u[4] = {acc[NW - 1][m][0], acc[NW - 1][m][1], acc[NW - 1][m][2], acc[NW - 1][m][3]};
        rows_finish_glu(a, tok, f, g, u);
        continue;
      }
#pragma unroll
      for (int n = 0; n < NW; ++n) {
        const int col = n0 + 16 * n + 4 * g4;
        if (col >= a.N) continue;
        float v[4] = {acc[n][m][0], acc[n][m][1], acc[n][m][2], acc[n][m][3]};
        rows_finish(a, tok, col, v);
      }
    }
    return;
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int tok = 16 * m + l16;
    if (tok >= a.T) continue;
#pragma unroll
    for (int n = 0; n < NW; ++n) {
      const int in = gated ? n0 + 4 * g4 : n0 + 16 * n + 4 * g4;
      if (in >= (gated ? half : a.N)) continue;
      float* at = a.part + ((int64_t)part * a.T + tok) * a.N + in + (gated && n ? half : 0);
      if (a.tickets) xgk::st16_sc1(at, acc[n][m]);
      else *reinterpret_cast<f32x4_t*>(at) = acc[n][m];
    }
  }
  if (!a.tickets) return;
  if (!xgk::agent_ticket(a.tickets + bx, S - 1, reinterpret_cast<int*>(lds))) return;
  const int c0 = gated ? bx * (COLS / 2) : bx * COLS;
#define XGM_TAIL(SS)                                                  \
  if (S == SS) {                                                      \
    if (gated) rows_tail<COLS / 2, 64 * WV, SS>(a, c0, true);         \
    else rows_tail<COLS, 64 * WV, SS>(a, c0, false);                  \
  }
  XGM_TAIL(2)
  XGM_TAIL(4)
  XGM_TAIL(8)
#undef XGM_TAIL
}

// Workgroup: COLS = 16 NT WN weight rows, the whole K. Of a chunk of 128 the four waves along K take 32 each, with all MT
// tiles of x and NT of w (WN groups of such waves side by side); their sums meet in LDS. Gated: half of a wave's tiles are rows
// of w's first half, half the same rows of its second.
template <int MT, int NT, int WN, int NS>
__global__ __launch_bounds__(256 * WN, 1) void rows_whole_kernel(const RowsArgs a) {
  constexpr int WK = 4, WV = WK * WN, KC = 32 * WK, RB = KC * 2, GPR = KC / 8, RPI = 1024 / RB;
  constexpr int XROWS = 16 * MT, COLS = 16 * NT * WN, TILES = MT * NT, NH = NT / 2;
  constexpr int XI = XROWS / RPI / WV, WI = COLS / RPI / WV, G = XI + WI;
  constexpr int SLOT = (XROWS + COLS) * RB, SUMS = WV * TILES * 1024;
  static_assert(XI >= 1 && WI >= 1 && XROWS % (RPI * WV) == 0 && COLS % (RPI * WV) == 0 && NS * SLOT <= 160 * 1024 &&
                SUMS <= NS * SLOT && (NS - 2) * G < 64, "rows_whole geometry");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[NS * SLOT];
  const int lane = threadIdx.x & 63, g4 = lane >> 4, l16 = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wk = wv % WK, wn = wv / WK;
  const int bx = blockIdx.x, nch = a.K / KC;
  const bool gated = NT % 2 == 0 && a.act >= kActGlu;
  const int half = a.N / 2, lim = gated ? half : a.N, n0 = bx * (gated ? COLS / 2 : COLS);
  const int dr = lane / GPR, dj = lane % GPR;
  const bf16 *ws[WI], *xs[XI];
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int r = RPI * (wv * WI + i) + dr, rr = r % (16 * NT), f = n0 + 8 * NT * (r / (16 * NT)) + rr % (8 * NT);
    const int n = gated ? min(f, half - 1) + (rr < 8 * NT ? 0 : half) : min(n0 + r, a.N - 1);
    ws[i] = a.w + (int64_t)n * a.K + 8 * (dj ^ (r & (GPR - 1)));
  }
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int r = RPI * (wv * XI + i) + dr;
    xs[i] = a.x + min(r, a.T - 1) * a.ld_x + 8 * (dj ^ (r & (GPR - 1)));
  }
  int at = (int)((unsigned)bx * 37u % (unsigned)nch), left = nch;   // (neighbouring tiles start at different chunks, as above)
  auto issue = [&](int s) {   // (past the end: the last chunk again, into a slot that nobody reads)
    uint8_t* slot = lds + s * SLOT;
#pragma unroll
    for (int i = 0; i < XI; ++i) xgk::glds16(xs[i] + at * KC, slot + RPI * (wv * XI + i) * RB);
#pragma unroll
    for (int i = 0; i < WI; ++i) xgk::glds16_nt(ws[i] + at * KC, slot + (XROWS + RPI * (wv * WI + i)) * RB);
    if (--left > 0) at = at + 1 == nch ? 0 : at + 1;
  };
  f32x4_t acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < NS - 1; ++c) issue(c);
  const int ph = ((4 * wk + g4) ^ (l16 & (GPR - 1))) * 16;
  int rd = 0, wr = NS - 1;
  for (int c = 0; c < nch; ++c) {
    xgk::wait_vmcnt<(NS - 2) * G>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    xgk::raw_barrier();
    const uint8_t* xl = lds + rd * SLOT;
    const uint8_t* wl = xl + (XROWS + 16 * NT * wn) * RB;
    uint4 b[MT], w[NT];
#pragma unroll
    for (int m = 0; m < MT; ++m) b[m] = *reinterpret_cast<const uint4*>(xl + (16 * m + l16) * RB + ph);
#pragma unroll
    for (int n = 0; n < NT; ++n) w[n] = *reinterpret_cast<const uint4*>(wl + (16 * n + l16) * RB + ph);
    issue(wr);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[n][m] = mfma16x16x32(as_frag(w[n]), as_frag(b[m]), acc[n][m]);
    rd = rd + 1 == NS ? 0 : rd + 1, wr = wr + 1 == NS ? 0 : wr + 1;
  }
  xgk::wait_vmcnt<0>();
  __syncthreads();   // (every wave is past its reads and its loads: the sums may lie over the ring)
  float4* sums = reinterpret_cast<float4*>(lds);
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m)
      sums[(wv * TILES + n * MT + m) * 64 + lane] = make_float4(acc[n][m][0], acc[n][m][1], acc[n][m][2], acc[n][m][3]);
  __syncthreads();
  // a unit: four columns of one row, as a lane of the products held them; the four waves' sums in their order
  auto total = [&](int u, float (&v)[4]) {
    float4 p[WK];
#pragma unroll
    for (int i = 0; i < WK; ++i) p[i] = sums[i * TILES * 64 + u];
    v[0] = p[0].x, v[1] = p[0].y, v[2] = p[0].z, v[3] = p[0].w;
#pragma unroll
    for (int i = 1; i < WK; ++i) v[0] += p[i].x, v[1] += p[i].y, v[2] += p[i].z, v[3] += p[i].w;
  };
  const int tn = gated ? NH : NT, units = WN * MT * tn * 64;
  for (int i = threadIdx.x; i < units; i += 64 * WV) {
    const int t = i >> 6, m = t % MT, n = t / MT % tn, g = t / (MT * tn);
    const int u = (g * WK * TILES + n * MT + m) * 64 + (i & 63);
    const int tok = 16 * m + (i & 15), col = n0 + 16 * (g * tn + n) + 4 * ((i >> 4) & 3);
    if (tok >= a.T || col >= lim) continue;
    float v[4];
    total(u, v);
    if (gated) {
      float q[4];
      total(u + NH * MT * 64, q);
      rows_finish_glu(a, tok, col, v, q);
    } else {
      rows_finish(a, tok, col, v);
    }
  }
}

template <int MT, int NS1, int WN2, int NT2, int NS2, int WN4, int NT4>
static void rows_whole(const RowsArgs& a, int cols, hipStream_t st) {
  const bool gated = a.act >= kActGlu;
  const int tile = gated ? cols / 2 : cols, grid = ((gated ? a.N / 2 : a.N) + tile - 1) / tile;
  if (cols == 16) rows_whole_kernel<MT, 1, 1, NS1><<<grid, 256, 0, st>>>(a);
  else if (cols == 32 && gated) rows_whole_kernel<MT, 2, 1, NS2><<<grid, 256, 0, st>>>(a);
  else if (cols == 32) rows_whole_kernel<MT, NT2, WN2, NS2><<<grid, 256 * WN2, 0, st>>>(a);
  else if (cols == 48) rows_whole_kernel<MT, 3, 1, 4><<<grid, 256, 0, st>>>(a);
  else rows_whole_kernel<MT, NT4, WN4, 4><<<grid, 256 * WN4, 0, st>>>(a);
}

// cols: weight rows of a workgroup: 64 or 128 (the gated activations: 128) of a part of K, or of the whole K (S = 1) 16, 32, 48 (gated:
// 32, 64). Returns 0, or -1 for sizes outside the contract: 1 <= T <= 64, K % 128 == 0, N % 4 == 0 (gated: N % 8 == 0), S in
// {1, 2, 4, 8} with at least one chunk of K per part, 16-byte aligned rows.
int rows_linear(const void* x, int64_t ld_x, const void* w, const void* bias, bool bias_f32, float* part, void* out,
                int* tickets, int T, int N, int K, int S, int act, float p0, float p1, int cols, hipStream_t st) {
  const bool gated = act >= kActGlu, whole = cols < (gated ? 128 : 64);
  if (T < 1 || T > 64 || N < 1 || K < 128 || K % 128 || N % (gated ? 8 : 4) || ld_x % 8 ||
      (gated && (bias || !xgk::glu_known(act - kActGlu))) || act < 0 || (S != 1 && S != 2 && S != 4 && S != 8) || S > K / 128 ||
      (S > 1 && !part) || (S > 1 && !tickets && (act != kActNone || bias)) ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)bias | (uintptr_t)part) & 15) || ((uintptr_t)out & 7) ||
      (!out && (S == 1 || tickets)) || (whole && S != 1) ||
      !(gated ? cols == 32 || cols == 64 || cols == 128 : cols == 16 || cols == 32 || cols == 48 || cols == 64 || cols == 128))
    return -1;
  RowsArgs a = {(const bf16*)x, (const bf16*)w, bias, part, (bf16*)out, tickets, ld_x, T, N, K, act, p0, p1, bias_f32};
  if (whole) {   // (groups of waves side by side where the rows of x fill their loads)
    if (T <= 16) rows_whole<1, 10, 1, 2, 6, 1, 4>(a, cols, st);
    else if (T <= 32) rows_whole<2, 6, 1, 2, 4, 1, 4>(a, cols, st);
    else if (T <= 48) rows_whole<3, 4, 1, 2, 4, 1, 4>(a, cols, st);
    else rows_whole<4, 4, 2, 1, 4, 2, 2>(a, cols, st);
    return 0;
  }
  const bool wide = cols == 128;
  const dim3 grid((N + cols - 1) / cols, S);
  // (128 weight rows: two x tiles also for up to 16 rows, 28672 x 4096 gated 40.4 us against 42.0 with one tile, 256-byte rows and
  // 144 KB of LDS; 32000 x 4096 43.5 against 45.5)
  if (T <= 16 && !wide) {
    rows_linear_kernel<1, 1, 4, 128, 4><<<grid, 256, 0, st>>>(a);
  } else if (T <= 32) {
    if (wide) rows_linear_kernel<2, 2, 4, 64, 6><<<grid, 256, 0, st>>>(a);
    else rows_linear_kernel<2, 1, 4, 64, 6><<<grid, 256, 0, st>>>(a);
  } else {
    if (wide) rows_linear_kernel<4, 2, 4, 64, 3><<<grid, 256, 0, st>>>(a);
    else rows_linear_kernel<4, 1, 4, 64, 4><<<grid, 256, 0, st>>>(a);
  }
  return 0;
}
}  // namespace xgm
