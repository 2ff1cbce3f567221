// Products of many activation rows (prompt steps) with a weight matrix, and what follows them:
//
//   tile_linear         out [M, N] = act(x [M, K] . w [N, K]^T + bias), or a gated activation of w's gate and up rows
//   tile_linear_sum     the same from the fp32 slabs that S parts of K leave
//
// Bound by the matrix cores from some 400 rows on, by the weights' bytes below. A workgroup of four waves, one per SIMD, owns a tile
// of 32 FM rows and 32 FN weight rows, 2 x 2 waves of 16 FM x 16 FN: with 128 x 128 products a wave reads 32 fragments from LDS per
// 128 matrix instructions (the tile 64 per 32 of K; eight waves of 128 x 64 read 96), and its accumulators fill the 256 accumulation
// registers.
// x and w come in by LDS DMA, 64 of K at a time, into a ring of RA and RW slots (160 KB for the large tiles: two of x, three of w,
// whose first reader waits for HBM). A K tile is two steps, one per 32 of K. Between the products of a step the other step's fragments
// are read (into the registers that the step before has used up) and, once the K tile's slots are free, the tiles RA and RW further on
// asked for, one instruction after every few products: in bunches they hold the matrix pipe up (8192 x 2048 x 8192, us: 211 in bunches
// and with a branch each, 184 one at a time). One barrier per K tile. The 16-byte granules of a row are permuted by the row, so that the
// reads of 16 rows fall on all banks; w's rows are dealt to the fragments in fours, so that a lane ends up with eight neighbouring
// columns (one 16-byte store), or with four gate and the four up columns they go with.
//
// Workgroups stay and take tile after tile: the next tile's first loads go out ahead of a tile's stores (8192 x 8192 x 2048: 229 us with
// a workgroup per tile, 200 so). S parts of K fill the chip where the tiles are few; their slabs are added by a second launch.
//
// The grouped form (tile_grouped) walks the tiles of all experts' sorted rows one expert after the other, with the rows of x gathered
// through the sort; a tile ends where its expert's rows do. Both products of 8 experts with sorting and sum, us, against 64-row tiles of
// grouped_rows.hip or 192 to 288-row ones of gemm_pf (tokens, two experts each): 2 x 3584 x 4096 300 240 -> 152, 700 242 -> 189, 4000
// 744 -> 631, 8192 1401 -> 1300; 2 x 2048 x 2048 1000 129 -> 85; 32 experts of 2 x 1024 x 2048, four each, 2000 239 -> 194.
//
// Measured, cold weights, us, against the library's product without what follows (M x N x K): 128 x 4096 x 14336 34 against 72;
// 512 x 4096 x 14336 64 against 86; 300 x 10304 x 2048 20 against 24; 2521 x 10304 x 2048 88 against 96; 4001 x 18560 x 4096 438 against 554;
// gated, 2521 x 16384 x 2048 141 against 192 with its activation, 8192 x 28672 x 4096 1319 against 1404; 8192 x 4096 x 14336 645 against 599
// (1.49 PFLOP/s at the power limit: the library's has the better of it in long plain products, which stay there).
#include <type_traits>

#include "attention_common.h"
#include "glds.h"
#include "glu.h"

namespace xgm {
using xgk::bf16x8_t;
using xgk::f32x4_t;

enum { kTileNone = 0, kTileXielu = 1, kTileRelu2 = 2, kTileGlu = 3 };   // kTileGlu + kind: glu.h
enum { kPairNone = 0, kPairHalves = 1, kPairBlocks = 2 };               // w's rows: [gate | up], or 16 gate, 16 up, ...

// Up to so many rows (grouped: per expert) neighbouring column tiles start at different places in K: else all of them ask for the same
// column of weight rows 2 K bytes apart, which few memory channels hold, at the same time. With more rows the workgroups of one row tile
// gain more from reading its rows together. us without / with: 128 x 28672 x 4096 57 / 50, 128 x 18560 x 4096 50 / 46, 192 x 4096 x 8192 31 /
// 29, 400 x 18560 x 4096 73 / 77, 1024 x 2048 x 8192 45 / 80; both products of 8 experts of 2 x 3584 x 4096 with 75 rows each 176 / 152,
// with 250 290 / 270.
constexpr int kRotateRows = 256;

struct TileArgs {
  const bf16 *x, *w;
  const void* bias;        // [N] fp32 or bf16, or nullptr
  float* part;             // [S, M, N] fp32 (gated: [gate | up] whatever the rows' order), or nullptr: the result is `out`
  bf16* out;               // [M, N], or [M, N / 2] for the gated activations (S > 1: what the slabs' sum is written to)
  int64_t ld_x;
  int M, N, K, S, act, pairs;
  float p0, p1;
  bool bias_f32;
  // grouped: row p of the experts' sorted rows is row rows[p] / top of x (rows nullptr: p; pads below 0: any), expert e's are
  // offs[e] .. offs[e + 1], its weights w + e w_stride
  const int32_t *rows, *offs;
  int E, top;
  int64_t w_stride;
  bool rotate;             // column tiles start at different K tiles
};

// LDS DMA of 16 bytes a lane from a uniform base and a lane's byte offset
__device__ __forceinline__ void tile_dma(const void* base, uint32_t off, uint32_t lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "{m0}"(lds) : "memory");
#endif
}

// acc += w . x^T in accumulation registers. (From the builtin hipcc moves accumulators between the two register files inside the
// loop, some 100 moves per 64 products. It puts no waits between these: an accumulator is read again by the same instruction on the
// same registers, which takes two wait states at most, and FM FN - 1 other products lie between, kMfmaApart at least; what follows the
// loop waits.)
constexpr int kMfmaApart = 5;
__device__ __forceinline__ void tile_mfma(f32x4_t& acc, bf16x8_t w, bf16x8_t x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(x));
#endif
}

// the accumulators' values (volatile as the products: behind the wait that follows them; one fragment at a time, or all of them would
// come into vector registers at once)
__device__ __forceinline__ f32x4_t tile_take(const f32x4_t& acc) {
  f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v[0]) : "a"(acc[0]));
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v[1]) : "a"(acc[1]));
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v[2]) : "a"(acc[2]));
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v[3]) : "a"(acc[3]));
#endif
  return v;
}

__device__ __forceinline__ void tile_bias(const TileArgs& a, int col, float* b) {
  float v[4];
  if (a.bias_f32) ld4((const float*)a.bias + col, v);
  else ld4((const bf16*)a.bias + col, v);
#pragma unroll
  for (int e = 0; e < 4; ++e) b[e] = v[e];
}
template <int ACT>
__device__ __forceinline__ float tile_act(const TileArgs& a, float v) {
  return ACT == kTileXielu ? xieluf(v, a.p0, a.p1) : ACT == kTileRelu2 ? relu2f(v) : v;
}
// glu.h's gates for a bf16 result, whose rounding is 2^-9: the exponential and reciprocal instructions (2^-23 each, and 2^-24 of the
// exponent from its rounding) instead of expf and a division, 20 instructions an output instead of 45. A tile's gates run on four waves while its matrix cores wait: 8192 x 16384 x 2048
// 440 -> 405 us, 2521 rows 152 -> 141, 8192 x 28672 x 4096 1381 -> 1319. Error of the result against fp64 over gates and factors of spread
// 0.3, 1 and 3: 1.649554e-3, 1.660321e-3, 1.654740e-3 (tanh-GELU; the others likewise), the same to seven digits as with those.
template <int KIND>
__device__ __forceinline__ float tile_glu(const TileArgs& a, float g, float u) {
  if (KIND == xgk::kGluClamped) g = fminf(g, a.p0), u = fminf(fmaxf(u, -a.p0), a.p0) + 1.f;
  const float z = KIND == xgk::kGluGeluTanh ? fmaf(0.044715f * g * g, g, g) : g;
  const float c = KIND == xgk::kGluGeluTanh ? -2.302208198f : KIND == xgk::kGluClamped ? -kLog2e * a.p1 : -kLog2e;   // 2 sqrt(2 / pi) log2 e
  return g * rcp_fast(1.f + exp2_fast(c * z)) * u;
}

// f(the activation as a constant): one branch for a whole epilogue
template <bool PAIR, typename F>
__device__ __forceinline__ void tile_by_act(const TileArgs& a, F f) {
  if constexpr (PAIR) {
    if (a.act == kTileGlu + xgk::kGluGeluTanh) f(std::integral_constant<int, xgk::kGluGeluTanh>{});
    else if (a.act == kTileGlu + xgk::kGluClamped) f(std::integral_constant<int, xgk::kGluClamped>{});
    else f(std::integral_constant<int, xgk::kGluSilu>{});
  } else {
    if (a.act == kTileXielu) f(std::integral_constant<int, kTileXielu>{});
    else if (a.act == kTileRelu2) f(std::integral_constant<int, kTileRelu2>{});
    else f(std::integral_constant<int, kTileNone>{});
  }
}

template <int FM, int FN, int RA, int RW, int OCC, bool PAIR, bool GRP>
__global__ __launch_bounds__(256, OCC) void tile_linear_kernel(const TileArgs a) {
  constexpr int BM = 32 * FM, BN = 32 * FN, ASZ = BM * 128, WSZ = BN * 128;
  constexpr int LD = FM + FN;                      // fragment reads of a step, and DMA instructions of a K tile, per wave
  constexpr int ST = FM * FN / 2;   // stores of a whole tile (fp32 parts: twice that)
  constexpr int RS = FM * FN >= 2 * LD ? 3 * FM * FN / 4 / LD : 1, DS = FM * FN / LD;   // products between two reads (the last has a quarter to land), two loads
  static_assert(RS >= 1 && DS >= 1, "a step's reads and loads fit between its products");
  static_assert(FM * FN > kMfmaApart, "products on the same accumulators keep their distance");
  // loads behind the last one that the next tile needs (A of RA tiles ahead and then W of RW tiles ahead are asked for per tile)
  constexpr int CA = FN + (RA - 2) * LD, CW = (RW - 2) * LD, CNT = CA < CW ? CA : CW;
  constexpr int CA0 = FN + (RA - 1) * LD, CW0 = (RW - 1) * LD, CNT0 = CA0 < CW0 ? CA0 : CW0;   // ... and that tile 0 needs
  static_assert(RA >= 2 && RW >= RA && RW <= RA + 1 && OCC * (RA * ASZ + RW * WSZ) <= 160 * 1024 && CNT < 64, "tile_linear geometry");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[RA * ASZ + RW * WSZ];
  const int lane = threadIdx.x & 63, g4 = lane >> 4, l16 = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wv >> 1, wn = wv & 1;

  const int TN = (a.N + BN - 1) / BN;
  int total = (a.M + BM - 1) / BM * TN * a.S;
  if constexpr (GRP) {
    total = 0;
    for (int e = 0; e < a.E; ++e) total += (a.offs[e + 1] - a.offs[e] + BM - 1) / BM * TN;
    if ((int)blockIdx.x >= total) return;
  }
  const int nk_all = a.K / 64, half = a.N / 2, dr = lane >> 3, dj = lane & 7;
  int m0, m_hi = a.M, n0, s, nk, rot;
  uint32_t ao[FM], wo[FN];
  const char *xb, *wb;
  // the tile at place `at` of the order: neighbours on one XCD, columns of up to 8 row tiles next to each other. And what this
  // lane asks for: A pieces wv FM + i, W pieces wv FN + i, 8 rows of 128 bytes each.
  auto place = [&](int done) __attribute__((always_inline)) {
    const int nb = min((int)gridDim.x, total - done), bid = blockIdx.x, q8 = nb >> 3, r8 = nb & 7, xcd = bid & 7;
    const int v = done + (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (bid >> 3);
    int TM = (a.M + BM - 1) / BM, u = v, lo = 0, e = 0;
    if constexpr (GRP) {   // the experts' tiles one expert after the other
      for (;; ++e) {
        lo = a.offs[e], m_hi = a.offs[e + 1], TM = (m_hi - lo + BM - 1) / BM;
        if (u < TM * TN) break;
        u -= TM * TN;
      }
      s = 0;
    } else {
      s = v / (TM * TN), u = v - s * TM * TN;
    }
    const int GM = TM < 8 ? TM : 8, gid = u / (GM * TN), first = gid * GM;
    const int gm = TM - first < GM ? TM - first : GM, ug = u - gid * GM * TN;
    m0 = lo + (first + ug % gm) * BM, n0 = (ug / gm) * BN;
    const int kt_lo = s * nk_all / a.S;
    nk = (s + 1) * nk_all / a.S - kt_lo;
    rot = a.rotate ? (int)((unsigned)(ug / gm) * 37u % (unsigned)nk) : 0;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      int r = min(m0 + 8 * (wv * FM + i) + dr, m_hi - 1);
      if (GRP && a.rows) r = max(a.rows[r], 0) / a.top;
      ao[i] = (uint32_t)(GRP ? r : r - m0) * (uint32_t)(2 * a.ld_x) + 16 * (dj ^ dr);
    }
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const int p = wv * FN + i;
      int r;
      if (PAIR) {
        const int c = min(n0 / 2 + 4 * p + (dr & 3), half - 1);
        r = a.pairs == kPairHalves ? c + (dr >> 2) * half : 2 * (c & ~15) + (c & 15) + (dr >> 2) * 16;
      } else {
        r = min(n0 + 8 * p + dr, a.N - 1);
      }
      wo[i] = (uint32_t)r * (uint32_t)(2 * a.K) + 16 * (dj ^ ((dr & 3) | ((p & 1) << 2)));
    }
    xb = reinterpret_cast<const char*>(a.x + (GRP ? 0 : (int64_t)m0 * a.ld_x) + kt_lo * 64);
    wb = reinterpret_cast<const char*>(a.w + (GRP ? e * a.w_stride : 0) + kt_lo * 64);
  };
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t) reinterpret_cast<uintptr_t>((xgk::lds_void_t*)lds));
  auto dma = [&](int i, int t, int sa, int sw) __attribute__((always_inline)) {   // i-th of tile t's loads: A of tile t, or W of tile t
    int kt = t + rot;
    kt = kt >= nk ? kt - nk : kt;
    if (i < FM) tile_dma(xb + (int64_t)kt * 128, ao[i], lds0 + sa * ASZ + (wv * FM + i) * 1024);
    else tile_dma(wb + (int64_t)kt * 128, wo[i - FM], lds0 + RA * ASZ + sw * WSZ + (wv * FN + i - FM) * 1024);
  };

  // ---- fragment reads: x row 16 i + l16, W row 32 (i / 2) + 8 (l16 / 4) + l16 % 4 + 4 (i % 2); K half ks
  const uint8_t* ap = lds + (wm * 16 * FM + l16) * 128;
  const uint8_t* wp = lds + RA * ASZ + (wn * 16 * FN + 8 * (l16 >> 2) + (l16 & 3)) * 128;
  const int ka = 16 * (g4 ^ (l16 & 7)), kw = 16 * (g4 ^ ((l16 & 3) | (((l16 >> 2) & 1) << 2)));
  bf16x8_t af[2][FM], wf[2][FN];
  auto read = [&](int i, int ks, int sa, int sw) __attribute__((always_inline)) {   // x 0, all of W, the rest of x; where W is the larger: W 0, all of x, the rest of W
    constexpr bool XL = FM >= FN;
    if (XL ? i == 0 || i > FN : i >= 1 && i <= FM) {
      const int j = XL ? (i == 0 ? 0 : i - FN) : i - 1;
      af[ks][j] = *reinterpret_cast<const bf16x8_t*>(ap + sa * ASZ + j * 2048 + (ka ^ (64 * ks)));
    } else {
      const int j = XL ? i - 1 : (i == 0 ? 0 : i - FM);
      wf[ks][j] = *reinterpret_cast<const bf16x8_t*>(wp + sw * WSZ + (j >> 1) * 4096 + (j & 1) * 512 + (kw ^ (64 * ks)));
    }
  };
  f32x4_t acc[FM][FN];
  auto prologue = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = -RW; t < 0; ++t) {
      if (t + RA >= 0 && t + RA < nk)
#pragma unroll
        for (int i = 0; i < FM; ++i) dma(i, t + RA, t + RA, 0);
      if (t + RW < nk)
#pragma unroll
        for (int i = FM; i < LD; ++i) dma(i, t + RW, 0, t + RW);
    }
  };
  int sa, sw;          // slots of tile t
  bool behind;         // the last tile's ST stores are behind the prologue's loads

  // one step: the products of K half KS, and between them the other half's reads and (second half) the next loads, one at a time;
  // FULL: tiles t + RA and t + RW exist
  auto step = [&](int t, auto ks_c, auto full_c, int ra, int rw) __attribute__((always_inline)) {
    constexpr int KS = decltype(ks_c)::value;
    constexpr bool FULL = decltype(full_c)::value;
#pragma unroll
    for (int q = 0; q < FM * FN; ++q) {
      const int m = FM >= FN ? q / FN : q % FM, n = FM >= FN ? q % FN : q / FM;
      tile_mfma(acc[m][n], wf[KS][n], af[KS][m]);
      if (q % RS == 0 && q / RS < LD) read(q / RS, KS ^ 1, ra, rw);
      if (KS == 1 && q % DS == DS / 2 && q / DS < LD) {
        const int j = q / DS;
        if (FULL || t + (j < FM ? RA : RW) < nk) dma(j, t + (j < FM ? RA : RW), sa, sw);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto tile = [&](int t, auto full_c) __attribute__((always_inline)) {
    constexpr bool FULL = decltype(full_c)::value;
    step(t, std::integral_constant<int, 0>{}, full_c, sa, sw);
    // tile t's slots are read; tile t + 1 has landed, in every wave
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (FULL || t - 1 + RW < nk) {
      if (FULL && t == 0 && behind) xgk::wait_vmcnt<(CNT + ST < 63 ? CNT + ST : 63)>();
      else xgk::wait_vmcnt<CNT>();
    } else {
      xgk::wait_vmcnt<0>();
    }
    xgk::raw_barrier();
    const int na = sa + 1 == RA ? 0 : sa + 1, nw = sw + 1 == RW ? 0 : sw + 1;
    step(t, std::integral_constant<int, 1>{}, full_c, na, nw);
    sa = na, sw = nw;
  };
  place(0);
  prologue();
  behind = false;
  for (int done = 0;;) {
#pragma unroll
    for (int m = 0; m < FM; ++m)
#pragma unroll
      for (int n = 0; n < FN; ++n) {
        acc[m][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+a"(acc[m][n]));
      }
    asm volatile("s_nop 3" ::: "memory");   // (a product's accumulators may not be written right before it)
    if (RW - 1 < nk) {
      if (behind) xgk::wait_vmcnt<(CNT0 + ST < 63 ? CNT0 + ST : 63)>();
      else xgk::wait_vmcnt<(CNT0 < 63 ? CNT0 : 63)>();
    } else {
      xgk::wait_vmcnt<0>();
    }
    xgk::raw_barrier();
    sa = sw = 0;
#pragma unroll
    for (int i = 0; i < LD; ++i) read(i, 0, 0, 0);
    const int col0 = PAIR ? n0 / 2 + wn * 8 * FN + 4 * g4 : n0 + wn * 16 * FN + 8 * g4, cols = PAIR ? half : a.N;
    // (the biases ahead of the loop, whose last tiles wait for all loads anyway: a load between the stores would wait for those)
    const bool biased = !PAIR && a.bias && !a.part;
    float b[FN / 2][8];
    if (!PAIR) {
#pragma unroll
      for (int j = 0; j < FN / 2; ++j) {
#pragma unroll
        for (int e = 0; e < 8; ++e) b[j][e] = 0.f;
        if (biased && col0 + 32 * j < cols) tile_bias(a, col0 + 32 * j, b[j]), tile_bias(a, col0 + 32 * j + 4, b[j] + 4);
      }
    }
    int t = 0;
    for (; t < nk - RW; ++t) tile(t, std::true_type{});
    for (; t < nk; ++t) tile(t, std::false_type{});
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // the last products' results

    // ---- a lane holds 8 neighbouring columns of a row (two fragments), or 4 gate and 4 up columns. The next tile's first loads go
    // ahead of the stores (every wave is past its reads of this one since the last barrier).
    const int row0 = m0 + wm * 16 * FM + l16, part = s, end = m_hi;
    behind = m0 + BM <= m_hi && n0 + BN <= a.N;
    done += gridDim.x;
    const bool more = done + (int)blockIdx.x < total;
    if (more) place(done), prologue();
    // f(row, column, j, the two fragments) of what lies inside
    auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
      for (int m = 0; m < FM; ++m) {
        const int row = row0 + 16 * m;
        if (row >= end) continue;
#pragma unroll
        for (int j = 0; j < FN / 2; ++j) {
          const int col = col0 + (PAIR ? 16 : 32) * j;
          if (col < cols) f(row, col, j, tile_take(acc[m][2 * j]), tile_take(acc[m][2 * j + 1]));
        }
      }
    };
    if (a.part) {
      each([&](int row, int col, int j, f32x4_t lo, f32x4_t hi) __attribute__((always_inline)) {
        float* at = a.part + ((int64_t)part * a.M + row) * a.N + col;
        *reinterpret_cast<f32x4_t*>(at) = lo;
        *reinterpret_cast<f32x4_t*>(at + (PAIR ? half : 4)) = hi;
      });
    } else {
      tile_by_act<PAIR>(a, [&](auto act_c) __attribute__((always_inline)) {
        constexpr int ACT = decltype(act_c)::value;
        if constexpr (PAIR) {
          each([&](int row, int col, int j, f32x4_t lo, f32x4_t hi) __attribute__((always_inline)) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = tile_glu<ACT>(a, lo[e], hi[e]);
            st4(a.out + (int64_t)row * half + col, v);
          });
        } else {
          each([&](int row, int col, int j, f32x4_t lo, f32x4_t hi) __attribute__((always_inline)) {
            float o[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = tile_act<ACT>(a, lo[e] + b[j][e]), o[4 + e] = tile_act<ACT>(a, hi[e] + b[j][4 + e]);
            *reinterpret_cast<uint4*>(a.out + (int64_t)row * a.N + col) = xgk::pack8(o);
          });
        }
      });
    }
    if (!more) break;
  }
}

template <bool PAIR>
__global__ __launch_bounds__(256) void tile_linear_sum_kernel(const TileArgs a) {
  const int cols = (PAIR ? a.N / 2 : a.N) / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, slab = (int64_t)a.M * a.N;
  if (i >= (int64_t)a.M * cols) return;
  const int64_t row = i / cols;
  const int col = 4 * (int)(i - row * cols);
  const float* at = a.part + row * a.N + col;
  float v[4];
  ld4(at, v);
  add_slabs(at, slab, a.S, v);
  float up[4], b[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (PAIR) {
    ld4(at + a.N / 2, up);
    add_slabs(at + a.N / 2, slab, a.S, up);
  } else if (a.bias) {
    tile_bias(a, col, b);
  }
  tile_by_act<PAIR>(a, [&](auto act_c) __attribute__((always_inline)) {
    constexpr int ACT = decltype(act_c)::value;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = PAIR ? tile_glu<ACT>(a, v[e], up[e]) : tile_act<ACT>(a, v[e] + b[e]);
  });
  st4(a.out + row * (PAIR ? a.N / 2 : a.N) + col, v);
}

template <int FM, int FN, int RA, int RW, int OCC>
static void tile_launch(const TileArgs& a, int cus, hipStream_t st) {
  const int tiles = ((a.M + 32 * FM - 1) / (32 * FM)) * ((a.N + 32 * FN - 1) / (32 * FN));
  const int grid = tiles * a.S < cus * OCC ? tiles * a.S : cus * OCC;
  if (a.pairs) tile_linear_kernel<FM, FN, RA, RW, OCC, true, false><<<grid, 256, 0, st>>>(a);
  else tile_linear_kernel<FM, FN, RA, RW, OCC, false, false><<<grid, 256, 0, st>>>(a);
}

template <int FM, int FN, int RA, int RW>
static void tile_launch_grouped(const TileArgs& a, int cus, hipStream_t st) {
  const int64_t tiles = (int64_t)(a.M / (32 * FM) + a.E) * ((a.N + 32 * FN - 1) / (32 * FN));   // at most
  const int grid = tiles < cus ? (int)tiles : cus;
  if (a.pairs) tile_linear_kernel<FM, FN, RA, RW, 1, true, true><<<grid, 256, 0, st>>>(a);
  else tile_linear_kernel<FM, FN, RA, RW, 1, false, true><<<grid, 256, 0, st>>>(a);
}

int tile_linear(const void* x, int64_t ld_x, const void* w, const void* bias, bool bias_f32, float* part, void* out, int M,
                int N, int K, int S, int act, int pairs, float p0, float p1, int fm, int fn, int cus, hipStream_t st) {
  const bool gated = act >= kTileGlu;
  if (M < 1 || N < 8 || N % 8 || K < 64 || K % 64 || ld_x < K || ld_x % 8 || S < 1 || S > K / 64 || act < 0 || gated != (pairs != 0) ||
      (gated && !xgk::glu_known(act - kTileGlu)) || cus < 1 || pairs < 0 || pairs > 2 || (gated && (bias || N % (pairs == kPairBlocks ? 32 : 8))) || (S > 1 && !part) ||
      (!out && (S == 1 || act != kTileNone || bias)) ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)bias | (uintptr_t)part | (uintptr_t)out) & 15) ||
      (int64_t)N * K * 2 >= (1LL << 32) || 256 * ld_x * 2 >= (1LL << 32))
    return -1;
  TileArgs a = {(const bf16*)x, (const bf16*)w, bias, S > 1 ? part : nullptr, (bf16*)out, ld_x, M, N, K, S, act, pairs, p0, p1, bias_f32,
                nullptr, nullptr, 0, 1, 0, M <= kRotateRows};
// (a round of workgroups costs the same full or nearly empty: sizes between the powers of two are there for the row counts that
// leave such a round; 160 x 192 and 128 x 192 were the fastest too rarely, by 1 to 6 %)
#define XGM_TILE(FM, FN, RA, RW, OCC) else if (fm == FM && fn == FN) tile_launch<FM, FN, RA, RW, OCC>(a, cus, st);
  if (false) {}
  XGM_TILE(8, 8, 2, 3, 1)
  XGM_TILE(7, 8, 2, 3, 1)
  XGM_TILE(6, 8, 2, 3, 1)
  XGM_TILE(5, 8, 2, 3, 1)
  XGM_TILE(4, 8, 3, 3, 1)
  XGM_TILE(8, 6, 2, 3, 1)
  XGM_TILE(7, 6, 3, 3, 1)
  XGM_TILE(6, 6, 3, 3, 1)
  XGM_TILE(8, 4, 3, 4, 1)
  XGM_TILE(7, 4, 3, 4, 1)
  XGM_TILE(6, 4, 4, 4, 1)
  XGM_TILE(5, 4, 4, 4, 1)
  XGM_TILE(4, 4, 5, 5, 1)
  XGM_TILE(3, 4, 5, 5, 1)
  XGM_TILE(4, 2, 6, 6, 1)
  XGM_TILE(3, 2, 3, 3, 2)
  else return -1;
#undef XGM_TILE
  if (S > 1 && out) {   // (without a result the slabs are it: the next kernel adds them)
    const int64_t n = (int64_t)M * (gated ? N / 2 : N) / 4;
    if (gated) tile_linear_sum_kernel<true><<<(unsigned)((n + 255) / 256), 256, 0, st>>>(a);
    else tile_linear_sum_kernel<false><<<(unsigned)((n + 255) / 256), 256, 0, st>>>(a);
  }
  return 0;
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
      x_rows * ld_x * 2 >= (1LL << 32))
    return -1;
  TileArgs a = {(const bf16*)x, (const bf16*)w, nullptr, y, (bf16*)out, ld_x, M, N, K, 1, act, gated ? kPairHalves : kPairNone, p0, p1,
                false, rows, offs, E, top, (int64_t)N * K, M <= (int64_t)kRotateRows * E};
#define XGM_TILE(FM, FN, RA, RW) else if (fm == FM && fn == FN) tile_launch_grouped<FM, FN, RA, RW>(a, cus, st);
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
