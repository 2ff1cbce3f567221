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
// are read (into the registers that the step before has used up) and the tiles RA and RW further on asked for, x in the second step and
// w in the next one's first, in even distances and not beside a read: with all of them in the second step, their addresses computed
// beside them, a K tile of 256 x 256 took 2670 clocks for 2048 of products, so 2400 (8192 x 4096 x 14336, us: 673 -> 625, of which 5 are
// the order of products, row after row there and back, so that the operand at the turn stays: less power). One barrier per K tile. The
// 16-byte granules of a row are permuted by the row, so that the
// reads of 16 rows fall on all banks; w's rows are dealt to the fragments in fours, so that a lane ends up with eight neighbouring
// columns (one 16-byte store), or with four gate and the four up columns they go with.
//
// Workgroups stay and take tile after tile, and the ring runs through: where a tile has RA tiles of K to go, the loads go over to the
// next one, and its first step takes the results out of an accumulator right before the product that starts it anew. The stores go
// through buffer descriptors, which drop what lies outside, so that there is no branch between the products. us, without (and
// with all loads in the second step) / with, on one box: 8192 x 8192 x 2048 228 / 208, 5000 x 5000 x 448 on 128 x 128 60 / 47, 8192 x 28672 x
// 4096 gated 1336 / 1311 (the gates' vector work is the matrix cores' wait either way); one tile a workgroup, 512 x 6144 x 4096 41.8 / 40.6.
// S parts of K fill the chip where the tiles are few; their slabs are added by a second launch. K of one or two tiles has no ring to run:
// all of it is loaded first, a workgroup per tile (SHORT).
//
// The grouped form (tile_grouped) walks the tiles of all experts' sorted rows one expert after the other, with the rows of x gathered
// through the sort; a tile ends where its expert's rows do. Both products of 8 experts with sorting and sum, us, against 64-row tiles of
// grouped_rows.hip or 192 to 288-row ones of gemm_pf (tokens, two experts each): 2 x 3584 x 4096 300 240 -> 152, 700 242 -> 189, 4000
// 744 -> 631, 8192 1401 -> 1300; 2 x 2048 x 2048 1000 129 -> 85; 32 experts of 2 x 1024 x 2048, four each, 2000 239 -> 194.
//
// Measured, cold weights, us, against the library's product without what follows (M x N x K), on the same box: 128 x 4096 x 14336 37 against
// 79; 512 x 4096 x 14336 72 against 95; 300 x 10304 x 2048 23 against 28; 2521 x 10304 x 2048 98 against 105; 4001 x 18560 x 4096 447 against
// 560; gated, 2521 x 16384 x 2048 140 against 191 with its activation, 8192 x 28672 x 4096 1311 against 1417; 8192 x 4096 x 14336 625 against
// 615 (1.54 PFLOP/s at the power limit: the library's has the better of it in long plain products, which stay there).
#pragma once

#include <type_traits>
#include <utility>

#include "attention_common.h"
#include "glds.h"
#include "glu.h"

namespace xgm {
using xgk::bf16x8_t;
using xgk::f32x4_t;

enum { kTileNone = 0, kTileXielu = 1, kTileRelu2 = 2, kTileGlu = 3, kTilePart = -1 };   // kTileGlu + kind: glu.h
enum { kPairNone = 0, kPairHalves = 1, kPairBlocks = 2 };               // w's rows: [gate | up], or 16 gate, 16 up, ...

// Up to so many rows (grouped: per expert) neighbouring column tiles start at different places in K: else all of them ask for the same
// column of weight rows 2 K bytes apart, which few memory channels hold, at the same time. With more rows the workgroups of one row tile
// gain more from reading its rows together. us without / with: 128 x 28672 x 4096 57 / 50, 128 x 18560 x 4096 50 / 46, 192 x 4096 x 8192 31 /
// 29, 400 x 18560 x 4096 73 / 77, 1024 x 2048 x 8192 45 / 80; both products of 8 experts of 2 x 3584 x 4096 with 75 rows each 176 / 152,
// with 250 290 / 270.
// All row tiles take K in the same order, so that a row's result does not depend on where it is in the step. (With up to eight of them in
// orders of their own, each fetching a share of the weight that the others find in L2, a Llama prompt of 512 takes 2042 us instead of
// 2162, and equal rows differ by a rounding.)
constexpr int kRotateRows = 256;
constexpr int kTileColumns = 1 << 22;   // a wave's 128 rows of fp32 results are less than 2^31 bytes

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
  int rotate;              // groups of so many columns start at different K tiles (0: all at the first)
};

// LDS DMA of 16 bytes a lane from a uniform base and a lane's byte offset
__device__ __forceinline__ void tile_dma(const void* base, uint32_t off, uint32_t lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "{m0}"(lds) : "memory");
#endif
}

// Accumulator I of a wave: accumulation registers 4 I .. 4 I + 3, by name. (As values of the compiler's they are moved between register
// files inside the loop, some 100 moves per 64 products, and where a branch joins two ways to write them, behind a product that has
// not written them yet. Every statement names what it writes, but the compiler does not know that these registers hold something
// between two statements: the build looks whether it has put anything of its own there, and fails if so, _build.check_accumulators.)
// There are no waits between products: an accumulator is read again by the same
// instruction on the same registers, which takes two wait states at most, and kMfmaApart other products lie between at least.
//   mul, mul_dma, first   acc += w . x^T; the same and an LDS DMA behind it (M0 is written ahead of the product, which is the wait
//                         state between the two); acc = w . x^T
//   take                  the value, kMfmaApart products or a wait behind the last product on it
constexpr int kMfmaApart = 4;
template <int I>
struct TileAcc;
#if defined(__HIP_DEVICE_COMPILE__)
#define XGM_ACC_MUL(A, D) "v_mfma_f32_16x16x32_bf16 a[" #A ":" #D "], %0, %1, a[" #A ":" #D "]"
#define XGM_ACC_ASM(...) asm volatile(__VA_ARGS__)
#else
#define XGM_ACC_ASM(...)
#endif
#define XGM_ACC(I, A, B, C, D)                                                                                                     \
  template <>                                                                                                                      \
  struct TileAcc<I> {                                                                                                              \
    static __device__ __forceinline__ void mul(bf16x8_t w, bf16x8_t x) {                                                          \
      XGM_ACC_ASM(XGM_ACC_MUL(A, D) : : "v"(w), "v"(x) : "a" #A, "a" #B, "a" #C, "a" #D);                                          \
    }                                                                                                                              \
    static __device__ __forceinline__ void first(bf16x8_t w, bf16x8_t x) {                                                        \
      XGM_ACC_ASM("v_mfma_f32_16x16x32_bf16 a[" #A ":" #D "], %0, %1, 0" : : "v"(w), "v"(x) : "a" #A, "a" #B, "a" #C, "a" #D);     \
    }                                                                                                                              \
    static __device__ __forceinline__ void mul_dma(bf16x8_t w, bf16x8_t x, const void* base, uint32_t off, uint32_t lds) {        \
      XGM_ACC_ASM(XGM_ACC_MUL(A, D) "\n\tglobal_load_lds_dwordx4 %2, %3"                                                          \
                  : : "v"(w), "v"(x), "v"(off), "s"(base), "{m0}"(lds) : "memory", "a" #A, "a" #B, "a" #C, "a" #D);                \
    }                                                                                                                              \
    static __device__ __forceinline__ f32x4_t take() {                                                                             \
      f32x4_t v = {0.f, 0.f, 0.f, 0.f};                                                                                            \
      XGM_ACC_ASM("v_accvgpr_read_b32 %0, a" #A : "=v"(v[0]));                                                                     \
      XGM_ACC_ASM("v_accvgpr_read_b32 %0, a" #B : "=v"(v[1]));                                                                     \
      XGM_ACC_ASM("v_accvgpr_read_b32 %0, a" #C : "=v"(v[2]));                                                                     \
      XGM_ACC_ASM("v_accvgpr_read_b32 %0, a" #D : "=v"(v[3]));                                                                     \
      return v;                                                                                                                    \
    }                                                                                                                              \
  };
XGM_ACC(0, 0, 1, 2, 3) XGM_ACC(1, 4, 5, 6, 7) XGM_ACC(2, 8, 9, 10, 11) XGM_ACC(3, 12, 13, 14, 15)
XGM_ACC(4, 16, 17, 18, 19) XGM_ACC(5, 20, 21, 22, 23) XGM_ACC(6, 24, 25, 26, 27) XGM_ACC(7, 28, 29, 30, 31)
XGM_ACC(8, 32, 33, 34, 35) XGM_ACC(9, 36, 37, 38, 39) XGM_ACC(10, 40, 41, 42, 43) XGM_ACC(11, 44, 45, 46, 47)
XGM_ACC(12, 48, 49, 50, 51) XGM_ACC(13, 52, 53, 54, 55) XGM_ACC(14, 56, 57, 58, 59) XGM_ACC(15, 60, 61, 62, 63)
XGM_ACC(16, 64, 65, 66, 67) XGM_ACC(17, 68, 69, 70, 71) XGM_ACC(18, 72, 73, 74, 75) XGM_ACC(19, 76, 77, 78, 79)
XGM_ACC(20, 80, 81, 82, 83) XGM_ACC(21, 84, 85, 86, 87) XGM_ACC(22, 88, 89, 90, 91) XGM_ACC(23, 92, 93, 94, 95)
XGM_ACC(24, 96, 97, 98, 99) XGM_ACC(25, 100, 101, 102, 103) XGM_ACC(26, 104, 105, 106, 107) XGM_ACC(27, 108, 109, 110, 111)
XGM_ACC(28, 112, 113, 114, 115) XGM_ACC(29, 116, 117, 118, 119) XGM_ACC(30, 120, 121, 122, 123) XGM_ACC(31, 124, 125, 126, 127)
XGM_ACC(32, 128, 129, 130, 131) XGM_ACC(33, 132, 133, 134, 135) XGM_ACC(34, 136, 137, 138, 139) XGM_ACC(35, 140, 141, 142, 143)
XGM_ACC(36, 144, 145, 146, 147) XGM_ACC(37, 148, 149, 150, 151) XGM_ACC(38, 152, 153, 154, 155) XGM_ACC(39, 156, 157, 158, 159)
XGM_ACC(40, 160, 161, 162, 163) XGM_ACC(41, 164, 165, 166, 167) XGM_ACC(42, 168, 169, 170, 171) XGM_ACC(43, 172, 173, 174, 175)
XGM_ACC(44, 176, 177, 178, 179) XGM_ACC(45, 180, 181, 182, 183) XGM_ACC(46, 184, 185, 186, 187) XGM_ACC(47, 188, 189, 190, 191)
XGM_ACC(48, 192, 193, 194, 195) XGM_ACC(49, 196, 197, 198, 199) XGM_ACC(50, 200, 201, 202, 203) XGM_ACC(51, 204, 205, 206, 207)
XGM_ACC(52, 208, 209, 210, 211) XGM_ACC(53, 212, 213, 214, 215) XGM_ACC(54, 216, 217, 218, 219) XGM_ACC(55, 220, 221, 222, 223)
XGM_ACC(56, 224, 225, 226, 227) XGM_ACC(57, 228, 229, 230, 231) XGM_ACC(58, 232, 233, 234, 235) XGM_ACC(59, 236, 237, 238, 239)
XGM_ACC(60, 240, 241, 242, 243) XGM_ACC(61, 244, 245, 246, 247) XGM_ACC(62, 248, 249, 250, 251) XGM_ACC(63, 252, 253, 254, 255)
#undef XGM_ACC

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
// exponent from its rounding) instead of expf and a division, 20 instructions an output instead of 45. A tile's gates run on four waves while
// its matrix cores wait: with rings that end with the tile, 8192 x 16384 x 2048 440 -> 405 us, 2521 rows 152 -> 141. Error of the result
// against fp64 over gates and factors of spread 0.3, 1 and 3: 1.649554e-3, 1.660321e-3, 1.654740e-3 (tanh-GELU; the others likewise), the
// same to seven digits as with those.
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

// the same in all lanes, and in a scalar register
__device__ __forceinline__ int tile_one(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ const char* tile_one(const char* p) {
  const uint64_t v = reinterpret_cast<uintptr_t>(p);
  uint64_t u = (uint64_t)(uint32_t)tile_one((int)(v >> 32)) << 32 | (uint32_t)tile_one((int)(uint32_t)v);
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_nop 4" : "+s"(u));   // (a load's base that a vector instruction wrote)
#endif
  return reinterpret_cast<const char*>(u);
}
// (what follows from it is computed where it is used, and takes no registers before)
__device__ __forceinline__ int tile_opaque(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(v));
#endif
  return v;
}

// A tile of the result: rows m0 .. hi - 1 (BM of them at most), columns n0 .., part s of K (nk K tiles of 64 from kt_lo on), expert e.
// K tiles are asked for from number `rot` on and around: the same for all row tiles, so that equal rows give equal bits.
struct TileAt { int m0, hi, n0, s, kt_lo, nk, rot, e; };
// ... number v of `total` = TN column tiles for every row tile and part: columns of up to 8 row tiles next to each other
template <int BM, int BN, bool GRP>
__device__ __forceinline__ TileAt tile_at(const TileArgs& a, int TN, int v) {
  TileAt t;
  int TM = (a.M + BM - 1) / BM, u = v, lo = 0;
  t.hi = a.M, t.s = t.e = 0;
  if constexpr (GRP) {   // the experts' tiles one expert after the other
    for (;; ++t.e) {
      lo = a.offs[t.e], t.hi = a.offs[t.e + 1], TM = (t.hi - lo + BM - 1) / BM;
      if (u < TM * TN) break;
      u -= TM * TN;
    }
  } else {
    t.s = v / (TM * TN), u = v - t.s * TM * TN;
  }
  const int GM = TM < 8 ? TM : 8, gid = u / (GM * TN), first = gid * GM;
  const int gm = TM - first < GM ? TM - first : GM, ug = u - gid * GM * TN, tn = ug / gm;
  t.m0 = lo + (first + ug - tn * gm) * BM, t.n0 = tn * BN;
  const int nk_all = a.K / 64;
  t.kt_lo = t.s * nk_all / a.S;
  t.nk = (t.s + 1) * nk_all / a.S - t.kt_lo;
  t.rot = a.rotate ? (unsigned)(t.n0 / a.rotate) * 37u % (unsigned)t.nk : 0;
  return t;
}
// the block's place among nb neighbours in that order: neighbours on one XCD
__device__ __forceinline__ int tile_order(int nb) {
  const int bid = blockIdx.x, q8 = nb >> 3, r8 = nb & 7, xcd = bid & 7;
  return (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (bid >> 3);
}
// what a lane asks for of a K tile, from the tile's bases: x pieces wv FM + i, w pieces wv FN + i, 8 rows of 128 bytes each
template <int FM, int FN, bool PAIR, bool GRP>
__device__ __forceinline__ void tile_offsets(const TileArgs& a, const TileAt& t, int wv, int lane, uint32_t (&ao)[FM], uint32_t (&wo)[FN]) {
  const int at = tile_opaque(lane), dr = at >> 3, dj = at & 7, half = a.N / 2;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    int r = min(8 * (wv * FM + i) + dr, t.hi - 1 - t.m0);
    if (GRP) r += t.m0;
    if (GRP && a.rows) r = max(a.rows[r], 0) / a.top;
    ao[i] = (uint32_t)r * (uint32_t)(2 * a.ld_x) + 16 * (dj ^ dr);
  }
#pragma unroll
  for (int i = 0; i < FN; ++i) {
    const int p = wv * FN + i;
    int r;
    if (PAIR) {
      const int c = min(t.n0 / 2 + 4 * p + (dr & 3), half - 1);
      r = a.pairs == kPairHalves ? c + (dr >> 2) * half : 2 * (c & ~15) + (c & 15) + (dr >> 2) * 16;
    } else {
      r = min(t.n0 + 8 * p + dr, a.N - 1);
    }
    wo[i] = (uint32_t)r * (uint32_t)(2 * a.K) + 16 * (dj ^ ((dr & 3) | ((p & 1) << 2)));
  }
}

// Where a wave's results go: a lane holds 8 neighbouring columns of a row (two fragments), or 4 gate and 4 up columns. Through a buffer
// descriptor of the rows that there are: a lane outside stores nothing, and needs no branch.
template <bool PAIR>
struct TileOut {
  char* dst;
  uint32_t bytes, place, at, row_bytes, esz, half;   // place: this lane's row and columns from the first; at: with a column group's
  int cols, g4;
  // `rows` rows from row `row` on, columns from `col` of the result on
  __device__ __forceinline__ void start(const TileArgs& a, int s, int row, int rows, int col, int l16, int g) {
    half = a.N / 2, cols = PAIR ? half : a.N, esz = a.part ? 4 : 2, row_bytes = (uint32_t)(a.part ? a.N : cols) * esz, g4 = g;
    char* base = a.part ? reinterpret_cast<char*>(a.part) + ((int64_t)s * a.M + row) * row_bytes + col * 4
                        : reinterpret_cast<char*>(a.out) + (int64_t)row * row_bytes + col * 2;
    const uint32_t all = (uint32_t)max(0, rows) * row_bytes;   // (the last row ends col columns ahead of so many bytes)
    dst = const_cast<char*>(tile_one(base)), bytes = tile_one(all > col * esz ? all - col * esz : 0u);
    place = (uint32_t)tile_opaque(l16) * row_bytes + (PAIR ? 4 : 8) * g4 * esz;
  }
  __device__ __forceinline__ void columns(int j, int col) {   // group j, lane 0's first column being `col`
    at = (PAIR ? 4 : 8) * g4 < cols - col ? place + (PAIR ? 16 : 32) * j * esz : 0x80000000u;   // (a wave's rows are less than 2^31 bytes)
  }
  template <int ACT>
  __device__ __forceinline__ void put(const TileArgs& a, int m, f32x4_t lo, f32x4_t hi, const float (&b)[8]) {
    typedef __attribute__((ext_vector_type(4))) uint32_t u4;
    typedef __attribute__((ext_vector_type(2))) uint32_t u2;
    const uint32_t off = at + 16 * m * row_bytes;
    const auto to = __builtin_amdgcn_make_buffer_rsrc(dst, 0, bytes, 0x00020000);
    if constexpr (ACT == kTilePart) {
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, lo), to, off, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, hi), to, PAIR ? off + half * 4 : off + 16, 0, 0);
    } else if constexpr (PAIR) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = tile_glu<ACT>(a, lo[e], hi[e]);
      __builtin_amdgcn_raw_buffer_store_b64(u2{xgk::pack2(v[0], v[1]), xgk::pack2(v[2], v[3])}, to, off, 0, 0);
    } else {
      float o[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = tile_act<ACT>(a, lo[e] + b[e]), o[4 + e] = tile_act<ACT>(a, hi[e] + b[4 + e]);
      const u4 v = {xgk::pack2(o[0], o[1]), xgk::pack2(o[2], o[3]), xgk::pack2(o[4], o[5]), xgk::pack2(o[6], o[7])};
      __builtin_amdgcn_raw_buffer_store_b128(v, to, off, 0, 0);
    }
  }
};

// f(0) .. f(N - 1), each index a constant
template <typename F, int... I>
__device__ __forceinline__ void tile_each(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void tile_each(F f) {
  tile_each(std::make_integer_sequence<int, N>{}, f);
}
// the load behind product q (-1: none): n of them in even distances dist, but not beside a read (one every rs products)
constexpr int tile_load_at(int q, int n, int dist, int rs) {
  for (int j = 0; j < n; ++j) {
    int p = dist * j + dist / 2;
    if (p % rs == 0 && dist > 2 && rs > 1) ++p;
    if (p == q) return j;
  }
  return -1;
}
constexpr int tile_loads(int products, int n, int dist, int rs) {
  int found = 0;
  for (int q = 0; q < products; ++q) found += tile_load_at(q, n, dist, rs) >= 0;
  return found;
}

template <int FM, int FN, int RA, int RW, int OCC, bool PAIR, bool GRP, bool SHORT>
// (one wave per SIMD as the bound, also where two workgroups fit a CU, with 180 registers a wave: for two the compiler keeps to 128 vector
// registers and puts the rest where the accumulators are)
__global__ __launch_bounds__(256, 1) void tile_linear_kernel(const TileArgs a) {
  constexpr int BM = 32 * FM, BN = 32 * FN, ASZ = BM * 128, WSZ = BN * 128;
  constexpr int LD = FM + FN;                      // fragment reads of a step, and DMA instructions of a K tile, per wave
  constexpr int ST = FM * FN / 2;                  // stores of a whole tile (fp32 parts: twice that)
  constexpr int RS = FM * FN >= 2 * LD ? 3 * FM * FN / 4 / LD : 1;   // products between two reads (the last has a quarter of the step to land)
  static_assert(FM * FN > kMfmaApart + 1, "products on the same accumulators keep their distance");
  // loads that may be under way where tile t + 1 has to be there (x of tile t + RA follows half way through tile t, w of tile t + RW one
  // step later), and where tile 0 has to
  constexpr int CA = FN + (RA - 2) * LD, CW = (RW - 2) * LD, CNT = CA < CW ? CA : CW;
  constexpr int CA0 = (RA - 1) * LD, CW0 = (RW - 1) * LD - FN, CNT0 = CA0 < CW0 ? CA0 : CW0;
  constexpr int TB = RW == RA ? RA - 2 : RA - 1;   // ... to which the stores of the tile before come up to here
  static_assert(tile_loads(FM * FN, FM, FN, RS) == FM && tile_loads(FM * FN, FN, FM, RS) == FN, "every load has its place");
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
  TileAt ld, cur;      // the tile that is loaded, and the one whose products run
  uint32_t ao[FM], wo[FN], kx, kw;   // what this lane asks for; place in a row
  const char *xb, *wb;
  int done = 0;
  auto place = [&]() __attribute__((always_inline)) {   // the block's next tile
    ld = tile_at<BM, BN, GRP>(a, TN, done + tile_order(min((int)gridDim.x, total - done)));
    tile_offsets<FM, FN, PAIR, GRP>(a, ld, wv, lane, ao, wo);
    xb = tile_one(reinterpret_cast<const char*>(a.x + (GRP ? 0 : (int64_t)ld.m0 * a.ld_x) + ld.kt_lo * 64));
    wb = tile_one(reinterpret_cast<const char*>(a.w + (GRP ? ld.e * a.w_stride : 0) + ld.kt_lo * 64));
    ld.m0 = tile_one(ld.m0), ld.hi = tile_one(ld.hi), ld.n0 = tile_one(ld.n0), ld.s = tile_one(ld.s), ld.nk = tile_one(ld.nk);
    kx = kw = tile_one(ld.rot) * 128u;
  };
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t) reinterpret_cast<uintptr_t>((xgk::lds_void_t*)lds));
  const uint32_t lds_a = lds0 + wv * FM * 1024, lds_w = lds0 + RA * ASZ + wv * FN * 1024;
  auto next = [&](uint32_t& k) __attribute__((always_inline)) { k = k + 128 == (uint32_t)ld.nk * 128 ? 0 : k + 128; };

  // ---- fragment reads: x row 16 i + l16, W row 32 (i / 2) + 8 (l16 / 4) + l16 % 4 + 4 (i % 2); K half ks
  const uint8_t* ap = lds + (wm * 16 * FM + l16) * 128;
  const uint8_t* wp = lds + RA * ASZ + (wn * 16 * FN + 8 * (l16 >> 2) + (l16 & 3)) * 128;
  const int fa = 16 * (g4 ^ (l16 & 7)), fw = 16 * (g4 ^ ((l16 & 3) | (((l16 >> 2) & 1) << 2)));
  bf16x8_t af[2][FM], wf[2][FN];
  constexpr bool XL = FM >= FN;
  auto read = [&](int i, int ks, int sa, int sw) __attribute__((always_inline)) {   // x 0, all of W, the rest of x; where W is the larger: W 0, all of x, the rest of W
    if (XL ? i == 0 || i > FN : i >= 1 && i <= FM) {
      const int j = XL ? (i == 0 ? 0 : i - FN) : i - 1;
      af[ks][j] = *reinterpret_cast<const bf16x8_t*>(ap + sa * ASZ + j * 2048 + (fa ^ (64 * ks)));
    } else {
      const int j = XL ? i - 1 : (i == 0 ? 0 : i - FM);
      wf[ks][j] = *reinterpret_cast<const bf16x8_t*>(wp + sw * WSZ + (j >> 1) * 4096 + (j & 1) * 512 + (fw ^ (64 * ks)));
    }
  };
  int sa, sw;          // slots of the K tile at hand

  // ---- results
  TileAt old;          // the tile whose results are in the accumulators
  constexpr int NB = (16 * FN + 63) / 64;   // lane l holds the biases of the wave's columns l, l + 64: 16 lanes need the same eight
  float bias[NB], b[8];
  const bool biased = !PAIR && a.bias && !a.part;
#pragma unroll
  for (int i = 0; i < NB; ++i) bias[i] = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) b[e] = 0.f;
  auto biases = [&]() __attribute__((always_inline)) {
    if (!biased) return;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int col = min(cur.n0 + wn * 16 * FN + 64 * i + lane, a.N - 1);
      bias[i] = a.bias_f32 ? ((const float*)a.bias)[col] : ldf((const bf16*)a.bias + col);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) bias[i] = __int_as_float(tile_opaque(__float_as_int(bias[i])));   // (they are waited for here)
  };
  auto biases_of = [&](int j) __attribute__((always_inline)) {
    if (!biased) return;
    const int from = tile_opaque(32 * g4) + 4 * (32 * j & 63);
#pragma unroll
    for (int e = 0; e < 8; ++e) b[e] = __int_as_float(__builtin_amdgcn_ds_bpermute(from + 4 * e, __float_as_int(bias[32 * j / 64])));
  };
  TileOut<PAIR> out;

  // one step: the products of K half KS, and between them the other half's reads and the next loads, one at a time. MODE: loads go out;
  // none are left; the first step of a tile, which takes the last one's results out of the accumulators it starts
  enum { kRun, kLast, kStart, kJoin };
  auto step = [&](auto ks_c, auto mode_c, auto act_c, int ra, int rw, bool load) __attribute__((always_inline)) {
    constexpr int KS = decltype(ks_c)::value, MODE = decltype(mode_c)::value;
    constexpr int DN = KS ? FM : FN, DD = FM * FN / DN;
    const char* src = KS ? xb + kx : wb + kw;
    const uint32_t at = KS ? lds_a + sa * ASZ : lds_w + (sw == 0 ? RW - 1 : sw - 1) * WSZ;
    f32x4_t lo, hi;
    if constexpr (MODE == kJoin) {
      const int row = old.m0 + wm * 16 * FM;
      out.start(a, old.s, row, min(old.hi - row, 16 * FM), PAIR ? old.n0 / 2 + wn * 8 * FN : old.n0 + wn * 16 * FN, l16, g4);
    }
    tile_each<FM * FN>([&](auto q_c) __attribute__((always_inline)) {
      constexpr int q = decltype(q_c)::value, IN = XL ? FN : FM;
      constexpr int o = q / IN, i = o & 1 ? IN - 1 - q % IN : q % IN;   // there and back: the operand at the turn stays
      constexpr int m = MODE >= kStart ? q / 2 % FM : XL ? o : i, n = MODE >= kStart ? q / (2 * FM) * 2 + q % 2 : XL ? i : o;
      constexpr int d = tile_load_at(q, DN, DD, RS);
      const uint32_t off = KS ? ao[d >= 0 && d < FM ? d : 0] : wo[d >= 0 && d < FN ? d : 0];
      if constexpr (MODE >= kStart) {
        if (MODE == kJoin && q % (2 * FM) == 0) {
          out.columns(n / 2, PAIR ? old.n0 / 2 + wn * 8 * FN + 8 * n : old.n0 + wn * 16 * FN + 16 * n);
          if (!PAIR) biases_of(n / 2);
        }
        if (MODE == kJoin && q % 2 == 0) lo = TileAcc<m * FN + (n & ~1)>::take(), hi = TileAcc<m * FN + (n | 1)>::take();
        TileAcc<m * FN + n>::first(wf[KS][n], af[KS][m]);
        if (d >= 0 && load) tile_dma(src, off, at + d * 1024);
        if (MODE == kJoin && q % 2 == 1) out.template put<decltype(act_c)::value>(a, m, lo, hi, b);
      } else if constexpr (MODE == kRun && d >= 0) {
        TileAcc<m * FN + n>::mul_dma(wf[KS][n], af[KS][m], src, off, at + d * 1024);
      } else {
        TileAcc<m * FN + n>::mul(wf[KS][n], af[KS][m]);
      }
      if (q % RS == 0 && q / RS < LD) read(q / RS, KS ^ 1, ra, rw);
      if (MODE != kLast && q == FM * FN - 2) KS ? next(kx) : next(kw);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  constexpr auto k0 = std::integral_constant<int, 0>{};
  constexpr auto k1 = std::integral_constant<int, 1>{};
  constexpr auto run = std::integral_constant<int, kRun>{};
  constexpr auto last = std::integral_constant<int, kLast>{};
  constexpr auto start = std::integral_constant<int, kStart>{};
  constexpr auto join = std::integral_constant<int, kJoin>{};

  // ---- the tiles. The loads are RA tiles of K ahead and go over to the next tile of the result where this one has as many to go, so
  // that it starts at once; its first step stores this one's results. (SHORT: one tile, K of up to RA tiles, all of it loaded first.)
  place();
#pragma unroll
  for (int t = -RW; t < 0; ++t) {
    if (t + RA >= 0 && (!SHORT || t + RA < ld.nk)) {
#pragma unroll
      for (int i = 0; i < FM; ++i) tile_dma(xb + kx, ao[i], lds_a + (t + RA) * ASZ + i * 1024);
      next(kx);
    }
    if (SHORT ? t + RW < ld.nk : t < -1) {
#pragma unroll
      for (int i = 0; i < FN; ++i) tile_dma(wb + kw, wo[i], lds_w + (t + RW) * WSZ + i * 1024);
      next(kw);
    }
  }
  done += gridDim.x;
  cur = old = ld;
  old.hi = 0;          // (no results yet)
  xgk::wait_vmcnt<SHORT ? 0 : CNT0 < 63 ? CNT0 : 63>();
  xgk::raw_barrier();
  sa = sw = 0;
#pragma unroll
  for (int i = 0; i < LD; ++i) read(i, 0, 0, 0);
  // half way through K tile t: its slots are read; tile t + 1 has landed, in every wave
  auto half_way = [&](bool stores) __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (stores) xgk::wait_vmcnt<(CNT + ST < 63 ? CNT + ST : 63)>();
    else xgk::wait_vmcnt<CNT>();
    xgk::raw_barrier();
  };
  auto first_half = [&](auto mode_c, bool load) __attribute__((always_inline)) { step(k0, mode_c, k0, sa, sw, load); };
  auto second_half = [&](auto mode_c) __attribute__((always_inline)) {
    const int na = sa + 1 == RA ? 0 : sa + 1, nw = sw + 1 == RW ? 0 : sw + 1;
    step(k1, mode_c, k0, na, nw, true);
    sa = na, sw = nw;
  };
  constexpr bool AHEAD = RW > RA;   // w's loads are half a K tile ahead of x's, else behind
  for (bool end = SHORT;;) {
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // the last products' results
    if (old.hi == 0) {
      first_half(start, !SHORT);
    } else if (a.part) {
      step(k0, join, std::integral_constant<int, kTilePart>{}, sa, sw, !end);
    } else {
      tile_by_act<PAIR>(a, [&](auto act_c) __attribute__((always_inline)) { step(k0, join, act_c, sa, sw, !end); });
    }
    int t = 0;         // the K tile at hand
    if (!end) {
      const int stop = cur.nk - (AHEAD ? 0 : 1);
      if (AHEAD) half_way(old.hi != 0), second_half(run), t = 1;
      for (int lim = cur.nk - RA;;) {
        for (; t < lim; ++t) {
          if (AHEAD) first_half(run, true);
          half_way(TB > (AHEAD ? 1 : 0) && old.hi != 0 && t < TB);
          second_half(run);
          if (!AHEAD) first_half(run, true);
        }
        if (lim == stop) break;
        biases();
        end = done + (int)blockIdx.x >= total;
        if (end) break;
        place();
        done += gridDim.x, lim = stop;
      }
      if (!end) {
        if (!AHEAD) half_way(false), second_half(run);
        old = cur, cur = ld;
        continue;
      }
      if (AHEAD) first_half(last, false);
    } else if (SHORT && old.hi == 0) {
      biases();
    } else {
      break;
    }
    for (;;) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      const int rest = cur.nk - 2 - t;   // K tiles behind the one that has to be there
      if (RA > 5 && rest >= 4) xgk::wait_vmcnt<(4 * LD < 63 ? 4 * LD : 63)>();
      else if (RA > 4 && rest == 3) xgk::wait_vmcnt<(3 * LD < 63 ? 3 * LD : 63)>();
      else if (RA > 3 && rest == 2) xgk::wait_vmcnt<2 * LD>();
      else if (RA > 2 && rest == 1) xgk::wait_vmcnt<LD>();
      else xgk::wait_vmcnt<0>();
      xgk::raw_barrier();
      second_half(last);
      if (++t == cur.nk) break;
      first_half(last, false);
    }
    old = cur;
  }
}

template <bool PAIR, int FM, int FN, int RA, int RW, int OCC, bool SHORT = false>
static void tile_launch(const TileArgs& a, int cus, hipStream_t st) {
  const int tiles = ((a.M + 32 * FM - 1) / (32 * FM)) * ((a.N + 32 * FN - 1) / (32 * FN));
  const int grid = SHORT || tiles * a.S < cus * OCC ? tiles * a.S : cus * OCC;
  tile_linear_kernel<FM, FN, RA, RW, OCC, PAIR, false, SHORT><<<grid, 256, 0, st>>>(a);
}

// K (a part of it) of up to RA tiles: the ring of this size does not turn. From three tiles on a ring of two does, on the nearest of three
// sizes, the smaller ones in two workgroups a CU; one or two are loaded whole, by a workgroup for every tile of the result and two a CU, so
// that one's stores run beside the other's loads. (Parts of two and of three tiles: the same with three slots.) Beyond kRotateRows rows all
// sizes give the same bits, as all sum K in the same order. Up to there a column begins where the number of its tile says, of the size that
// was asked for: what runs in its place has columns that fill that one's without a rest. us, rings that end with the tile / now (in brackets all of K loaded first, a workgroup a CU): 2521 x 2048 x 64
// 8.1 / 7.3 (9.2), 8192 x 8192 x 128 64 / 51 (79) and gated 48 / 43 (68), 8192 x 8192 x 192 78 / 61 (92), 2521 x 2048 x 256 9.8 / 9.1 (13.4), 300 x
// 16384 x 256 9.9 / 9.3 (13.4), 300 x 2048 x 192 5.0 / 4.8 (5.9); 32 experts of 128 x 2048, four each, 6000 tokens 170 / 177 (217).
template <bool PAIR>
static void tile_launch_short(const TileArgs& a, int fm, int fn, int least, int most, int cus, hipStream_t st) {
  const int area = fm * fn;
  const bool narrow = area <= 12 || (a.rotate && fn % 4);
  if (least > 2) {
    if (narrow) tile_launch<PAIR, 3, 2, 2, 3, 2>(a, cus, st);
    else if (area <= 28 || (a.rotate && fn == 4)) tile_launch<PAIR, 4, 4, 2, 3, 2>(a, cus, st);
    else tile_launch<PAIR, 5, 8, 2, 3, 1>(a, cus, st);
  } else if (most > 2) {
    if (narrow) tile_launch<PAIR, 3, 2, 3, 3, 2, true>(a, cus, st);
    else tile_launch<PAIR, 4, 4, 3, 3, 1, true>(a, cus, st);
  } else if (narrow) {
    tile_launch<PAIR, 3, 2, 2, 2, 2, true>(a, cus, st);
  } else {
    tile_launch<PAIR, 4, 4, 2, 2, 2, true>(a, cus, st);
  }
}

// the launch of one size (-1: there is none); gated products are compiled in tile_gated.hip
// (a round of workgroups costs the same full or nearly empty: sizes between the powers of two are there for the row counts that
// leave such a round; 160 x 192 and 128 x 192 were the fastest too rarely, by 1 to 6 %)
// (96 x 64 with rings of four, which two workgroups of a CU just have: w is asked for one step behind x, so that in rings of three it
// comes late. us, rings that end with the tile and ask for both at once / of three / of four: 400 x 2048 x 2048 12.1 / 12.6 / 11.5, 298 x
// 4096 x 4096 28.4 / 29.0 / 24.8, 65 x 16384 x 2048 20.2 / 20.2 / 17.7, in four parts 130 x 2048 x 2048 10.1 / 10.5 / 10.5. Four tiles of K, which
// a ring of four would not turn for, have three slots for x: 93 x 1088 x 2048 in eight parts 11.5 / 9.2)
template <bool PAIR>
static int tile_launch_size(const TileArgs& a, int fm, int fn, int cus, hipStream_t st) {
  const int nk = a.K / 64, least = nk / a.S, most = (nk + a.S - 1) / a.S;
  if (fm == 3 && fn == 2 && least == 4) {
    tile_launch<PAIR, 3, 2, 3, 4, 2>(a, cus, st);
    return 0;
  }
#define XGM_TILE(FM, FN, RA, RW, OCC)                                                   \
  if (fm == FM && fn == FN) {                                                           \
    if (least > RA) tile_launch<PAIR, FM, FN, RA, RW, OCC>(a, cus, st);                 \
    else tile_launch_short<PAIR>(a, FM, FN, least, most, cus, st);                      \
    return 0;                                                                           \
  }
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
  XGM_TILE(3, 2, 4, 4, 2)
#undef XGM_TILE
  return -1;
}
int tile_launch_gated(const TileArgs& a, int fm, int fn, int cus, hipStream_t st);   // tile_gated.hip
}  // namespace xgm
