// State-space recurrence over prompt portions of bf16 rows, in chunks of 64 tokens on the bf16 matrix cores, state fp32:
//
//   S_t = e^(-rate dt_t) S_(t-1) + dt_t B_t x_t^T,   o_t = S_t^T C_t + D x_t
//
// B, C and x are bf16, so a product of any of them with an fp32 number is exact to fp32 where that number goes in as three bf16
// (8 bits of its mantissa each): three instructions of 16x16x32 in the place of eight of fp32 16x16x4 that take twice the time each.
// Per chunk and 16 state columns (a wave; four waves share a workgroup of 64 columns)
//   o = pre (C S) + G x,        G_tj = C_t . B_j dt_j (decay behind j up to t) (+ D on the diagonal),   j <= t
//   S <- E S + B^T (post x)
// with pre the decay from the chunk's start through t, post dt times the decay behind a token to its end. Decays stay products
// carried in two floats (Prod), formed inside sub-chunks of 16 tokens and put together from their whole products, so nothing but a
// sub-chunk's own reciprocals (above 2^-90) is ever above 1. G is formed once per workgroup, three of its twelve 16 x 16 tiles a wave,
// split, and handed on through LDS in the order of the lanes. State row 32 i + 8 g + 4 k + r is register r of lane group g in tile
// 2 i + k, so that two tiles' registers are the B operand of C S as they lie; B^T and x come from LDS by transposed reads.
// A chunk with an input out of range (2^28 and above, infinities, NaN) or a sub-chunk below 2^-90 runs token by token, and so does a
// wave whose state is too large for C S, which meets the decays only after its sum: above 2^92 it could leave fp32 (128 terms, C below
// 2^28), above 2^40 what it leaves behind decays that underflow within the chunk could count.
// Chunks of up to four tokens (single tokens beside a prompt, remainders) run token by token for speed: 60 x 1 + 16 tokens of 64 heads 90 ->
// 63 us, 60 x 1 + 512 102 -> 76, 40 sequences of 2 / 3 / 4 tokens beside 100 70.5 -> 57 / 61 / 64, of 6 70 either way.
//
// Error against fp64 (2-norm, outputs / carried state; chunks of 16 tokens in fp32 in brackets, then the token loop), 400 tokens of 8
// heads of 128 x 64, A_log about 0 8.4e-8 / 6.3e-8 (8.8e-8 / 5.8e-8; 8.7e-8 / 6.2e-8), -0.5 8.4e-8 / 6.6e-8 (9.2e-8 / 6.9e-8; 8.8e-8 /
// 6.9e-8), -2 9.6e-8 / 9.4e-8 (1.18e-7 / 1.25e-7; 1.0e-7 / 1.24e-7), -4 3.6e-7 / 4.8e-7 (3.7e-7 / 5.1e-7; 3.6e-7 / 5.2e-7). That takes the
// parts below the first summed up by themselves, the chunk's terms added to E S as one sum, dt itself on G's diagonal, and the
// leading bits of post x (top4).
//
// Long portions of few sequences run in segments side by side: a first launch sums every segment but the last up from a zero state, the
// second puts its state together from those in front of it and runs with outputs. Segment z of a sequence of more than one has slot
// 2 (q0 / seg) + z, which no other has: the next such sequence begins floor(q / seg) >= 1 segments on at least, and ceil(q / seg) is at
// most twice that. Token (slot / 2 + 1) seg - 1 is one of the sequence's (z seg of its q tokens are in front of segment z), so a
// workgroup of a slot finds its sequence. The incoming state, which the last segment's workgroup replaces, is set aside in the place
// of that segment's sum, which nobody reads. Sequences of one segment (single tokens beside a prompt) have no part in the first
// launch and their states are read in place. (With a workgroup per sequence and possible segment, and every sequence's state set aside,
// 200 single tokens beside 256 of 64 heads took 448 us and 0.9 GB of scratch, now 208 and 34 MB.)
//
// Measured, heads of 128 x 64: 2521 ragged tokens of 64 heads 199 -> 78 us (81 traced in a step), 4 x 1024 of 128 276 -> 122, 4001 of
// 64 102. A chunk of one workgroup is 5 us by itself, 3.9 where two share a unit: 1.9 of vector work (splitting, scales, range checks:
// 1100 instructions a wave), 0.95 of matrix instructions, 1.2 of LDS reads, the rest waits between its three barriers. A token by itself
// is 200 vector instructions and one LDS latency (its eight reads go out at once; one behind the other 64 heads, 4001 such tokens 631 ->
// 605, 8 heads, 257 75 -> 73). No register of a lane is spilled; some 40 scalars that the loop does not hold are lane reads, 2 % of a
// chunk's instructions.
#include "mfma_f32.h"

namespace xgm {

using xgk::as_frag;
using xgk::ld16;
using xgk::mfma16x16x32;

constexpr int kSsTok = 64, kSsRing = 8;   // tokens per chunk; chunks whose step sizes are held
constexpr int kSsFew = 4;                                    // tokens of a chunk that run one by one
constexpr float kSsMinProd = 8.077935669463161e-28f;   // 2^-90
constexpr float kSsMinChunk = 7.888609052210118e-31f, kSsMaxState = 4.951760157141521e27f, kSsMaxFaded = 1099511627776.f;   // 2^-100, 2^92, 2^40

struct SsmChunkArgs {
  const bf16* rows;            // [x (H P) | B (G N) | C (G N)]
  int64_t ld;
  const bf16* dt;
  int64_t ld_dt;
  const float *dt_bias, *A_log, *skip;
  float* state;                // [slots, H, N, P]
  const int32_t *qsl, *seq_lens, *slots;
  float* o;                    // [T, H P]
  int ns, H, G, P, pass, seg, slots_seg;   // slots_seg: slots of segments, in front of the sequences in the grid (0 in one pass)
  float *decay, *sums;         // per (segment, head): its whole decay; its sum in the order of the lanes (S of a zero state; incoming S)
};

// granule (16 bytes) of a staged row: rows of 256 bytes and of 128; reads of 16 rows and transposed reads of 4 x 4 granules
// touch every bank once
__device__ __forceinline__ int ss_swz16(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }
__device__ __forceinline__ int ss_swz8(int r) { return (((r >> 1) & 1) << 2) | ((r >> 2) & 3); }

// x = h + m + l, 8 bits of its mantissa each: three bf16 (pairs in one register, the first element low)
__device__ __forceinline__ uint32_t hi_pair(float a, float b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
#else
  return 0;
#endif
}
__device__ __forceinline__ float top8(float x) { return __uint_as_float(__float_as_uint(x) & 0xFFFF0000u); }
__device__ __forceinline__ void split3(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = hi_pair(a, b);
  a -= top8(a), b -= top8(b);
  m = hi_pair(a, b);
  a -= top8(a), b -= top8(b);
  l = hi_pair(a, b);
}
// ... in front of them the four leading bits. A matrix instruction adds eight products at a time and cuts what lies 24 bits below
// the largest: with 8 + 8 bits that begins at terms of 1/256 of it, with 4 + 8 at 1/4096 (carried state, A_log about -0.5: 1.16 times
// the error of fp32 instructions and 0.97).
__device__ __forceinline__ float top4(float x) { return __uint_as_float(__float_as_uint(x) & 0xFFF00000u); }
struct Split8 {   // eight floats as the three operands of a product
  uint32_t p[3][4];
  __device__ __forceinline__ void set(int i, float a, float b) { split3(a, b, p[0][i], p[1][i], p[2][i]); }
  __device__ __forceinline__ xgk::bf16x8_t frag(int s) const { return as_frag(make_uint4(p[s][0], p[s][1], p[s][2], p[s][3])); }
};

__device__ __forceinline__ void ss_fence() {   // (bounds what the scheduler hoists: registers)
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_sched_barrier(0);
#endif
}

// the largest magnitudes seen, as pairs of 16 bits (they order as their bits do, NaN above them all)
__device__ __forceinline__ void see(uint4 v, uint32_t& seen) {
  using u16x2 = __attribute__((ext_vector_type(2))) uint16_t;
  const u16x2 m = __builtin_elementwise_max(
      __builtin_elementwise_max(__builtin_bit_cast(u16x2, v.x & 0x7FFF7FFFu), __builtin_bit_cast(u16x2, v.y & 0x7FFF7FFFu)),
      __builtin_elementwise_max(__builtin_bit_cast(u16x2, v.z & 0x7FFF7FFFu), __builtin_bit_cast(u16x2, v.w & 0x7FFF7FFFu)));
  seen = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, seen), m));
}

// lanes of a row of 16: from lane + O (1 past the end), from lane - O, and lane L's value for all
template <int CTRL>
__device__ __forceinline__ float row_move(float x, float other) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __uint_as_float(__builtin_amdgcn_update_dpp(__float_as_uint(other), __float_as_uint(x), CTRL, 0xF, 0xF, false));
#else
  return x;
#endif
}
template <int O> __device__ __forceinline__ Prod prod_down(Prod p) { return {row_move<0x100 + O>(p.h, 1.f), row_move<0x100 + O>(p.l, 0.f)}; }
template <int O> __device__ __forceinline__ Prod prod_up(Prod p) { return {row_move<0x110 + O>(p.h, 1.f), row_move<0x110 + O>(p.l, 0.f)}; }
__device__ __forceinline__ float lane_value(float x, int lane) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), lane));
#else
  return x;
#endif
}
__device__ __forceinline__ Prod prod_at(Prod p, int lane) { return {lane_value(p.h, lane), lane_value(p.l, lane)}; }
template <int O> __device__ __forceinline__ void prod_scan(Prod& suf, Prod& pfx) {
  suf = prod_mul(suf, prod_down<O>(suf));   // (past the row's ends: times 1)
  pfx = prod_mul(pfx, prod_up<O>(pfx));
}

template <int N, bool SUMS>
__global__ __launch_bounds__(256, 2) void ssm_chunk_kernel(const SsmChunkArgs a) {
  constexpr int C = kSsTok, MT = N / 16, KS = N / 32, GR = N / 8, RB = 2 * N;   // state tiles, steps along N, granules, bytes of a row
  constexpr int UN = C * GR / 256, UX = C * 8 / 256;                            // 16-byte units per thread: B (and C), x
  static_assert(N == 128 || N == 64, "ssm_chunk geometry");
  __shared__ __attribute__((aligned(16))) char cs[C * RB], bs[C * RB], xs[C * 128];
  __shared__ __attribute__((aligned(16))) uint4 gs[6 * 3 * 64];   // G of (block of 16 tokens, 32 tokens before): [pair][part][lane]
  __shared__ __attribute__((aligned(16))) float pre[kSsRing][C], post[kSsRing][C], ds[kSsRing][C], dts[kSsRing][C], ft[kSsRing][4][C];
  __shared__ float Eh[kSsRing], El[kSsRing];
  __shared__ int bad_step[kSsRing], flags[2][4];

  const int hx = blockIdx.x;
  int s = (int)blockIdx.y - a.slots_seg, z = 0;
  if (s < 0) {   // the sequence of the slot's token
    const int tok = (blockIdx.y / 2 + 1) * a.seg - 1, l = threadIdx.x & 63;
    s = 0;
    for (int i = 0; i < a.ns; i += 64) s += __popcll(__ballot(i + l < a.ns && a.qsl[min(i + l, a.ns - 1) + 1] <= tok));
    if (s >= a.ns) return;
    z = blockIdx.y - 2 * (a.qsl[s] / a.seg);
  }
  const int h = a.H % 8 == 0 ? (hx % 8) * (a.H / 8) + hx / 8 : hx;   // (an XCD takes neighbouring heads, which share B and C)
  const int q0 = a.qsl[s], qn = a.qsl[s + 1] - q0, slot = a.slots[s];
  const int c0 = z * a.seg, c1 = min(qn, c0 + a.seg), pass = SUMS ? 1 : a.pass;
  if (slot < 0 || c0 < 0 || c0 >= qn) return;
  const bool last_seg = c1 == qn, whole = qn <= a.seg;
  if (a.slots_seg && whole == ((int)blockIdx.y < a.slots_seg)) return;   // (a slot's token of a sequence of one segment, and the other way round)
  if (SUMS && last_seg) return;   // nobody reads its sum
  const int ctx = a.seq_lens[s] - qn;
  const int tid = threadIdx.x, lane = tid & 63, g4 = lane >> 4, l16 = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col0 = blockIdx.z * 64 + 16 * w, col = col0 + l16;
  const bool on = col0 < a.P;   // (P is a multiple of 16)
  // element (m, r) of a lane: state row 32 (m / 2) + 8 g4 + 4 (m % 2) + r, so that two tiles' registers are eight rows in a row
  float* Sg = a.state + ((int64_t)slot * a.H + h) * (int64_t)N * a.P + (int64_t)(8 * g4) * a.P + min(col, a.P - 1);
  const int64_t lane_tile = (int64_t)gridDim.z * 4 * MT * 64;   // float4s of a state in lane order
  const int64_t mine = ((int64_t)blockIdx.z * 4 + w) * MT * 64 + lane;
  const int64_t cs0 = 2 * (q0 / a.seg);
  float4* sums = reinterpret_cast<float4*>(a.sums) + (cs0 * a.H + h) * lane_tile + mine;
  const int64_t seg_step = (int64_t)a.H * lane_tile;
  float4* s_in = sums + (qn - 1) / a.seg * seg_step;

  f32x4_t S[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) S[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto row_at = [&](int m, int r) { return (int64_t)(32 * (m >> 1) + 4 * (m & 1) + r) * a.P; };
  if (SUMS || pass != 2 || whole) {
    if (on && ctx > 0 && z == 0)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[m][r] = Sg[row_at(m, r)];
    if (SUMS && z == 0)   // segments are summed up from zero; the incoming state is set aside
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        s_in[64 * m] = make_float4(S[m][0], S[m][1], S[m][2], S[m][3]);
        S[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
  } else {   // the state in front of this segment: what came in, and the sums of the segments before
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const float4 v = s_in[64 * m];
      S[m] = f32x4_t{v.x, v.y, v.z, v.w};
    }
    for (int y = 0; y < z; ++y) {
      const float f = a.decay[(cs0 + y) * a.H + h];
      float4 b[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) b[m] = sums[y * seg_step + 64 * m];
#pragma unroll
      for (int m = 0; m < MT; ++m) {   // (a product past fp32 of finite growths leaves a zero zero)
        S[m][0] = S[m][0] == 0.f ? b[m].x : fmaf(f, S[m][0], b[m].x), S[m][1] = S[m][1] == 0.f ? b[m].y : fmaf(f, S[m][1], b[m].y);
        S[m][2] = S[m][2] == 0.f ? b[m].z : fmaf(f, S[m][2], b[m].z), S[m][3] = S[m][3] == 0.f ? b[m].w : fmaf(f, S[m][3], b[m].w);
      }
    }
  }

  // ---- a chunk's rows into registers (rows past the end repeat the last: their step sizes are 0)
  const bf16* xg = a.rows + (int64_t)h * a.P + blockIdx.z * 64;
  const bf16* bg = a.rows + (int64_t)a.H * a.P + (h / (a.H / a.G)) * N;
  const int xlim = min(64, a.P - (int)blockIdx.z * 64);
  uint4 ub[UN], uc[UN], ux[UX];
  auto fetch = [&](int t0) {   // (uniform bases, 32-bit lane offsets)
    const int left = c1 - t0 - 1;
    const int64_t row0 = (int64_t)(q0 + t0) * a.ld;
    const bf16 *bp = bg + row0, *cp = bp + a.G * N, *xp = xg + row0;
    const uint32_t ld = (uint32_t)a.ld, b0 = tid / GR * ld + 8 * (tid % GR), x0 = tid / 8 * ld + min(8 * (tid % 8), xlim - 8);
    if (left >= C - 1) {
#pragma unroll
      for (int j = 0; j < UN; ++j) {
        ub[j] = ld16(bp + (256 / GR * j) * a.ld + b0);
        if (!SUMS) uc[j] = ld16(cp + (256 / GR * j) * a.ld + b0);
      }
#pragma unroll
      for (int j = 0; j < UX; ++j) ux[j] = ld16(xp + 32 * j * a.ld + x0);
      return;
    }
#pragma unroll
    for (int j = 0; j < UN; ++j) {
      const uint32_t at = (uint32_t)min(tid / GR + 256 / GR * j, left) * ld + 8 * (tid % GR);
      ub[j] = ld16(bp + at);
      if (!SUMS) uc[j] = ld16(cp + at);
    }
#pragma unroll
    for (int j = 0; j < UX; ++j) ux[j] = ld16(xp + ((uint32_t)min(tid / 8 + 32 * j, left) * ld + min(8 * (tid % 8), xlim - 8)));
  };
  auto stage = [&](int ci) {
    uint32_t seen = 0;
#pragma unroll
    for (int j = 0; j < UN; ++j) {
      const int u = tid + 256 * j, tok = u / GR, g = u % GR;
      const int at = tok * RB + 16 * (g ^ (GR == 16 ? ss_swz16(tok) : ss_swz8(tok)));
      see(ub[j], seen);
      *reinterpret_cast<uint4*>(bs + at) = ub[j];
      if (!SUMS) {
        see(uc[j], seen);
        *reinterpret_cast<uint4*>(cs + at) = uc[j];
      }
    }
#pragma unroll
    for (int j = 0; j < UX; ++j) {
      const int u = tid + 256 * j, tok = u / 8;
      see(ux[j], seen);
      *reinterpret_cast<uint4*>(xs + tok * 128 + 16 * ((u % 8) ^ ss_swz8(tok))) = ux[j];
    }
    const int any = __any(max(seen & 0xFFFFu, seen >> 16) >= (__float_as_uint(kChunkMaxIn) >> 16));
    if (lane == 0) flags[ci & 1][w] = any;
  };
  // ---- step sizes and decays of the four chunks from `ci` on, one a wave, a token a lane
  const float rate = expf(a.A_log[h]), dtb = a.dt_bias[h];
  bf16 dt_raw = 0;   // of the chunk that this wave's next call forms
  auto dt_load = [&](int ci) {
    const int t0 = c0 + C * (ci + w);
    if (t0 < c1) dt_raw = a.dt[(int64_t)(q0 + min(t0 + lane, c1 - 1)) * a.ld_dt + h];
  };
  auto steps = [&](int ci) {
    const int cc = ci + w, t0 = c0 + C * cc, left = c1 - t0;
    if (left <= 0) return;
    const float d = lane < left ? softplusf(bf2f(dt_raw) + dtb) : 0.f;
    const float dec = out_of_range(d) ? __builtin_nanf("") : expf(-rate * d);
    Prod suf = {dec, 0.f}, pfx = suf;   // from this token to the sub-chunk's end, from its start to this token
    prod_scan<1>(suf, pfx), prod_scan<2>(suf, pfx), prod_scan<4>(suf, pfx), prod_scan<8>(suf, pfx);
    const Prod after = prod_down<1>(suf);
    const Prod E0 = prod_at(suf, 0), E1 = prod_at(suf, 16), E2 = prod_at(suf, 32), E3 = prod_at(suf, 48);
    const Prod E01 = prod_mul(E0, E1), E12 = prod_mul(E1, E2), E23 = prod_mul(E2, E3), one = {1.f, 0.f};
    const Prod ahead = g4 == 0 ? one : g4 == 1 ? E0 : g4 == 2 ? E01 : prod_mul(E01, E2);        // from the chunk's start
    const Prod behind = g4 == 3 ? one : g4 == 2 ? E3 : g4 == 1 ? E23 : prod_mul(E1, E23);       // to the chunk's end
    const int at = cc % kSsRing;
    pre[at][lane] = prod_times(prod_mul(ahead, pfx), 1.f);
    post[at][lane] = prod_times(prod_mul(after, behind), d);
    ds[at][lane] = prod_times(after, d);
    dts[at][lane] = d;
    // factor of G's row t for tokens of sub-chunk i: what lies between, or 1 / s inside its own
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Prod mid = g4 - i <= 1 ? one : g4 - i == 2 ? (i == 0 ? E1 : E2) : E12;
      ft[at][i][lane] = i > g4 ? 0.f : i == g4 ? prod_rcp(after) : prod_times(prod_mul(mid, pfx), 1.f);
    }
    const bool bad = !(suf.h >= kSsMinProd);   // (a whole sub-chunk's product bounds the others; NaN too)
    const int any = __any(bad);
    if (lane == 0) {
      const Prod E = prod_mul(E01, E23);
      Eh[at] = E.h, El[at] = E.l, bad_step[at] = any;
    }
  };
  const float skip = a.skip[h];
  float ptot = 1.f;   // decay of the segment
  // LDS addresses of a lane; what varies is xored into bits 6 and 7 (64 bytes of a row) or added as a constant
  const int z16 = GR == 16 ? (l16 & 3) << 2 : ((l16 >> 1) & 1) << 2;
  const int c_at = l16 * RB + 16 * (z16 | (g4 ^ (l16 >> 2)));   // row l16, granule g4
  int b_tr[2], x_tr[2];   // rows 8 g4 + 4 i + l16 / 4 of a transposed read, granules l16 % 4 and (this wave's) (l16 % 4) / 2
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 8 * g4 + 4 * i + (l16 >> 2), zr = (2 * g4 + i) & 3;
    b_tr[i] = r * RB + 16 * ((GR == 16 ? (l16 >> 2) << 2 : (l16 >> 3) << 2) | ((l16 & 3) ^ zr));
    x_tr[i] = r * 128 + 16 * ((2 * w + ((l16 & 3) >> 1)) ^ (((l16 >> 3) << 2) | zr)) + 8 * (l16 & 1);
  }
  const uint32_t o_at = (uint32_t)(4 * g4) * (uint32_t)(a.H * a.P) + l16;
  dt_load(0);
  fetch(c0);
  steps(0);
  f32x4_t acc[4];
  auto store = [&](int t0) {
    float* ob = a.o + ((int64_t)(q0 + t0) * a.H + h) * a.P + col0;
    if (c1 - t0 >= C) {
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) (ob + (int64_t)(16 * b + r) * (a.H * a.P))[o_at] = acc[b][r];
      return;
    }
    const int n = c1 - t0 - 4 * g4;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (16 * b + r < n) (ob + (int64_t)(16 * b + r) * (a.H * a.P))[o_at] = acc[b][r];
  };
  for (int t0 = c0, ci = 0; t0 < c1; t0 += C, ++ci) {
    const int n = min(C, c1 - t0), rg = ci % kSsRing;
    if (ci) __syncthreads();   // every wave is past the chunk before
    stage(ci);
    if (ci % 4 == 1) dt_load(ci + 3);
    if (ci % 4 == 2) steps(ci + 2);
    __syncthreads();
    const float most = Eh[rg] >= kSsMinChunk ? kSsMaxState : kSsMaxFaded;
    const int odd = flags[ci & 1][0] | flags[ci & 1][1] | flags[ci & 1][2] | flags[ci & 1][3] | bad_step[rg];
    const bool slow = (n <= kSsFew) | (__builtin_amdgcn_readfirstlane(odd) != 0);
    // (a NaN goes token by token too; a chunk's whole decay bounds all of its own)
    float top = 0.f;
#pragma unroll
    for (int m = 0; m < MT; ++m) top = fmaxf(fmaxf(fabsf(S[m][0]), fabsf(S[m][1])), fmaxf(top, fmaxf(fabsf(S[m][2]), fabsf(S[m][3]))));
    const bool wslow = slow | (__any(!(top < most)) != 0);
    if (!SUMS && !slow) {
      // G^T of three of the twelve tiles: rows j = 32 q + 8 (i / 4) + 4 half + i % 4, columns token 16 b + l16
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int tile = 3 * w + k, pair = tile >> 1, half = tile & 1;
        const int b = pair < 2 ? pair : 2 + ((pair - 2) >> 1), q = pair < 2 ? 0 : (pair - 2) & 1;
        const int jl = 8 * (l16 >> 2) + 4 * half + (l16 & 3), tr = 16 * b + l16;
        const int j_at = (32 * q + jl) * RB + 16 * ((GR == 16 ? (jl & 3) << 2 : ((jl >> 1) & 1) << 2) | (g4 ^ ((jl >> 2) & 3)));
        const int t_at = 16 * b * RB + c_at;
        f32x4_t g2[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};   // two chains: half as many roundings in a row
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          g2[ks & 1] = mfma16x16x32(as_frag(*reinterpret_cast<const uint4*>(bs + (j_at ^ (ks << 6)))),
                                    as_frag(*reinterpret_cast<const uint4*>(cs + (t_at ^ (ks << 6)))), g2[ks & 1]);
        const f32x4_t g = g2[0] + g2[1];
        const int j0 = 32 * q + 8 * g4 + 4 * half;   // this lane's four tokens j
        const float f = ft[rg][2 * q + (g4 >> 1)][tr];
        const float dt_t = dts[rg][tr];
        float d[4], v[4];
        ld4(&ds[rg][j0], d);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[r] = j0 + r <= tr ? g[r] * (j0 + r < tr ? d[r] * f : dt_t) : 0.f;
          if (j0 + r == tr) v[r] += skip;
        }
        uint2 p[3];
        split3(v[0], v[1], p[0].x, p[1].x, p[2].x);
        split3(v[2], v[3], p[0].y, p[1].y, p[2].y);
#pragma unroll
        for (int i = 0; i < 3; ++i) reinterpret_cast<uint2*>(gs + (pair * 3 + i) * 64 + lane)[half] = p[i];
        ss_fence();
      }
      if (!wslow) {   // C S of the four blocks of 16 tokens
        f32x4_t low[4];   // the parts below the first by themselves: the sums of the first have KS roundings
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[b] = low[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          Split8 sp;
          sp.set(0, S[2 * ks][0], S[2 * ks][1]), sp.set(1, S[2 * ks][2], S[2 * ks][3]);
          sp.set(2, S[2 * ks + 1][0], S[2 * ks + 1][1]), sp.set(3, S[2 * ks + 1][2], S[2 * ks + 1][3]);
          xgk::bf16x8_t cf[4];
#pragma unroll
          for (int b = 0; b < 4; ++b) cf[b] = as_frag(*reinterpret_cast<const uint4*>(cs + (c_at ^ (ks << 6)) + 16 * b * RB));
#pragma unroll
          for (int b = 0; b < 4; ++b) low[b] = mfma16x16x32(cf[b], sp.frag(2), low[b]);
#pragma unroll
          for (int b = 0; b < 4; ++b) acc[b] = mfma16x16x32(cf[b], sp.frag(0), acc[b]);
#pragma unroll
          for (int b = 0; b < 4; ++b) low[b] = mfma16x16x32(cf[b], sp.frag(1), low[b]);
          ss_fence();
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          float p[4];
          ld4(&pre[rg][16 * b + 4 * g4], p);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[b][r] = (acc[b][r] + low[b][r]) * p[r];
        }
      }
    }
    __syncthreads();
    if (t0 + C < c1) fetch(t0 + C);   // (here: its registers are not wanted above)
    const Prod E = {Eh[rg], El[rg]};
    if (!wslow) {
      // x of tokens 32 q + 8 g4 + e, column l16: exact
      xgk::bf16x8_t xf[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        xgk::bf16x4_t v[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) v[i] = xgk::lds_read_tr16(reinterpret_cast<const uint16_t*>(xs + x_tr[i] + 32 * 128 * q));
        xf[q] = xgk::bf16x8_t{v[0][0], v[0][1], v[0][2], v[0][3], v[1][0], v[1][1], v[1][2], v[1][3]};
      }
      if (!SUMS) {   // the chunk's own terms
        f32x4_t low[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) low[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 2; i >= 0; --i)
#pragma unroll
          for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int b = 2 * q; b < 4; ++b) {
              const int pair = b < 2 ? b : 2 * b - 2 + q;
              const xgk::bf16x8_t g = as_frag(gs[(pair * 3 + i) * 64 + lane]);
              if (i) low[b] = mfma16x16x32(g, xf[q], low[b]);
              else acc[b] = mfma16x16x32(g, xf[q], acc[b]);
            }
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[b] += low[b];
        if (on) store(t0);
      }
      // S <- E S + B^T (post x)
      Split8 xp[2];
      uint32_t xt[2][4];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        float f[8], lo[4], hi[4];
        xgk::unpack8(__builtin_bit_cast(uint4, xf[q]), f);
        ld4(&post[rg][32 * q + 8 * g4], lo), ld4(&post[rg][32 * q + 8 * g4 + 4], hi);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float u = f[2 * i] * (i < 2 ? lo[2 * i] : hi[2 * i - 4]), v = f[2 * i + 1] * (i < 2 ? lo[2 * i + 1] : hi[2 * i - 3]);
          const float ut = top4(u), vt = top4(v);
          xt[q][i] = hi_pair(ut, vt);
          xp[q].set(i, u - ut, v - vt);
        }
      }
#pragma unroll
      for (int m0 = 0; m0 < MT; m0 += 2) {   // (the parts below the first by themselves: two roundings of the whole sum)
        xgk::bf16x8_t bf[2][2];
        f32x4_t add[2], low[2];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          add[m] = low[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            xgk::bf16x4_t v[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
              v[i] = xgk::lds_read_tr16(reinterpret_cast<const uint16_t*>(bs + (b_tr[i] ^ ((m0 >> 1) << 6)) + 32 * RB * q + 8 * m));
            bf[q][m] = xgk::bf16x8_t{v[0][0], v[0][1], v[0][2], v[0][3], v[1][0], v[1][1], v[1][2], v[1][3]};
          }
        }
#pragma unroll
        for (int i = 2; i >= 0; --i)
#pragma unroll
          for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int m = 0; m < 2; ++m) low[m] = mfma16x16x32(bf[q][m], xp[q].frag(i), low[m]);
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int m = 0; m < 2; ++m)
            add[m] = mfma16x16x32(bf[q][m], as_frag(make_uint4(xt[q][0], xt[q][1], xt[q][2], xt[q][3])), add[m]);
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r) S[m0 + m][r] = fmaf(E.h, S[m0 + m][r], fmaf(E.l, S[m0 + m][r], low[m][r]) + add[m][r]);
        if (m0 % 4) ss_fence();
      }
    } else {
      for (int t = 0; t < n; ++t) {
        const float dec = expf(-rate * dts[rg][t]);
        const int c = 2 * w + (l16 >> 3);
        const float vv = bf2f(*reinterpret_cast<const bf16*>(xs + t * 128 + 16 * (c ^ ss_swz8(t)) + 2 * (l16 & 7))), vd = vv * dts[rg][t];
        float part[4] = {0.f, 0.f, 0.f, 0.f};
        uint4 bu[KS], cu[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int at = t * RB + 16 * ((4 * ks + g4) ^ (GR == 16 ? ss_swz16(t) : ss_swz8(t)));
          bu[ks] = *reinterpret_cast<const uint4*>(bs + at);
          if (!SUMS) cu[ks] = *reinterpret_cast<const uint4*>(cs + at);
        }
        ss_fence();   // (all of a token's reads under way at once)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          float bb[8], cc[8];
          xgk::unpack8(bu[ks], bb);
          if (!SUMS) xgk::unpack8(cu[ks], cc);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            float& v = reinterpret_cast<float(&)[4]>(S[2 * ks + (e >> 2)])[e & 3];
            v = fmaf(dec, v, bb[e] * vd);
            if (!SUMS) part[e & 3] = fmaf(v, cc[e], part[e & 3]);
          }
        }
        if (!SUMS) {
          float sum = (part[0] + part[1]) + (part[2] + part[3]);
          sum += __shfl_xor(sum, 16, 64);
          sum += __shfl_xor(sum, 32, 64);
          if (on && g4 == 0) a.o[((int64_t)(q0 + t0 + t) * a.H + h) * a.P + col] = fmaf(skip, vv, sum);
        }
      }
    }
    if (SUMS) {
      if (!slow) {
        ptot = prod_times(E, ptot);
      } else {
        for (int t = 0; t < n; ++t) ptot *= expf(-rate * dts[rg][t]);
      }
    }
  }
  // ---- outgoing state, or the segment's sum
  if (SUMS) {
#pragma unroll
    for (int m = 0; m < MT; ++m) sums[z * seg_step + 64 * m] = make_float4(S[m][0], S[m][1], S[m][2], S[m][3]);
    if (tid == 0 && blockIdx.z == 0) a.decay[(cs0 + z) * a.H + h] = ptot;
  } else if (on && last_seg) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) Sg[row_at(m, r)] = S[m][r];
  }
}

// ================================================================== host launchers
// floats: per segment and head its decay and sum (columns in blocks of 64)
static int64_t ssm_chunk_slots(int T_, int seg) { return 2 * (int64_t)(T_ / seg) + 2; }
int64_t ssm_chunk_scratch_floats(int T_, int H, int N, int P, int seg) {
  const int64_t tile = (int64_t)N * ((P + 63) / 64 * 64), cslots = ssm_chunk_slots(T_, seg);
  return (cslots * H + 3) / 4 * 4 + cslots * H * tile;
}

int ssm_chunk(const void* xbc, int64_t ld_x, const void* dt_raw, int64_t ld_dt, const float* dt_bias, const float* A_log,
              const float* Dskip, float* state, const int32_t* qsl, const int32_t* seq_lens, const int32_t* slots, float* y, int ns,
              int max_q, int T_, int H, int G, int N, int P, int seg, float* scratch, hipStream_t st) {
  if (ns <= 0 || max_q <= 0) return 0;
  if (H < 1 || G < 1 || H % G || (N != 64 && N != 128) || P < 16 || P % 16 || (uintptr_t)xbc % 16 || ld_x % 8 || ld_x >= 1 << 25 || (H * P) % 8 ||
      (scratch && ((uintptr_t)scratch % 16 || seg < kSsTok || seg % kSsTok)))
    return -1;
  if (!scratch) seg = (max_q + kSsTok - 1) / kSsTok * kSsTok;
  SsmChunkArgs a = {};
  a.rows = (const bf16*)xbc, a.ld = ld_x, a.dt = (const bf16*)dt_raw, a.ld_dt = ld_dt, a.dt_bias = dt_bias, a.A_log = A_log;
  a.skip = Dskip, a.state = state, a.qsl = qsl, a.seq_lens = seq_lens, a.slots = slots, a.o = y, a.H = H, a.G = G, a.P = P;
  const bool two = max_q > seg;
  const int64_t n_slots = two ? ssm_chunk_slots(T_, seg) : 0;
  if ((two && !scratch) || ns + n_slots > 65535) return -1;
  a.ns = ns, a.seg = seg, a.slots_seg = (int)n_slots;
  if (scratch) a.decay = scratch, a.sums = scratch + (ssm_chunk_slots(T_, seg) * H + 3) / 4 * 4;
  for (int pass = two ? 1 : 0; pass < (two ? 3 : 1); ++pass) {
    const dim3 grid(H, n_slots + (pass == 1 ? 0 : ns), (P + 63) / 64);
    a.pass = pass;
    if (N == 128 && pass == 1) ssm_chunk_kernel<128, true><<<grid, 256, 0, st>>>(a);
    else if (N == 128) ssm_chunk_kernel<128, false><<<grid, 256, 0, st>>>(a);
    else if (pass == 1) ssm_chunk_kernel<64, true><<<grid, 256, 0, st>>>(a);
    else ssm_chunk_kernel<64, false><<<grid, 256, 0, st>>>(a);
  }
  return 0;
}

}  // namespace xgm
