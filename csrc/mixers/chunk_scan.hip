// Outer-product recurrences with an fp32 state over prompt portions, in chunks of 16 tokens on the fp32 matrix cores:
//
//   gates   S_t = diag(f_t) S_(t-1) + k_t v_t^T,             o_t = S_t^T q_t        (k_t = 1 - f_t when it is not given)
//   ssm     S_t = e^(-rate dt_t) S_(t-1) + dt_t B_t x_t^T,   o_t = S_t^T C_t + D x_t
//
// The inputs are those of gated_linear_scan (fp32 tensors, or raw projection columns whose gates are formed while they are
// staged) and ssm_scan. Token by token, either scan is a chain of one LDS round trip per token: 0.36 - 0.57 us a token
// whatever the grid. With s_t the product of the decays behind token t up to the chunk's end and E that of all of them, a chunk is
//   S' = E S,   P_ij = sum_d (q_i / s_i) (k_j s_j) (j <= i),   o = P v + (q / s) S',   S <- S' + (k s)^T v
// and a scalar decay (ssm) factors out of the sums: P_ij = C_i . B_j dt_j s_j / s_i, no factor above 1 at all. Everything stays
// fp32: v_mfma_f32_16x16x4_f32 multiplies and adds in fp32 (bf16 rows of the second run in ssm_chunk.hip) and the products
// of decays are carried as two floats (Prod). Referred to the chunk's end, the terms that enter the state have one rounding each,
// as in the token loop; their reciprocals meet the outputs alone, where what came in goes first and the chunk's terms follow in
// their order (summed apart and added, decays around 0.5 had 1.05 to 1.17 times the loop's error, so 0.97 to 1.10).
// Error against fp64 (2-norm, carried state / outputs, the token loop's in brackets): 64 x 128, 400 tokens, decays around 0.5
// 6.0e-8 / 6.1e-8 (6.0e-8 / 6.1e-8), 0.95 3.6e-7 / 1.8e-7 (4.5e-7 / 2.1e-7), 0.999 1.5e-6 / 8.5e-7 (1.8e-6 / 1.0e-6); ssm,
// 128 x 64, A around -1 7.3e-8 / 1.2e-7 (7.7e-8 / 1.2e-7), -2.7 8.2e-8 / 1.0e-7 (7.6e-8 / 1.1e-7). Sums of log2 decays in the place
// of the products gave 3.3e-7 / 1.1e-7 in the first.
//
// One workgroup = (sequence, head, 16 NW value columns). A wave keeps 16 columns of the state in accumulator layout, which is
// also the B operand of (q / s) S' when the contraction index runs (tile, register, row quad); v comes straight from memory
// in the layout both products want; P is computed transposed, so that its accumulator layout is the A operand of P v. The
// waves divide P's contraction and add their shares through LDS: one barrier per chunk, behind which only P v is left.
// The next chunk is staged and the one after it loaded meanwhile.
//
// A chunk whose factors could leave the fp32 range (products of decays outside 2^-60 .. 2^60, inputs of 2^28 and above,
// infinities, NaN) is run token by token in the same layout.
//
// Measured (bf16 rows): 4001 tokens of 16 heads of 64 x 128 401 -> 92 us, 4 x 2048 of them 735 -> 155; ssm, 2521 ragged tokens
// of 64 heads of 128 x 64 777 -> 199, 4 x 1024 of 128 heads 1030 -> 276 (log sums: 87, 145, 187, 250). What is left is 2.3 us of
// a compute unit per chunk of the large state, 0.9 of them matrix instructions (68 a wave); the rest is LDS round trips between
// them. Workgroups of four waves, two to a compute unit, because a lane holds 32 rows of state besides its fragments (186
// registers).
//
// Long portions of few sequences are cut into segments that run side by side: pass 1 sums every segment up from a zero state
// (and sets the incoming state aside), a fold turns the sums into each segment's incoming state, pass 2 runs with outputs.
// Segment slot of (sequence s, segment z): q0_s / seg + s + z, distinct for all segments of a step.
#include <type_traits>

#include "mfma_f32.h"

namespace xgm {

using xgk::ld16;
using xgk::unpack8;

constexpr int kCsRaw = 0, kCsPlain = 1, kCsSsm = 2;
constexpr int kCsTok = 16;
constexpr float kCsMaxProd = 1152921504606846976.f, kCsMinProd = 1.f / kCsMaxProd;   // 2^60
__device__ __forceinline__ bool prod_out_of_range(float p) { return !(fabsf(p) > kCsMinProd && fabsf(p) < kCsMaxProd); }

struct ChunkScanArgs {
  const float *q, *f, *k;      // plain: fp32 [T][H dk] (k may be null)
  const void* raw;             // raw: projection rows, columns off_q / off_f;  ssm: rows [x (H dv) | B (G dk) | C (G dk)]
  int64_t ld_raw;
  int off_q, off_f;
  const float *f_bias, *lower;
  const void* v;               // gates: value rows [T][H dv]
  int64_t ld_v;
  const void* dt;              // ssm
  int64_t ld_dt;
  const float *dt_bias, *A_log, *skip;
  int G;
  float* state;
  const int32_t *qsl, *seq_lens, *slots;
  float* o;
  int H, dk, dv, pass, nc, seg;
  float *chA, *chB, *s_in;
};

// eight elements as loaded
template <typename T> struct Raw8;
template <> struct Raw8<bf16> {
  uint4 v;
  __device__ __forceinline__ void load(const bf16* p) { v = ld16(p); }
  __device__ __forceinline__ void get(float (&f)[8]) const { unpack8(v, f); }
  __device__ __forceinline__ bool any_out_of_range() const {   // magnitudes order as their bits do, NaN above them all
    using u16x2 = __attribute__((ext_vector_type(2))) uint16_t;
    const u16x2 m = __builtin_elementwise_max(
        __builtin_elementwise_max(__builtin_bit_cast(u16x2, v.x & 0x7FFF7FFFu), __builtin_bit_cast(u16x2, v.y & 0x7FFF7FFFu)),
        __builtin_elementwise_max(__builtin_bit_cast(u16x2, v.z & 0x7FFF7FFFu), __builtin_bit_cast(u16x2, v.w & 0x7FFF7FFFu)));
    return max(m.x, m.y) >= (__float_as_uint(kChunkMaxIn) >> 16);
  }
};
template <> struct Raw8<float> {
  float4 a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  }
  __device__ __forceinline__ void get(float (&f)[8]) const {
    f[0] = a.x, f[1] = a.y, f[2] = a.z, f[3] = a.w, f[4] = b.x, f[5] = b.y, f[6] = b.z, f[7] = b.w;
  }
  __device__ __forceinline__ bool any_out_of_range() const {
    float f[8];
    get(f);
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) m = max(m, __float_as_uint(f[i]) & 0x7FFFFFFFu);
    return m >= __float_as_uint(kChunkMaxIn);
  }
};

template <typename T, int MODE, int DK, int NW>
__global__ __launch_bounds__(64 * NW, NW == 8 && DK == 64 ? 4 : 2) void chunk_scan_kernel(const ChunkScanArgs a) {
  constexpr bool DENSE = NW == 8 && DK == 64;   // two workgroups of eight waves to a compute unit (one: 4001 tokens 112 us, not 85)
  constexpr int C = kCsTok, MT = DK / 16, NTH = 64 * NW, QE = DK + 4;
  constexpr bool SSM = MODE == kCsSsm;
  constexpr int PT = (MT + NW - 1) / NW;       // 16-channel tiles of P's contraction per wave
  constexpr int CW = DK / NW, TG = 64 / CW, TL = C / TG;   // gates: channels per wave, token groups, tokens per lane
  constexpr int TLN = SSM ? 1 : TL;
  constexpr int BLK = 64, RING = SSM ? 2 * BLK : 1;   // ssm: the step sizes of 64 chunks are formed together, 32 ahead
  constexpr int UN = (2 * C * DK / 8 + NTH - 1) / NTH;   // ssm: 8-channel units of [C | B] per thread
  __shared__ __attribute__((aligned(16))) float qs[2][C * QE], ks[2][C * QE];
  __shared__ __attribute__((aligned(16))) float ws[SSM ? 1 : 2][SSM ? 4 : C * QE];   // decays of a chunk run token by token
  __shared__ __attribute__((aligned(16))) float eh[SSM ? 1 : 2][SSM ? 4 : DK], el[SSM ? 1 : 2][SSM ? 4 : DK];   // E per channel
  __shared__ __attribute__((aligned(16))) float ps[2][NW][256];
  __shared__ __attribute__((aligned(16))) float ri[RING][C], ds[RING][C], dts[RING][C];   // ssm: 1 / s, dt s, dt
  __shared__ float Eh[RING], El[RING], ptot[SSM ? 4 : DK];   // ssm: E per chunk; gates: decay of the segment per channel
  __shared__ int flags[4][NW];

  // workgroups go to the 8 XCDs in turn: heads first, so that short sequences' missing segments empty no XCD, and an XCD
  // takes neighbouring heads (which share B and C)
  const int s = blockIdx.y / a.nc, z = blockIdx.y % a.nc, hx = blockIdx.x;
  const int h = a.H % 8 == 0 ? (hx % 8) * (a.H / 8) + hx / 8 : hx;
  const int q0 = a.qsl[s], qn = a.qsl[s + 1] - q0, slot = a.slots[s];
  const int c0 = z * a.seg, c1 = min(qn, c0 + a.seg);
  if (slot < 0 || c0 >= qn) return;
  const int pass = a.pass, dk = a.dk, dv = a.dv;
  const bool last_seg = c1 == qn;
  if (pass == 1 && last_seg && z > 0) return;   // nobody reads its sum
  const int ctx = a.seq_lens[s] - qn;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, l16 = lane & 15;
  const int col = (blockIdx.z * NW + w) * 16 + l16;
  const bool cok = col < dv;
  const int64_t cs0 = q0 / a.seg + s;
  float* Sg = a.state + (((int64_t)slot * a.H + h) * dk) * dv;
  float* s_in = a.s_in + ((int64_t)s * a.H + h) * (int64_t)dk * dv;

  // ---- incoming state: rows 16 m + 4 g4 + r, column col (rows past dk stay zero)
  f32x4_t S[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) S[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (cok && (pass == 2 || ctx > 0)) {   // (pass 2: the fold left each segment's incoming state in the sum before it)
    const float* first = pass != 2 ? Sg : z == 0 ? s_in : a.chB + ((cs0 + z - 1) * a.H + h) * (int64_t)dk * dv;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * m + 4 * g4 + r;
        if (row < dk) S[m][r] = first[(int64_t)row * dv + col];
      }
  }
  if (pass == 1) {   // segments are summed up from zero; the incoming state is set aside
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * m + 4 * g4 + r;
        if (z == 0 && cok && row < dk) s_in[(int64_t)row * dv + col] = S[m][r];
        S[m][r] = 0.f;
      }
    if (last_seg) return;
  }
  if (!SSM)
    for (int i = tid; i < DK; i += NTH) ptot[i] = 1.f;

  // ---- loads of a chunk into registers, unconverted (a conversion would wait for them); rows past the end repeat the last
  const T* raw = (const T*)a.raw;
  const T* vb = SSM ? raw + h * dv : (const T*)a.v + h * dv;
  const int64_t ld_v = SSM ? a.ld_raw : a.ld_v;
  using F = std::conditional_t<MODE == kCsPlain, float, T>;
  const int cl = lane % CW, tg = lane / CW, ch = CW * w + cl;   // gates: this lane's channel and tokens tg TL ..
  const uint32_t vcol = min(col, dv - 1), ccol = min(ch, dk - 1);
  T vraw[4];                                           // v of tokens 4 r + g4 (positions 4 g4 + r), column col
  F rq[TLN], rf[TLN];
  float rk[MODE == kCsPlain ? TLN : 1];
  Raw8<T> un[SSM ? UN : 1];
  const int gofs = SSM ? a.H * dv + (h / (a.H / a.G)) * dk : 0;   // B's columns; C's are G dk further on
  auto fetch = [&](int t0) {   // (uniform bases, 32-bit lane offsets)
    const int left = max(c1 - t0, 1) - 1;
    const int64_t row0 = q0 + min(t0, c1 - 1);
    const T* vp = vb + row0 * ld_v;
#pragma unroll
    for (int r = 0; r < 4; ++r) vraw[r] = vp[(uint32_t)min(4 * r + g4, left) * (uint32_t)ld_v + vcol];
    if constexpr (SSM) {
      const T* rp = raw + row0 * a.ld_raw + gofs;
#pragma unroll
      for (int j = 0; j < UN; ++j) {
        const int u = tid + NTH * j, is_b = u >= C * DK / 8, tok = (u / (DK / 8)) % C, c = 8 * (u % (DK / 8));
        un[j].load(rp + ((uint32_t)min(tok, left) * (uint32_t)a.ld_raw + (uint32_t)(is_b ? 0 : a.G * dk) + min(c, dk - 8)));
      }
    } else if constexpr (MODE == kCsRaw) {
      const T* rp = raw + row0 * a.ld_raw + h * dk;
#pragma unroll
      for (int i = 0; i < TL; ++i) {
        const uint32_t at = (uint32_t)min(TL * tg + i, left) * (uint32_t)a.ld_raw + ccol;
        rf[i] = rp[at + a.off_f], rq[i] = rp[at + a.off_q];
      }
    } else {
      const int64_t base = (row0 * a.H + h) * dk;
#pragma unroll
      for (int i = 0; i < TL; ++i) {
        const uint32_t at = (uint32_t)(min(TL * tg + i, left) * a.H) * dk + ccol;
        rf[i] = (a.f + base)[at], rq[i] = (a.q + base)[at];
        rk[i] = a.k ? (a.k + base)[at] : 0.f;
      }
    }
  };
  // ---- gates and running decays of the loaded chunk `ci`; whether it must run token by token
  const float rate = SSM ? expf(a.A_log[h]) : 0.f, dtb = SSM ? a.dt_bias[h] : 0.f;
  float vnew[4];
  float fq[TLN], ff[TLN], fk[TLN];
  Prod sg[TLN], E = {1.f, 0.f};
  const float low = MODE == kCsRaw ? a.lower[h * dk + ccol] : 0.f;
  const float fb = MODE == kCsRaw && a.f_bias ? a.f_bias[h * dk + ccol] : 0.f;
  // ssm: step sizes and decays of the BLK chunks from chunk `ci` on (a chunk is 16 lanes)
  auto steps = [&](int ci) {
    const int t0 = c0 + C * ci;
    if (t0 >= c1) return;
    const T* dp = (const T*)a.dt + (int64_t)(q0 + t0) * a.ld_dt + h;
#pragma unroll
    for (int j = 0; j < BLK * C / NTH; ++j) {
      const int t = tid + NTH * j, left = c1 - t0;
      const float d = t < left ? softplusf(ldf(dp + (int64_t)min(t, left - 1) * a.ld_dt) + dtb) : 0.f;
      Prod p = {out_of_range(d) ? __builtin_nanf("") : expf(-rate * d), 0.f};   // (not a number: the chunk runs token by token)
#pragma unroll
      for (int o = 1; o < C; o <<= 1) {   // from this token to the chunk's end
        const Prod dn = {__shfl_down(p.h, o, C), __shfl_down(p.l, o, C)};
        if (l16 + o < C) p = prod_mul(p, dn);
      }
      Prod s = {__shfl_down(p.h, 1, C), __shfl_down(p.l, 1, C)};
      if (l16 == C - 1) s = {1.f, 0.f};
      const int at = (ci + t / C) % RING, pos = tok_pos(l16);
      ri[at][pos] = prod_rcp(s), ds[at][pos] = prod_times(s, d), dts[at][pos] = d;
      if (l16 == 0) Eh[at] = p.h, El[at] = p.l;
    }
  };
  auto gates = [&](int ci, int t0) {
    const int n = c1 - t0;
    bool bad = false;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      vnew[r] = cok && 4 * r + g4 < n ? ldf(&vraw[r]) : 0.f;
      bad |= out_of_range(vnew[r]);
    }
    if constexpr (SSM) {   // C . B is formed before dt x joins: large ones would leave the range where the token loop does not
#pragma unroll
      for (int j = 0; j < UN; ++j) bad |= un[j].any_out_of_range();
    } else {
#pragma unroll
      for (int i = 0; i < TL; ++i) {
        const bool on = TL * tg + i < n && ch < dk;
        if constexpr (MODE == kCsRaw) {
          const float zq = ldf(&rq[i]);
          ff[i] = on ? low + (1.f - low) * sigmoidf(ldf(&rf[i]) + fb) : 1.f;
          fq[i] = on ? siluf(zq) : 0.f;
          fk[i] = 1.f - ff[i];
        } else {
          ff[i] = on ? rf[i] : 1.f;
          fq[i] = on ? rq[i] : 0.f;
          fk[i] = a.k ? (on ? rk[i] : 0.f) : 1.f - ff[i];
        }
        bad |= out_of_range(fq[i]) || out_of_range(fk[i]);
      }
      Prod run = {1.f, 0.f};
#pragma unroll
      for (int i = TL - 1; i >= 0; --i) {
        sg[i] = run;
        run = prod_mul(run, ff[i]);
      }
#pragma unroll
      for (int o = 1; o < TG; o <<= 1) {   // run: from this lane's group to the chunk's end
        const Prod dn = {__shfl_down(run.h, o * CW, 64), __shfl_down(run.l, o * CW, 64)};
        if (tg + o < TG) run = prod_mul(run, dn);
      }
      Prod after = {__shfl_down(run.h, CW, 64), __shfl_down(run.l, CW, 64)};
      if (tg == TG - 1) after = {1.f, 0.f};
#pragma unroll
      for (int i = 0; i < TL; ++i) {
        sg[i] = prod_mul(sg[i], after);
        bad |= prod_out_of_range(sg[i].h);
      }
      E = run;   // (of the first group's lanes)
      bad |= prod_out_of_range(E.h);
    }
    const int any = __any(bad);
    if (lane == 0) flags[ci & 3][w] = any;
  };
  auto flagged = [&](int ci) {
    int f = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) f |= flags[ci & 3][i];
    // (ssm: a chunk's whole product bounds them all)
    return __builtin_amdgcn_readfirstlane(f | (SSM && prod_out_of_range(Eh[ci % RING]))) != 0;
  };
  // ---- the loaded chunk's operands into LDS buffer `buf`
  auto stage = [&](int buf, bool slow, int n) {
    if constexpr (SSM) {
#pragma unroll
      for (int j = 0; j < UN; ++j) {
        const int u = tid + NTH * j, is_b = u >= C * DK / 8, tok = (u / (DK / 8)) % C, c = 8 * (u % (DK / 8));
        if (u < 2 * C * DK / 8) {
          float f[8];
          un[j].get(f);
          const bool on = tok < n && c < dk;
          float* to = (is_b ? ks[buf] : qs[buf]) + tok_pos(tok) * QE + c;
          *reinterpret_cast<float4*>(to) = on ? make_float4(f[0], f[1], f[2], f[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
          *reinterpret_cast<float4*>(to + 4) = on ? make_float4(f[4], f[5], f[6], f[7]) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < TL; ++i) {
        const int at = tok_pos(TL * tg + i) * QE + ch;
        qs[buf][at] = slow ? fq[i] : prod_div(fq[i], sg[i]);
        ks[buf][at] = slow ? fk[i] : prod_times(sg[i], fk[i]);
        if (slow) ws[buf][at] = ff[i];
      }
      if (tg == 0) {
        eh[buf][ch] = E.h, el[buf][ch] = E.l;
        ptot[ch] = slow ? ptot[ch] * E.h : prod_times(E, ptot[ch]);
      }
    }
  };

  const float skip = SSM ? a.skip[h] : 0.f;
  float ptot_h = 1.f;   // ssm: decay of the segment
  float v[4];
  // chunk 0 staged, chunk 1 in registers
  fetch(c0);
  if (SSM) steps(0);
  gates(0, c0);
  __syncthreads();
  bool slow = flagged(0);
  stage(0, slow, c1 - c0);
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = vnew[r];
  fetch(c0 + C);
  gates(1, c0 + C);
  __syncthreads();
  for (int t0 = c0, ci = 0; t0 < c1; t0 += C, ++ci) {
    const int buf = ci & 1, n = min(C, c1 - t0);
    // the next chunk's operands, and the one after it on its way behind this one's products
    const bool next_slow = flagged(ci + 1), more = t0 + 2 * C < c1;
    float vn[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) vn[r] = vnew[r];
    if (t0 + C < c1) stage(buf ^ 1, next_slow, c1 - t0 - C);
    if (more) fetch(t0 + 2 * C);
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};   // o: tokens 4 r + g4, column col
    const float* Q = qs[buf];
    const float* K = ks[buf];
    if (slow) {
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int tg = 0; tg < 4; ++tg) {
          const int at = 4 * tg + tt;   // token 4 tt + tg
          if (4 * tt + tg < n) {
            float vv = __shfl(v[tt], 16 * tg + l16, 64), dec = 0.f, part[4] = {0.f, 0.f, 0.f, 0.f};
            if (SSM) {
              dec = expf(-rate * dts[ci % RING][at]);
              vv *= dts[ci % RING][at];
              ptot_h *= dec;
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
              float qr[4], kr[4], wr[4] = {dec, dec, dec, dec};
              ld4(Q + at * QE + 16 * m + 4 * g4, qr);
              ld4(K + at * QE + 16 * m + 4 * g4, kr);
              if (!SSM) ld4(ws[SSM ? 0 : buf] + at * QE + 16 * m + 4 * g4, wr);
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                S[m][r] = MODE == kCsRaw ? fmaf(wr[r], S[m][r] - vv, vv) : fmaf(wr[r], S[m][r], kr[r] * vv);
                part[r] = fmaf(S[m][r], qr[r], part[r]);
              }
            }
            float sum = (part[0] + part[1]) + (part[2] + part[3]);
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
            if (g4 == tg) acc[tt] = sum;
          }
        }
    } else {
      // the state's own decay first
      if constexpr (SSM) {
        const Prod Ec = {Eh[ci % RING], El[ci % RING]};
        ptot_h = prod_times(Ec, ptot_h);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r) S[m][r] = prod_times(Ec, S[m][r]);
      } else {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          float e[4], f[4];
          ld4(eh[SSM ? 0 : buf] + 16 * m + 4 * g4, e);
          ld4(el[SSM ? 0 : buf] + 16 * m + 4 * g4, f);
#pragma unroll
          for (int r = 0; r < 4; ++r) S[m][r] = prod_times({e[r], f[r]}, S[m][r]);
        }
      }
      if (pass != 1) {
        // this wave's share of P^T: positions j = 4 g4 + r, column i = l16
        f32x4_t pt[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) pt[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 0; p < PT; ++p) {
          const int m = w + NW * p;
          if (m < MT) {
            float kr[4], qr[4];
            ld4(K + l16 * QE + 16 * m + 4 * g4, kr);
            ld4(Q + l16 * QE + 16 * m + 4 * g4, qr);
#pragma unroll
            for (int r = 0; r < 4; ++r) pt[r] = mfma_f32(kr[r], qr[r], pt[r]);
          }
        }
        *reinterpret_cast<float4*>(&ps[buf][w][4 * lane]) = make_float4(
            (pt[0][0] + pt[1][0]) + (pt[2][0] + pt[3][0]), (pt[0][1] + pt[1][1]) + (pt[2][1] + pt[3][1]),
            (pt[0][2] + pt[1][2]) + (pt[2][2] + pt[3][2]), (pt[0][3] + pt[1][3]) + (pt[2][3] + pt[3][3]));
        // four tiles' fragments in flight; sums side by side for short chains of roundings (two in the form that 128 registers hold)
        constexpr int MB = MT < 4 ? MT : 4, NP = DENSE ? 2 : MB;
        f32x4_t part[NP];
#pragma unroll
        for (int m = 0; m < NP; ++m) part[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m0 = 0; m0 < MT; m0 += 4) {
          float qr[MB][4];
#pragma unroll
          for (int m = 0; m < MB; ++m) ld4(Q + l16 * QE + 16 * (m0 + m) + 4 * g4, qr[m]);
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int m = 0; m < MB; ++m) part[m % NP] = mfma_f32(qr[m][r], S[m0 + m][r], part[m % NP]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = NP == 4 ? (part[0][r] + part[1][r]) + (part[NP - 2][r] + part[NP - 1][r]) : part[0][r] + part[1][r];
        if (SSM) {
          float x[4];
          ld4(&ri[ci % RING][4 * g4], x);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[r] *= x[r];
        }
      }
      float vs[4];
      if constexpr (SSM) {
        float d[4];
        ld4(&ds[ci % RING][4 * g4], d);
#pragma unroll
        for (int r = 0; r < 4; ++r) vs[r] = v[r] * d[r];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) vs[r] = v[r];
      }
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < 4; ++t) S[m] = mfma_f32(K[(4 * g4 + t) * QE + 16 * m + l16], vs[t], S[m]);
    }
    if (more) gates(ci + 2, t0 + 2 * C);
    if (SSM && ci % BLK == BLK / 2) steps(ci + BLK / 2);
    __syncthreads();
    if (pass != 1) {
      if (!slow) {
        constexpr int NP = MT < NW ? MT : NW;   // (2, 4 or 8 shares, added in pairs)
        float p[4], x[NP][4];
#pragma unroll
        for (int i = 0; i < NP; ++i) ld4(&ps[buf][i][4 * lane], x[i]);
#pragma unroll
        for (int o = NP / 2; o > 0; o >>= 1)
#pragma unroll
          for (int i = 0; i < o; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) x[i][r] += x[i + o][r];
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = x[0][r];
        if constexpr (SSM) {
          float d[4];
          ld4(&ds[ci % RING][4 * g4], d);
          const float x = ri[ci % RING][l16];
#pragma unroll
          for (int r = 0; r < 4; ++r) p[r] *= d[r] * x;
        }
        // (what came in, then the chunk's terms in their order: one rounding of the whole)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc = mfma_f32(4 * r + g4 <= tok_pos(l16) ? p[r] : 0.f, v[r], acc);
      }
      if (cok) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (4 * r + g4 < n)
            a.o[((int64_t)(q0 + t0 + 4 * r + g4) * a.H + h) * dv + col] = SSM ? fmaf(skip, v[r], acc[r]) : acc[r];
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = vn[r];
    slow = next_slow;
  }
  // ---- outgoing state, or the segment's sum
  float* last = pass == 1 ? a.chB + ((cs0 + z) * a.H + h) * (int64_t)dk * dv : Sg;
  if (cok && (pass == 1 || last_seg)) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * m + 4 * g4 + r;
        if (row < dk) last[(int64_t)row * dv + col] = S[m][r];
      }
  }
  if (pass == 1 && blockIdx.z == 0)
    for (int i = tid; i < dk; i += NTH) a.chA[((cs0 + z) * a.H + h) * dk + i] = SSM ? ptot_h : ptot[SSM ? 0 : i];
}

// ================================================================== host launchers
int64_t chunk_scan_scratch_floats(int T_, int ns, int H, int dk, int dv, int seg) {
  const int64_t cslots = T_ / seg + ns + 1;
  return (cslots * (dv + 1) + (int64_t)ns * dv) * H * dk;
}

// Incoming states of the segments: a thread walks one state element over the segments of its sequence and leaves the state
// behind segment z in z's own sum.
__global__ __launch_bounds__(256) void chunk_scan_fold_kernel(const ChunkScanArgs a) {
  const int s = blockIdx.y, h = blockIdx.z, i = blockIdx.x * 256 + threadIdx.x, n = a.dk * a.dv;
  const int q0 = a.qsl[s], qn = a.qsl[s + 1] - q0;
  if (a.slots[s] < 0 || i >= n) return;
  const int nseg = (qn + a.seg - 1) / a.seg - 1;   // (nobody needs the state behind the last one)
  const int64_t cs0 = q0 / a.seg + s, stride = (int64_t)a.H * n;
  float* B = a.chB + (cs0 * a.H + h) * n + i;
  const float* A = a.chA + (cs0 * a.H + h) * a.dk + i / a.dv;
  float S = a.s_in[((int64_t)s * a.H + h) * n + i];
  for (int z0 = 0; z0 < nseg; z0 += 8) {
    float b[8], f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int z = min(z0 + j, nseg - 1);
      b[j] = B[z * stride], f[j] = A[(int64_t)z * a.H * a.dk];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (z0 + j < nseg) {
        S = S == 0.f ? b[j] : fmaf(f[j], S, b[j]);   // (a product past fp32 of finite growths leaves a zero zero)
        B[(z0 + j) * stride] = S;
      }
    }
  }
}

static int run_chunk_scan(ChunkScanArgs a, bool f32, int mode, int ns, int max_q, int T_, int seg, float* scratch,
                          hipStream_t st) {
  if (ns <= 0 || max_q <= 0) return 0;
  if (a.H < 1 || a.dk < 1 || a.dk > 128 || a.dv < 1 || (scratch && (seg < kCsTok || seg % kCsTok))) return -1;
  if (!scratch) seg = (max_q + kCsTok - 1) / kCsTok * kCsTok;
  const int64_t cslots = T_ / seg + ns + 1;
  a.seg = seg, a.nc = (max_q + seg - 1) / seg;
  a.chA = scratch, a.chB = scratch ? scratch + cslots * a.H * a.dk : nullptr;
  a.s_in = scratch ? a.chB + cslots * a.H * a.dk * a.dv : nullptr;
  const int nw = a.dv > 64 && mode != kCsSsm ? 8 : 4;   // (ssm: the wide state leaves registers for one wave per SIMD and more)
  if ((int64_t)ns * a.nc > 65535) return -1;
  const dim3 grid(a.H, ns * a.nc, (a.dv + 16 * nw - 1) / (16 * nw));
#define XGM_CS3(MODE, DK, NW)                                                              \
  XGM_DISPATCH_T(f32, for (int pass = a.nc > 1 ? 1 : 0; pass < (a.nc > 1 ? 3 : 1); ++pass) { \
    a.pass = pass;                                                                         \
    chunk_scan_kernel<T, MODE, DK, NW><<<grid, 64 * NW, 0, st>>>(a);                        \
    if (pass == 1) chunk_scan_fold_kernel<<<dim3((a.dk * a.dv + 255) / 256, ns, a.H), 256, 0, st>>>(a); \
  })                                                                                       \
  return 0;
#define XGM_CS2(MODE, DK) \
  if (nw == 8) { XGM_CS3(MODE, DK, 8) } else { XGM_CS3(MODE, DK, 4) }
#define XGM_CS(DK)                          \
  if (mode == kCsSsm) { XGM_CS3(kCsSsm, DK, 4) } \
  if (mode == kCsRaw) { XGM_CS2(kCsRaw, DK) }    \
  XGM_CS2(kCsPlain, DK)
  if (a.dk <= 32) { XGM_CS(32) }
  if (a.dk <= 64) { XGM_CS(64) }
  XGM_CS(128)
#undef XGM_CS
#undef XGM_CS2
#undef XGM_CS3
}

// the inputs of gated_linear_scan (without a constant decay or a bonus); scratch: chunk_scan_scratch_floats, or null
int chunk_scan_gates(const float* q, const float* f, const float* k, const void* raw, int64_t ld_raw, int off_q, int off_f,
                     const float* f_bias, const float* lower, const void* v, bool v_f32, int64_t ld_v, float* state,
                     const int32_t* qsl, const int32_t* seq_lens, const int32_t* slots, float* o, int ns, int max_q, int T_,
                     int H, int dk, int dv, int seg, float* scratch, hipStream_t st) {
  if (raw ? !lower : (!q || !f)) return -1;
  ChunkScanArgs a = {};
  a.q = q, a.f = f, a.k = k, a.raw = raw, a.ld_raw = ld_raw, a.off_q = off_q, a.off_f = off_f, a.f_bias = f_bias;
  a.lower = lower, a.v = v, a.ld_v = ld_v, a.G = 1, a.state = state, a.qsl = qsl, a.seq_lens = seq_lens, a.slots = slots;
  a.o = o, a.H = H, a.dk = dk, a.dv = dv;
  return run_chunk_scan(a, v_f32, raw ? kCsRaw : kCsPlain, ns, max_q, T_, seg, scratch, st);
}

// the inputs of ssm_scan; B and C are read 8 channels at a time: N a multiple of 8, rows and their B / C columns on 16 bytes
int chunk_scan_ssm(const void* xbc, bool f32, int64_t ld_x, const void* dt_raw, int64_t ld_dt, const float* dt_bias,
                   const float* A_log, const float* Dskip, float* state, const int32_t* qsl, const int32_t* seq_lens,
                   const int32_t* slots, float* y, int ns, int max_q, int T_, int H, int G, int N, int P, int seg,
                   float* scratch, hipStream_t st) {
  const int64_t al = f32 ? 4 : 8;
  if (H <= 0 || G <= 0 || H % G != 0 || N % 8 || (uintptr_t)xbc % 16 || ld_x % al || (H * P) % al) return -1;
  ChunkScanArgs a = {};
  a.raw = xbc, a.ld_raw = ld_x, a.dt = dt_raw, a.ld_dt = ld_dt, a.dt_bias = dt_bias, a.A_log = A_log, a.skip = Dskip;
  a.G = G, a.state = state, a.qsl = qsl, a.seq_lens = seq_lens, a.slots = slots, a.o = y, a.H = H, a.dk = N, a.dv = P;
  return run_chunk_scan(a, f32, kCsSsm, ns, max_q, T_, seg, scratch, st);
}

}  // namespace xgm
