// Generalized delta rule over prompt portions, in chunks of 16 tokens on the fp32 matrix cores (bf16 or fp32 rows, fp32 state):
//
//   S_t = diag(w_t) S_(t-1) - b_t (u_t^T S_(t-1)) + k_t v_t^T,   o_t = S_t^T r_t,      b = a u, u = k / |k|, w = e^(-c sigmoid)
//
// Token by token this is a chain of two reductions per token (0.45 us). Let s_t be the product of the decays behind token t up to
// the chunk's end, E that of all of them, S' = E S, and u' = u / s_(t-1), b' = b s_t, k' = k s_t, r' = r / s_t (a decay is at
// least 0.545: 2^-14 over a chunk). With M = u' b'^T and N = u' k'^T strictly below the diagonal, P = r' k'^T and Q = r' b'^T up
// to it and T = (1 + M)^-1, what token t takes out of the state is y = T (u' S' + N v), and
//   y = (U E) S + V,       U = T u', V = T N v,
//   o = (R E) S + O,       R = r' - Q U, O = P v - Q V,
//   S <- E S + k'^T v - b'^T y.
// (U E and R E are formed from u and r times the decays before them, R E = r E / s - Q U E: one rounding less for each factor.)
// Only the right factors meet the state, so a first launch forms U E, V, R E, O, k', b' of all chunks at once (one wave per chunk
// and head; T by forward substitution: the compact form of a product of rank-one updates, Bischof and Van Loan 1987, as Yang et al.
// 2024 use it for the delta rule over chunks of a sequence) and the chain that is left is three matrix products per 16 tokens. All of
// it is fp32 arithmetic, the products of decays two floats each (Prod).
//
// Error against fp64 (2-norm, carried state / outputs, the token loop's in brackets), 497 to 1024 tokens of 32 heads of 64, r with
// a share of k: decays around 0.97 3.03e-7 / 1.99e-7 (3.03e-7 / 1.97e-7), 0.73 6.6e-8 / 4.9e-8 (6.6e-8 / 4.9e-8), 0.55 4.7e-8 /
// 4.3e-8 (4.6e-8 / 4.5e-8); heads of 32 0.92 to 1.03 of the loop's. (Sums of log2 decays and one chain per sum gave 1.8e-7 / 2.3e-7
// in the second.) That takes: separate sums, because k . r has one sign in a trained model and a chain of 64 rounds at the
// whole sum's size, and P in two floats (4.9e-8 in the second; 6.1e-8 in one, from half as many chains); what is taken out of the
// state and of the outputs summed up by itself and before the tokens' own terms, the latest and largest of them last; E in two
// floats.
//
// The second launch has a wave per 16 x 16 of the state: the waves of a column tile (four for heads of 64) sum y and the outputs over
// their rows and hand each other the sums through LDS, y at the one barrier of a chunk and the outputs' behind it, to be added and
// stored behind the next. A workgroup takes 32 columns, so a head of 64 has two and 32 heads of 4 sequences fill the chip, two waves to
// a SIMD. The first launch writes every operand in the order of the matrix instructions' lanes; the waves bring it in by LDS DMA, four
// chunks ahead, and read a chunk's operands while the one before it still adds to the state. A chunk with an input out of range
// (infinities, NaN, 2^28 and above) is stored as w, b, u, k, r and run token by token.
//
// Measured, bf16 rows, 4 x 2048 tokens of 32 heads of 64 in a step, us: the first launch 186 -> 169 (in one trace; it writes 24.6 KB per chunk and head,
// 570 MB with its reads; three exponentials per token and channel, which a branch per token kept from overlapping, and 80 addresses
// formed lane by lane were the difference), the second 168 -> 138, 1.1 us a chunk. It was two waves per 16 columns and one to a
// SIMD, which waited for each of its instructions: with DMA addresses kept instead of formed (a third of 260 instructions a chunk)
// and the outputs' products behind y's 146, with four waves 144, with no branches between the products 138. What is left of a chunk is the
// way from one matrix instruction to the next and through LDS, 0.43 us of it the instructions: with every load from the same 25 KB
// it takes 137, with nothing stored 133.
#include "glds.h"
#include "mfma_f32.h"

namespace xgm {

constexpr int kDcTok = 16;
constexpr float kDeltaDecay = -0.6065306597126334f;   // log w = this * sigmoid

// floats per (chunk, head): [U E | R E | k' | -b' | V | O] in lane order, then E per channel (at 0 and 2 D), the flag at D
constexpr int dc_stride(int D) { return 6 * kDcTok * D + 256; }

template <typename T, int D>
__global__ __launch_bounds__(64, 2) void delta_chunk_prep_kernel(const T* __restrict__ proj, int64_t ld, int off_r, int off_k,
                                                                 int off_v, int off_a, const T* __restrict__ wl,
                                                                 int64_t ld_wl, const float* __restrict__ a_bias,
                                                                 const float* __restrict__ w0, const int32_t* __restrict__ qsl,
                                                                 const int32_t* __restrict__ slots, float* __restrict__ prep,
                                                                 int H) {
  constexpr int C = kDcTok, MT = D / 16, QE = D + 4, TPL = C * D / 64;   // (token, channel) pairs per lane
  constexpr int TG = 64 / D, TT = C / TG;                                // token groups, tokens per lane
  static_assert(D == 64 || D == 32, "a lane owns one channel");
  __shared__ __attribute__((aligned(16))) float us[C * QE], rs[C * QE], ks[C * QE], bs[C * QE], ts[C * 20];
  const int h = blockIdx.x, c = blockIdx.y, s = blockIdx.z;
  const int q0 = qsl[s], qn = qsl[s + 1] - q0, n = min(C, qn - C * c);
  if (slots[s] < 0 || n <= 0) return;
  const int lane = threadIdx.x, g4 = lane >> 4, l16 = lane & 15, d = lane % D, tg = lane / D;
  float* dst = prep + ((int64_t)(q0 / C + s + c) * H + h) * dc_stride(D);
  const T* row = proj + (int64_t)(q0 + C * c) * ld + h * D;
  const T* wrow = wl + (int64_t)(q0 + C * c) * ld_wl + h * D;

  // ---- this lane's channel, tokens tg TT .. (rows past the end repeat the last and are masked)
  T xr[TT], xk[TT], xa[TT], xw[TT], xv[MT][4];
  const int t0 = TG == 1 ? 0 : min(TT * tg, n - 1);   // (heads of 64: the same for all lanes, and so the rows' addresses)
  const T *at = row + t0 * ld, *wat = wrow + t0 * ld_wl;
#pragma unroll
  for (int i = 0; i < TT; ++i) {
    xk[i] = (at + off_k)[(uint32_t)d], xw[i] = wat[(uint32_t)d];
    xa[i] = (at + off_a)[(uint32_t)d], xr[i] = (at + off_r)[(uint32_t)d];
    const bool more = (TG == 1 ? 0 : TT * tg) + i + 1 < n;
    at += more ? ld : 0, wat += more ? ld_wl : 0;
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const T* at = row + off_v + l16 + (int64_t)min(4 * t + g4, n - 1) * ld;
#pragma unroll
    for (int m = 0; m < MT; ++m) xv[m][t] = at[16 * m];
  }
  const float ab = a_bias[h * D + d], wb = w0[h * D + d];
  bool bad = false;
  float k[TT];
#pragma unroll
  for (int i = 0; i < TT; ++i) {
    k[i] = TT * tg + i < n ? ldf(&xk[i]) : 0.f;
    bad |= out_of_range(k[i]);
    ks[tok_pos(TT * tg + i) * QE + d] = k[i];
  }
  __syncthreads();
  float ksq = 0.f;   // |k|^2 of the token at position l16
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    float x[4];
    ld4(ks + l16 * QE + 16 * m + 4 * g4, x);
#pragma unroll
    for (int r = 0; r < 4; ++r) ksq = fmaf(x[r], x[r], ksq);
  }
  ksq += __shfl_xor(ksq, 16, 64);
  ksq += __shfl_xor(ksq, 32, 64);
  const float inv = 1.f / sqrtf(ksq + 1e-6f);
  float v[MT][4];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      v[m][t] = 4 * t + g4 < n ? ldf(&xv[m][t]) : 0.f;
      bad |= out_of_range(v[m][t]);
    }
  float wt[TT], u[TT], a[TT], r_[TT];
#pragma unroll
  for (int i = 0; i < TT; ++i) {
    const bool on = TT * tg + i < n;
    u[i] = k[i] * __shfl(inv, tok_pos(TT * tg + i), 64);
    // (formed for the repeated rows too: a branch per token keeps one token's exponentials waiting for the other's)
    wt[i] = expf(kDeltaDecay * sigmoidf(ldf(&xw[i]) + wb)), a[i] = sigmoidf(ldf(&xa[i]) + ab);
    asm volatile("" : "+v"(wt[i]), "+v"(a[i]));
    wt[i] = on ? wt[i] : 1.f, a[i] = on ? a[i] : 0.f;
    r_[i] = on ? ldf(&xr[i]) : 0.f;
    bad |= out_of_range(r_[i]) || out_of_range(a[i]) || out_of_range(wt[i]);
  }
  const bool slow = __any(bad);
  if (lane == 0) dst[6 * C * D + D] = slow ? 1.f : 0.f;
  if (slow) {   // [w | b | u | k | r] as rows
#pragma unroll
    for (int i = 0; i < TT; ++i) {
      float* to = dst + (TT * tg + i) * D + d;
      to[0] = wt[i], to[C * D] = a[i] * u[i], to[2 * C * D] = u[i], to[3 * C * D] = k[i], to[4 * C * D] = r_[i];
    }
    return;
  }
  __syncthreads();   // (ks is rewritten)
  Prod run = {1.f, 0.f}, pre = run;   // from the token behind this one to the chunk's end, from the chunk's start to this one
  if (TG == 2) {
#pragma unroll
    for (int i = 0; i < TT; ++i) run = prod_mul(run, wt[i]);
    const Prod up = {__shfl_xor(run.h, D % 64, 64), __shfl_xor(run.l, D % 64, 64)};
    run = tg ? Prod{1.f, 0.f} : up;
    pre = tg ? up : Prod{1.f, 0.f};
  }
#pragma unroll
  for (int i = TT - 1; i >= 0; --i) {
    const int at = tok_pos(TT * tg + i) * QE + d;
    rs[at] = prod_div(r_[i], run), ks[at] = prod_times(run, k[i]), bs[at] = prod_times(run, a[i] * u[i]);
    run = prod_mul(run, wt[i]);
    us[at] = prod_div(u[i], run);
  }
  if (tg == 0) dst[6 * C * D + d] = run.h, dst[6 * C * D + 2 * D + d] = run.l;
  // u and r referred to the chunk's start, one rounding each: what U E and R E are made of
  float ue[TT], re[TT];
#pragma unroll
  for (int i = 0; i < TT; ++i) {
    ue[i] = prod_times(pre, u[i]);
    pre = prod_mul(pre, wt[i]);
    re[i] = prod_times(pre, r_[i]);
  }
  __syncthreads();

  // ---- the four 16 x 16 products, transposed: lane holds [position l16][position 4 g4 + r], the A operand of what follows. Each is
  // the sum of four chains (k . r of a trained model has one sign: a chain of 64 would round at the size of the whole sum).
  f32x4_t Mc[4], Nc[4], Pc[8], Qc[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) Mc[r] = Nc[r] = Pc[r] = Pc[4 + r] = Qc[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    float xu[4], xrr[4], xkk[4], xb[4];
    const int at = l16 * QE + 16 * m + 4 * g4;
    ld4(us + at, xu), ld4(rs + at, xrr), ld4(ks + at, xkk), ld4(bs + at, xb);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      Mc[r] = mfma_f32(xb[r], xu[r], Mc[r]);
      Nc[r] = mfma_f32(xkk[r], xu[r], Nc[r]);
      Pc[4 * (m % 2) + r] = mfma_f32(xkk[r], xrr[r], Pc[4 * (m % 2) + r]);
      Qc[r] = mfma_f32(xb[r], xrr[r], Qc[r]);
    }
  }
  float M[4], N[4], P[4], Pl[4], Q[4];   // P as two floats: its part of an output is the output's size
  const int ti = tok_pos(l16);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int j = 4 * r + g4;   // the token at position 4 g4 + r
    M[r] = j < ti ? (Mc[0][r] + Mc[1][r]) + (Mc[2][r] + Mc[3][r]) : 0.f;
    N[r] = j < ti ? (Nc[0][r] + Nc[1][r]) + (Nc[2][r] + Nc[3][r]) : 0.f;
    const Prod p0 = two_sum(Pc[0][r] + Pc[1][r], Pc[2][r] + Pc[3][r]), p1 = two_sum(Pc[4][r] + Pc[5][r], Pc[6][r] + Pc[7][r]);
    const Prod p = two_sum(p0.h, p1.h);
    P[r] = j <= ti ? p.h : 0.f, Pl[r] = j <= ti ? p.l + (p0.l + p1.l) : 0.f;
    Q[r] = j <= ti ? -((Qc[0][r] + Qc[1][r]) + (Qc[2][r] + Qc[3][r])) : 0.f;   // (Q enters with its sign)
  }
  *reinterpret_cast<float4*>(ts + l16 * 20 + 4 * g4) = make_float4(M[0], M[1], M[2], M[3]);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TT; ++i) {
    const int at = tok_pos(TT * tg + i) * QE + d;
    us[at] = ue[i], rs[at] = re[i];
  }
  // ---- T = (1 + M)^-1: lane l16 solves for token l16's column, x_i = delta - sum_(j < i) M_ij x_j
  float x[C];
#pragma unroll
  for (int i = 0; i < C; ++i) {
    float acc = i == l16 ? 1.f : 0.f;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      if (a < i) {
        float mm[4];   // tokens a, a + 4, a + 8, a + 12
        ld4(ts + tok_pos(i) * 20 + 4 * a, mm);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (a + 4 * r < i) acc = fmaf(-mm[r], x[a + 4 * r], acc);
      }
    }
    x[i] = acc;
  }
  __syncthreads();
  if (g4 == 0) {
#pragma unroll
    for (int i = 0; i < C; ++i) ts[tok_pos(i) * 20 + tok_pos(l16)] = x[i];
  }
  __syncthreads();
  float Tf[4];
  ld4(ts + l16 * 20 + 4 * g4, Tf);   // T[l16][4 g4 + r]

  auto put = [&](int which, int m, f32x4_t y) {
    *reinterpret_cast<float4*>(dst + which * C * D + 256 * m + 4 * lane) = make_float4(y[0], y[1], y[2], y[3]);
  };
  // ---- U E (transposed product: position l16, channels 16 m + 4 g4 + r); k' and -b' as the A operands of the state's update
  f32x4_t U[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    U[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    f32x4_t kk, bb;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int at = (4 * g4 + t) * QE + 16 * m + l16;
      U[m] = mfma_f32(us[at], Tf[t], U[m]);
      kk[t] = ks[at], bb[t] = -bs[at];
    }
    put(0, m, U[m]), put(2, m, kk), put(3, m, bb);
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < MT; ++m)
    *reinterpret_cast<float4*>(us + l16 * QE + 16 * m + 4 * g4) = make_float4(U[m][0], U[m][1], U[m][2], U[m][3]);
  __syncthreads();
  // ---- R E, then V and O column tile by column tile
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    float r0[4];
    ld4(rs + l16 * QE + 16 * m + 4 * g4, r0);
    f32x4_t y = {0.f, 0.f, 0.f, 0.f}, V = y, O = y, R = y;   // (what is taken out is summed up first: fewer roundings of the whole)
#pragma unroll
    for (int t = 0; t < 4; ++t) R = mfma_f32(us[(4 * g4 + t) * QE + 16 * m + l16], Q[t], R);
#pragma unroll
    for (int t = 0; t < 4; ++t) R[t] += r0[t];
    put(1, m, R);
#pragma unroll
    for (int t = 0; t < 4; ++t) y = mfma_f32(N[t], v[m][t], y);
#pragma unroll
    for (int t = 0; t < 4; ++t) V = mfma_f32(Tf[t], y[t], V);
#pragma unroll
    for (int t = 0; t < 4; ++t) O = mfma_f32(Q[t], V[t], O);
#pragma unroll
    for (int t = 0; t < 4; ++t) O = mfma_f32(Pl[t], v[m][t], O);
#pragma unroll
    for (int t = 0; t < 4; ++t) O = mfma_f32(P[t], v[m][t], O);
    put(4, m, V), put(5, m, O);
  }
}

template <typename T, int D>
__global__ __launch_bounds__(8 * D, 1) void delta_chunk_scan_kernel(const float* __restrict__ prep, const T* __restrict__ proj,
                                                                    int64_t ld, int off_v, float* __restrict__ state,
                                                                    const int32_t* __restrict__ qsl,
                                                                    const int32_t* __restrict__ seq_lens,
                                                                    const int32_t* __restrict__ slots, float* __restrict__ o,
                                                                    int H) {
  constexpr int C = kDcTok, MT = D / 16, W = 2 * MT, RING = D == 64 ? 5 : 6;
  constexpr int OPS = 4 * C * D * 4, VO = 2 * C * 32 * 4, FRAG = OPS + VO;   // bytes: [U | R | k' | -b'], this half's [V | O]
  constexpr int VROWS = C * 32 * sizeof(T), SLOT = FRAG + 1024 + VROWS;      // ... [E, flag | v rows]
  constexpr int NE = FRAG / 1024, NP = NE + 1 + VROWS / 1024, DMA = (NP + W - 1) / W;   // kilobytes of a chunk, loads per wave
  constexpr int HAND = 2 * W * 1024;                                         // handed over: y of all waves, then their outputs' sums
  constexpr int VL = 32 * sizeof(T) / 16;                                    // lanes per v row
  constexpr int NO = 4 / MT;                                                 // of a lane's four output rows the wave's share
  static_assert(RING * SLOT + 2 * HAND <= 160 * 1024 && (RING - 2) * DMA < 64 && W * (DMA - 1) <= NE, "delta_chunk_scan geometry");
  __shared__ __attribute__((aligned(1024))) char lds[RING * SLOT + 2 * HAND];
  const int h = blockIdx.x, s = blockIdx.y, half = blockIdx.z;
  const int q0 = qsl[s], qn = qsl[s + 1] - q0, slot = slots[s];
  if (slot < 0 || qn <= 0) return;
  const int ctx = seq_lens[s] - qn;
  const int lane = threadIdx.x & 63, g4 = lane >> 4, l16 = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ct = w / MT, par = w % MT;
  const int col = 32 * half + 16 * ct + l16;
  float* Sg = state + ((int64_t)slot * H + h) * D * D + (16 * par + 4 * g4) * D + col;
  f32x4_t S;   // rows 16 par + 4 g4 ..
#pragma unroll
  for (int r = 0; r < 4; ++r) S[r] = ctx > 0 ? Sg[r * D] : 0.f;
  const int nch = (qn + C - 1) / C;
  const float* base = prep + ((int64_t)(q0 / C + s) * H + h) * dc_stride(D);
  const int64_t step = (int64_t)H * dc_stride(D) * 4;

  // Every wave issues DMA loads, past the last chunk too (its waits count them, and the last chunk is brought in again; so is a slot's
  // last kilobyte where the waves have more loads than there are). An address is the chunk's, the same for all lanes, plus what a
  // lane keeps: formed anew for every load, these were a third of the loop's instructions. The last of a wave's loads, which may be
  // v's, goes from a pointer of the lane's.
  uint32_t from[DMA];
#pragma unroll
  for (int i = 0; i < DMA; ++i) {
    const int kb = W * i + w, vo = kb - OPS / 1024;   // (V and O: two of their MT kilobytes each)
    from[i] = 16 * lane + 1024 * (kb == NE ? 6 * C * D / 256 : vo < 0 ? kb : OPS / 1024 + (vo >> 1) * MT + 2 * half + (vo & 1));
  }
  const int kb_last = min(W * (DMA - 1) + w, NP - 1);
  const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const char *p_last = reinterpret_cast<const char*>(base) + from[DMA - 1], *p_end = p_last + (nch - 1) * step;
  int64_t p_step = step;
  if (kb_last > NE) {
    const int r = (kb_last - NE - 1) * (64 / VL) + lane / VL;
    const T* at = proj + (int64_t)q0 * ld + off_v + h * D + 32 * half + (lane % VL) * (16 / sizeof(T));
    p_last = reinterpret_cast<const char*>(at + min(r, qn - 1) * ld);
    p_end = reinterpret_cast<const char*>(at + min(C * (nch - 1) + r, qn - 1) * ld);
    p_step = C * ld * sizeof(T);
  }
  int c_in = 0;              // the chunk that is asked for next,
  uint32_t at_in = ring;     // and its slot
  auto operands = [&]() __attribute__((always_inline)) {
    const uint64_t at = (uint64_t)(uintptr_t)base + (uint64_t)c_in * step;   // (said to be one for all lanes, which it is)
    return (const char*)(uintptr_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32 |
                                    (uint32_t)__builtin_amdgcn_readfirstlane((int)at));
  };
  auto issue1 = [&](int i, const char* ahead) __attribute__((always_inline)) {
    if (i < DMA - 1)
      xgk::glds16_at(ahead, from[i], at_in + 1024 * (W * i + w));
    else
      xgk::glds16_v(p_last, at_in + 1024 * kb_last);
  };
  auto issued = [&]() __attribute__((always_inline)) {   // (all of them: on to the next)
    c_in = min(c_in + 1, nch - 1);
    p_last = c_in == nch - 1 ? p_end : p_last + p_step;
    at_in = at_in == ring + (RING - 1) * SLOT ? ring : at_in + SLOT;
  };
  auto issue = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < DMA; ++i) issue1(i, operands());
    issued();
  };
  for (int c = 0; c < RING - 1; ++c) issue();
  asm volatile("" : "+v"(S));   // (the state is here: its loads are not waited for inside the loop)
  xgk::wait_vmcnt<(RING - 2) * DMA>();
  xgk::raw_barrier();
  // A chunk's operands in registers: read while the chunk before it still adds to the state, in the order they are wanted, so that
  // the first product waits for nothing.
  struct Ops {
    float4 u, r, e, el, k, b, v0;
    float o0[NO], flag;
    T v[4];
  };
  uint32_t at_out = 0;   // the slot of the chunk that is read next
  auto load = [&](Ops& x, int part) __attribute__((always_inline)) {
    const char* at = lds + at_out;
    const float4* p4 = reinterpret_cast<const float4*>(at) + lane;
    const float* pe = reinterpret_cast<const float*>(at + FRAG);
    if (part == 0) x.flag = pe[D], x.u = p4[64 * par], x.e = *reinterpret_cast<const float4*>(pe + 16 * par + 4 * g4);
    if (part == 1) x.el = *reinterpret_cast<const float4*>(pe + 2 * D + 16 * par + 4 * g4), x.r = p4[64 * (MT + par)];
    if (part == 2) {
      const T* pv = reinterpret_cast<const T*>(at + FRAG + 1024) + 16 * ct + l16;
#pragma unroll
      for (int t = 0; t < 4; ++t) x.v[t] = pv[(4 * t + g4) * 32];
      x.v0 = p4[64 * (4 * MT + ct)], x.b = p4[64 * (3 * MT + par)];
    }
    if (part == 3) {
      x.k = p4[64 * (2 * MT + par)];
#pragma unroll
      for (int i = 0; i < NO; ++i) x.o0[i] = reinterpret_cast<const float*>(p4 + 64 * (4 * MT + 2 + ct))[par + MT * i];
      at_out = at_out == (RING - 1) * SLOT ? 0 : at_out + SLOT;
    }
  };
  auto load_all = [&](Ops& x) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) load(x, i);
  };
  // The waves of a column tile hand each other y before a chunk's barrier, and the outputs' sums behind it: those are read, added and
  // stored behind the next one, a part of the rows by each wave. Two buffers, in turn.
  char* const hand = lds + RING * SLOT;
  float o0_was[NO];   // of the chunk before, whose outputs are not stored yet: this wave's part of O,
  int n_was = 0;      // and its rows
  float* ob = o + ((int64_t)q0 * H + h) * D + col + (int64_t)(4 * par + g4) * H * D;   // (the next one to be stored)
  auto sums = [&](const char* at, float* out) __attribute__((always_inline)) {   // the outputs' sums of the column tile's waves
    const float* p = reinterpret_cast<const float*>(at + (W + MT * ct) * 1024) + 64 * par + lane;
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      out[i] = p[64 * MT * i] + p[256 + 64 * MT * i];
      if (MT == 4) out[i] += p[512] + p[768];
    }
  };
  auto store = [&](const float* out) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NO; ++i)
      if (4 * (par + MT * i) + g4 < n_was) ob[(int64_t)(4 * MT * i) * H * D] = out[i] + o0_was[i];
    ob += (int64_t)C * H * D;
  };
  auto chunk = [&](int c, Ops& x, Ops& next) __attribute__((always_inline)) {
    const int n = min(C, qn - C * c);
    char *now = hand + (c & 1) * HAND, *was = hand + (~c & 1) * HAND;
    auto meet = [&]() __attribute__((always_inline)) {   // the next chunk has landed, in every wave
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      xgk::wait_vmcnt<(RING - 2) * DMA>();
      xgk::raw_barrier();
    };
    if (__builtin_amdgcn_readfirstlane(x.flag != 0.f)) {
      const float* p = reinterpret_cast<const float*>(lds + (c % RING) * SLOT);
      __syncthreads();   // (what the chunk before handed over is there, and y has been read)
      if (n_was) {
        float out[NO];
        sums(was, out);
        store(out);
      }
      n_was = 0;
      float* xs = reinterpret_cast<float*>(hand);                // [wave][lane], sums into the state, then the outputs' (below `sums`)
      const float* rr0 = base + c * (step / 4) + 4 * C * D;      // (r lies where V would: only half of that is in LDS)
      const T* pv = reinterpret_cast<const T*>(lds + (c % RING) * SLOT + FRAG + 1024) + 16 * ct + l16;
      float* to = ob - (int64_t)(4 * par + g4) * H * D;
      auto tile_sum = [&](float* xs, float y) __attribute__((always_inline)) {
        y += __shfl_xor(y, 16, 64);
        y += __shfl_xor(y, 32, 64);
        xs[64 * w + lane] = y;
        __syncthreads();
        y += xs[64 * (w ^ 1) + lane];
        return MT == 4 ? y + (xs[64 * (w ^ 2) + lane] + xs[64 * (w ^ 3) + lane]) : y;
      };
      for (int t = 0; t < n; ++t) {
        const float vv = ldf(pv + t * 32);
        const int ch = t * D + 16 * par + 4 * g4;
        float u[4], wr[4], b[4], k[4], rr[4], uS = 0.f, sum = 0.f;
        ld4(p + 2 * C * D + ch, u);
#pragma unroll
        for (int r = 0; r < 4; ++r) uS = fmaf(u[r], S[r], uS);
        uS = tile_sum(xs, uS);
        ld4(p + ch, wr), ld4(p + ch + C * D, b), ld4(p + ch + 3 * C * D, k), ld4(rr0 + ch, rr);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          S[r] = wr[r] * S[r] - b[r] * uS + k[r] * vv;
          sum = fmaf(S[r], rr[r], sum);
        }
        sum = tile_sum(xs + 64 * W, sum);
        if (par == 0 && g4 == 0) to[(int64_t)t * H * D] = sum;
      }
      ob += (int64_t)C * H * D;
      issue();
      meet();
      load_all(next);
      return;
    }
    // one chain over this wave's 16 of the state's rows; between its products the loads of the chunk RING - 1 on, into the slot of the
    // chunk before, which every wave is past, and E S
    f32x4_t yc = {0.f, 0.f, 0.f, 0.f}, oc = yc, ES;
    auto mul = [&](const float4& a, const f32x4_t& y, int q, f32x4_t z) __attribute__((always_inline)) {
      return mfma_f32(q == 0 ? a.x : q == 1 ? a.y : q == 2 ? a.z : a.w, y[q], z);
    };
    const char* ahead = operands();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      yc = mul(x.u, S, q, yc);
#pragma unroll
      for (int i = q * DMA / 4; i < (q + 1) * DMA / 4; ++i) issue1(i, ahead);
    }
    issued();
    ES = f32x4_t{prod_times({x.e.x, x.el.x}, S[0]), prod_times({x.e.y, x.el.y}, S[1]), prod_times({x.e.z, x.el.z}, S[2]),
                 prod_times({x.e.w, x.el.w}, S[3])};
    asm volatile("" : "+v"(ES));   // (formed here, beside the products, and not where it is used)
    float4* ex = reinterpret_cast<float4*>(now) + lane;
    ex[64 * w] = make_float4(yc[0], yc[1], yc[2], yc[3]);
    // the outputs' products with S: one half while y is on its way to the other waves, one while theirs is on its way here
    oc = mul(x.r, S, 0, oc), oc = mul(x.r, S, 1, oc);
    f32x4_t v;
#pragma unroll
    for (int t = 0; t < 4; ++t) v[t] = 4 * t + g4 < n ? ldf(&x.v[t]) : 0.f;
    __builtin_amdgcn_sched_barrier(0);
    meet();
    const float4 y1 = ex[64 * (w ^ 1)];
    float4 y2 = make_float4(0.f, 0.f, 0.f, 0.f), y3 = y2;
    if (MT == 4) y2 = ex[64 * (w ^ 2)], y3 = ex[64 * (w ^ 3)];
    float out[NO];
    sums(was, out);
    __builtin_amdgcn_sched_barrier(0);
    oc = mul(x.r, S, 2, oc), oc = mul(x.r, S, 3, oc);
    // what is taken out, summed up by itself, then the tokens' terms in their order; the next chunk is read meanwhile
    const f32x4_t y = {((yc[0] + y1.x) + (y2.x + y3.x)) + x.v0.x, ((yc[1] + y1.y) + (y2.y + y3.y)) + x.v0.y,
                       ((yc[2] + y1.z) + (y2.z + y3.z)) + x.v0.z, ((yc[3] + y1.w) + (y2.w + y3.w)) + x.v0.w};
    f32x4_t by = mul(x.b, y, 0, f32x4_t{0.f, 0.f, 0.f, 0.f});
    __builtin_amdgcn_sched_barrier(0);
    load(next, 0);
    by = mul(x.b, y, 1, by);
    __builtin_amdgcn_sched_barrier(0);
    load(next, 1);
    by = mul(x.b, y, 2, by);
    __builtin_amdgcn_sched_barrier(0);
    load(next, 2);
    by = mul(x.b, y, 3, by);
    __builtin_amdgcn_sched_barrier(0);
    load(next, 3);
    float* exo = reinterpret_cast<float*>(now) + 256 * (W + w) + lane;   // (row by row: a wave reads one of the four, or two)
    exo[0] = oc[0], exo[64] = oc[1], exo[128] = oc[2], exo[192] = oc[3];
    S = mul(x.k, v, 0, ES + by);
    S = mul(x.k, v, 1, S);
    if (n_was) store(out);
    S = mul(x.k, v, 2, S);
    S = mul(x.k, v, 3, S);
#pragma unroll
    for (int i = 0; i < NO; ++i) o0_was[i] = x.o0[i];
    n_was = n;
  };
  Ops x0, x1;
  load_all(x0);
  for (int c = 0; c < nch; c += 2) {
    chunk(c, x0, x1);
    if (c + 1 < nch) chunk(c + 1, x1, x0);
  }
  xgk::wait_vmcnt<0>();   // (no load may land after the workgroup's LDS is given on)
  __syncthreads();
  if (n_was) {
    float out[NO];
    sums(hand + (~nch & 1) * HAND, out);
    store(out);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) Sg[r * D] = S[r];
}

// ================================================================== host launchers
int64_t delta_chunk_scratch_floats(int T_, int ns, int H, int D) {
  return (int64_t)(T_ / kDcTok + ns + 1) * H * dc_stride(D);
}

int delta_chunk(const void* proj, bool f32, int64_t ld, int off_r, int off_k, int off_v, int off_a, const void* wl, int64_t ld_wl,
                const float* a_bias, const float* w0, float* state, const int32_t* qsl, const int32_t* seq_lens,
                const int32_t* slots, float* o, int ns, int max_q, int H, int D, float* scratch, hipStream_t st) {
  if (ns <= 0 || max_q <= 0) return 0;
  const int nc = (max_q + kDcTok - 1) / kDcTok;
  const int64_t al = f32 ? 4 : 8;   // (v rows come in 16 bytes at a time)
  if ((uintptr_t)proj % 16 || ld % al || off_v % al || (uintptr_t)scratch % 16) return -1;
  if ((D != 32 && D != 64) || H < 1 || !scratch || nc > 65535 || ns > 65535) return -1;
#define XGM_DC(D)                                                                                                          \
  XGM_DISPATCH_T(f32, delta_chunk_prep_kernel<T, D><<<dim3(H, nc, ns), 64, 0, st>>>((const T*)proj, ld, off_r, off_k, off_v, \
                                                                                    off_a, (const T*)wl, ld_wl, a_bias, w0, \
                                                                                    qsl, slots, scratch, H);                \
                 delta_chunk_scan_kernel<T, D><<<dim3(H, ns, D / 32), 8 * D, 0, st>>>(scratch, (const T*)proj, ld, off_v, state, qsl, \
                                                                              seq_lens, slots, o, H);)                       \
  return 0;
  if (D == 32) { XGM_DC(32) }
  XGM_DC(64)
#undef XGM_DC
}

}  // namespace xgm
