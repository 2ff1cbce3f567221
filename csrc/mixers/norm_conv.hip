// What follows a product in a prompt step: the residual sum, its RMS norm and the short convolution over time that the next block
// begins with, in one pass.
//
//   v = alpha x + y1 + bias  (KEEP)  or  x + a1 y1 + a2 y2
//   n = v / sqrt(mean(v^2) + eps) * (off + g)
//   x' <- n (KEEP) or v;  n32, nact <- n;  h <- n + sum_j cw[:, j] (n of the TAPS - 1 rows before, then n)
//
// Bound by memory in large steps (x and y are read and x' and h written once, where the norm's launch and the convolution's write the
// rows and read them again: 201 instead of 301 MB for 8192 x 2048), by a wave's instructions in small ones (some 40 for each of its
// elements). A workgroup takes a strip of a sequence's rows, two at a time, with the next four on their way (a store's answer comes
// before that of the loads behind it, so with one pair on its way a group waits for the stores of the one before): one exchange of
// sums for both, and the rows that the convolution looks back on stay in registers. What it needs of the strip before it forms again,
// TAPS - 1 rows; so x' is another tensor than x. The carried inputs of a sequence are read by its first strip alone. Where there are
// any, it writes them back too, forming the last rows once more if they are another strip's; at a sequence's start the last strip
// writes them.
//
// A strip is 8 rows, with those before it, while that leaves a CU without a second workgroup, else as short as leaves two for each of
// them (one of rows beyond 2048 columns): the weights that a workgroup loads are four rows' bytes. us, KEEP / the other form, the two
// launches in brackets (four sets of rows in turn): 8192 x 2048 in strips of 20 47.8 (57.1) and 63.5 (86.5), 2521 x 2048 in 12 19.2 (21.6)
// and 28.2 (32.3), 8192 x 4096 in 36 89.3 (110) and 118 (175), 2599 x 4096 in 16 34.0 (38.8) and 45.2 (62.7), 512 x 2048 9.5 (9.7) and 10.4
// (12.0), 300 x 4096 12.5 (11.5) and 14.2 (14.6), 96 single tokens of 2048 5.4 (7.1) and 5.8 (8.1), 256 of 4096 10.3 (14.1) and 11.2 (16.8).
// Rows of 2048 up to some 200 (100 8.2 (7.8) and 9.0 (8.7)) and with two branches of 4096 (100 13.1 (11.2)) are slower than in two launches
// on the card, but not in a step, which the host launches: 65 rows Dofivik 1b 1215 (1221), Vizonex 1b 833 (863), 8b 724 (723), 200 rows 1169
// (1190), 913 (930), 968 (974). (The caller keeps the two launches for 65 to 699 rows of 4096 with one branch.)
//
// Threads have one quad of columns up to 1024 columns (with two, half of them idle: 1500 x 1024 10.8 / 12.1 instead of 12.1 / 15.1), and in
// strips of 8 rows up to 2048, where a wave's instructions count (512 x 2048 9.5 / 10.4 instead of 9.5 / 11.4); else two.
#include "glds.h"
#include "mixers_common.h"

namespace xgm {

struct NormConvArgs {
  const float* x;
  const bf16 *y1, *y2;     // [T, W] of row strides ld1, ld2 (KEEP: y1 alone; else y2 may be nullptr)
  int64_t ld1, ld2;
  const float *a1, *a2, *bias, *g, *cw;   // [W] (cw: [W][TAPS]); a1, a2, bias may be nullptr
  float alpha, off, eps;
  float* state;            // [slots][TAPS - 1][W]
  const int32_t *qsl, *seq_lens, *slots;
  float *x_out, *n32;      // n32, nact: may be nullptr
  bf16 *nact, *h;
  int T, W, ns, rows;      // rows: of a strip
};

// a strip's rows of one of the results; what lies outside (of the rows, or a lane's columns of the width) is dropped by the descriptor
struct StripOut {
  void* base;
  uint32_t bytes;
  __device__ __forceinline__ void put(uint32_t off, const float (&f)[4], float) const {
    typedef __attribute__((ext_vector_type(4))) uint32_t u4;
    const u4 v = {__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]), __float_as_uint(f[3])};
    __builtin_amdgcn_raw_buffer_store_b128(v, __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00020000), off, 0, 0);
  }
  __device__ __forceinline__ void put(uint32_t off, const float (&f)[4], bf16) const {
    typedef __attribute__((ext_vector_type(2))) uint32_t u2;
    __builtin_amdgcn_raw_buffer_store_b64(u2{xgk::pack2(f[0], f[1]), xgk::pack2(f[2], f[3])},
                                          __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00020000), off, 0, 0);
  }
};

// NTHR threads of NV quads of columns each: W <= 4 NV NTHR
template <bool KEEP, int TAPS, int NTHR, int NV>
__global__ __launch_bounds__(NTHR, 2) void norm_conv_kernel(const NormConvArgs a) {
  constexpr int NH = TAPS - 1, NW = NTHR / 64, ROWS = 2, DEPTH = 2;
  constexpr int AGAIN = (NH + ROWS - 1) / ROWS;   // groups of the last rows
  // a row's sum is that of 256 threads, each with every 256th quad: of the two rows of a group twice as many threads take one each
  constexpr bool SWAP = NTHR > 256;
  static_assert(!SWAP || NTHR == 256 * ROWS, "rows of a group and threads");
  __shared__ float red[2][ROWS][SWAP ? 4 : NW];
  __shared__ __attribute__((aligned(16))) float held[SWAP ? ROWS : 1][SWAP ? 4 * NV * NTHR : 4];
  const int s = blockIdx.y, W = a.W;
  // the rows behind the last sequence are normed as well, and not convolved
  const int q0 = a.qsl[s], q = (s < a.ns ? a.qsl[s + 1] : a.T) - q0, slot = s < a.ns ? a.slots[s] : -1;
  const int ctx = s < a.ns ? a.seq_lens[s] - q : 0;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int col[NV];
  bool on[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) col[j] = 4 * (threadIdx.x + NTHR * j), on[j] = col[j] < W, col[j] = on[j] ? col[j] : W - 4;
  const float* x0 = a.x + (int64_t)q0 * W;
  const bf16 *y10 = a.y1 + q0 * a.ld1, *y20 = a.y2 ? a.y2 + q0 * a.ld2 : nullptr;
  for (int t0 = blockIdx.x * a.rows; t0 < q; t0 += gridDim.x * a.rows) {
    const int t1 = min(t0 + a.rows, q), first = t0 ? t0 - NH : 0;
    const bool begins = t0 == 0 && slot >= 0 && ctx > 0;
    const bool more = begins && q > a.rows;                            // ... and the last rows for the carried inputs
    const bool keeps = slot >= 0 && (ctx > 0 ? t0 == 0 : t1 == q);
    const int groups = (t1 - first + ROWS - 1) / ROWS + (more ? AGAIN : 0);
    float hist[NH][NV][4], w[NV][4 * TAPS], g[NV][4], s1[NV][4], s2[NV][4];
    Raw4<float> xr[DEPTH][ROWS][NV];
    Raw4<bf16> yr[DEPTH][ROWS][NV], zr[KEEP ? 1 : DEPTH][KEEP ? 1 : ROWS][NV];
    auto row_of = [&](int it) { return more && it >= groups - AGAIN ? q - ROWS * (groups - it) : first + ROWS * it; };
    auto load = [&](int d, int it) __attribute__((always_inline)) {
      const int t = row_of(it);
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        const int r = min(t + i, q - 1);
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          xr[d][i][j].load(x0 + (int64_t)r * W + col[j]);
          yr[d][i][j].load(y10 + r * a.ld1 + col[j]);
          if constexpr (!KEEP) {
            zr[d][i][j].zero();
            if (y20) zr[d][i][j].load(y20 + r * a.ld2 + col[j]);
          }
        }
      }
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (d < groups) load(d, d);
    float* st = a.state + (int64_t)max(slot, 0) * NH * W;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      float f[4];
#pragma unroll
      for (int k = 0; k < TAPS; ++k) {
        ld4(a.cw + (int64_t)col[j] * TAPS + 4 * k, f);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[j][4 * k + e] = f[e];
      }
      ld4(a.g + col[j], g[j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) s1[j][e] = KEEP ? 0.f : 1.f, s2[j][e] = 1.f;
      if (KEEP ? a.bias != nullptr : a.a1 != nullptr) ld4((KEEP ? a.bias : a.a1) + col[j], s1[j]);
      if (!KEEP && a.a2) ld4(a.a2 + col[j], s2[j]);
#pragma unroll
      for (int k = 0; k < NH; ++k) {
#pragma unroll
        for (int e = 0; e < 4; ++e) hist[k][j][e] = 0.f;
        if (begins && ctx - NH + k >= 0) ld4(st + (int64_t)k * W + col[j], hist[k][j]);
      }
    }
    if (keeps && q < NH) {   // carried inputs that stay (a sequence of one strip)
#pragma unroll
      for (int k = 1; k < NH; ++k)
        if (k >= q)
#pragma unroll
          for (int j = 0; j < NV; ++j)
            if (on[j]) st4(st + (int64_t)(k - q) * W + col[j], hist[k][j]);
    }
    const int64_t at0 = (int64_t)(q0 + t0) * W;
    const uint32_t vals = (uint32_t)(t1 - t0) * W;
    const StripOut xo = {a.x_out + at0, 4 * vals}, no = {a.n32 + at0, a.n32 ? 4 * vals : 0}, ao = {a.nact + at0, a.nact ? 2 * vals : 0},
                   ho = {a.h + at0, slot >= 0 ? 2 * vals : 0}, so = {st, (uint32_t)(4 * NH * W)};
    auto add_squares = [](const float (&f)[4], float& sum) __attribute__((always_inline)) {   // (each form as the separate launch rounds it)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum = KEEP ? sum + f[e] * f[e] : fmaf(f[e], f[e], sum);
    };
    auto group = [&](int d, int it) __attribute__((always_inline)) {
      const int t = row_of(it);
      float v[ROWS][NV][4], ss[ROWS];
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        ss[i] = 0.f;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          float f[4], y[4];
          xr[d][i][j].get(f), yr[d][i][j].get(y);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (KEEP) {
              v[i][j][e] = a.alpha * f[e] + y[e] + s1[j][e];
            } else {
              v[i][j][e] = f[e] + s1[j][e] * y[e];
            }
          }
          if constexpr (!KEEP) {
            zr[d][i][j].get(y);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[i][j][e] += s2[j][e] * y[e];
          }
          if constexpr (SWAP) {
            if (on[j]) st4(held[i] + col[j], v[i][j]);
          } else if (on[j]) {
            add_squares(v[i][j], ss[i]);
          }
        }
      }
      if (it + DEPTH < groups) load(d, it + DEPTH);
      if constexpr (SWAP) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        xgk::raw_barrier();
        const int i = wv / 4;
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < NV * ROWS; ++j) {
          const int c = 4 * ((int)(threadIdx.x & 255) + 256 * j);
          float f[4];
          if (c < W) {
            ld4(held[i] + c, f);
            add_squares(f, sum);
          }
        }
        sum = wave_sum(sum);
        if (lane == 0) red[it & 1][i][wv & 3] = sum;
      } else {
#pragma unroll
        for (int i = 0; i < ROWS; ++i) ss[i] = wave_sum(ss[i]);
        if (lane == 0)
#pragma unroll
          for (int i = 0; i < ROWS; ++i) red[it & 1][i][wv] = ss[i];
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      xgk::raw_barrier();   // (two sets of sums in turn: one barrier between those who write a set and those who still read it)
      float rs[ROWS];
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        float sum = 0.f;
#pragma unroll
        for (int k = 0; k < (SWAP ? 4 : NW); ++k) sum += red[it & 1][i][k];
        rs[i] = 1.f / sqrtf(sum / (float)W + a.eps);
      }
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        const float r = rs[i];
        const uint32_t row = (uint32_t)(t + i - t0) * W;   // (where it is in the strip)
        const bool in = t + i >= t0 && t + i < t1 && !(more && it >= groups - AGAIN);
        const bool carry = keeps && t + i < q && t + i >= q - NH && (!more || it >= groups - AGAIN);
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          float n[4], o[4];
          const uint32_t off = in && on[j] ? row + col[j] : 0x20000000u;
#pragma unroll
          for (int e = 0; e < 4; ++e) n[e] = KEEP ? v[i][j][e] * r * (a.off + g[j][e]) : v[i][j][e] * r * g[j][e];
          xo.put(4 * off, KEEP ? n : v[i][j], 0.f);
          if constexpr (!KEEP) {
            if (a.n32) no.put(4 * off, n, 0.f);
            ao.put(2 * off, n, bf16{});
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            o[e] = n[e];
#pragma unroll
            for (int k = 0; k < NH; ++k) o[e] += w[j][TAPS * e + k] * hist[k][j][e];
            o[e] += w[j][TAPS * e + NH] * n[e];
          }
          ho.put(2 * off, o, bf16{});
          if (carry) so.put(on[j] ? 4 * (uint32_t)((t + i - (q - NH)) * W + col[j]) : 0x80000000u, n, 0.f);
#pragma unroll
          for (int k = 0; k < NH; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) hist[k][j][e] = k + 1 < NH ? hist[k + 1 < NH ? k + 1 : k][j][e] : n[e];
        }
      }
    };
    for (int it = 0; it < groups; it += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d)
        if (it + d < groups) group(d, it + d);
    }
    __syncthreads();   // (the sums are written anew)
  }
}

// Strips, with the TAPS - 1 rows before them, of 8 to 36 rows: the shortest that need no more than the workgroups named above, of `cus` CUs.
// Sequences of up to max_q rows; those without a slot and the rows behind the last one are normed and not convolved. Returns -1 for sizes
// or alignments outside this contract.
int norm_conv(const float* x, const void* y1, int64_t ld1, const void* y2, int64_t ld2, const float* a1, const float* a2,
              const float* bias, float alpha, const float* g, float off, float eps, bool keep_norm, float* x_out, float* n32, void* nact,
              const float* cw, int taps, float* state, const int32_t* qsl, const int32_t* seq_lens, const int32_t* slots, void* h,
              int ns, int max_q, int T_, int W, int cus, hipStream_t st) {
  if (T_ <= 0) return 0;
  auto rows_ok = [&](const void* p, int64_t ld) { return ld % 4 == 0 && ld >= W && (uintptr_t)p % 8 == 0; };
  if (W < 4 || W > 4096 || W % 4 || taps < 2 || taps > 4 || ns < 0 || ns > 65534 || max_q < 0 || !y1 || !rows_ok(y1, ld1) ||
      (y2 && !rows_ok(y2, ld2)) || (keep_norm && (y2 || a1 || a2 || n32 || nact)) || (!keep_norm && bias) || !x_out || x_out == x || !h ||
      cus < 1 ||
      (((uintptr_t)x | (uintptr_t)x_out | (uintptr_t)a1 | (uintptr_t)a2 | (uintptr_t)bias | (uintptr_t)g | (uintptr_t)n32 | (uintptr_t)cw |
        (uintptr_t)state) & 15) || (((uintptr_t)nact | (uintptr_t)h) & 7))
    return -1;
  const int64_t fill = W <= 2048 ? 2ll * cus : cus;
  int strip = 8;
  while (strip < 36 && (T_ + strip - taps) / (strip + 1 - taps) > (strip == 8 ? cus : fill)) strip += 4;
  const int rows = strip - (taps - 1);
  const NormConvArgs a = {x, (const bf16*)y1, (const bf16*)y2, ld1, ld2, a1, a2, bias, g, cw, alpha, off, eps, state,
                          qsl, seq_lens, slots, x_out, n32, (bf16*)nact, (bf16*)h, T_, W, ns, rows};
  const int n = max(1, (max_q + rows - 1) / rows);
  const dim3 grid(n < 65535 ? n : 65535, ns + 1);
#define XGM_NC(KEEP, TAPS)                                                                          \
  if (W <= 1024) norm_conv_kernel<KEEP, TAPS, 256, 1><<<grid, 256, 0, st>>>(a);                     \
  else if (W <= 2048 && strip == 8) norm_conv_kernel<KEEP, TAPS, 512, 1><<<grid, 512, 0, st>>>(a);  \
  else if (W <= 2048) norm_conv_kernel<KEEP, TAPS, 256, 2><<<grid, 256, 0, st>>>(a);                \
  else norm_conv_kernel<KEEP, TAPS, 512, 2><<<grid, 512, 0, st>>>(a);
#define XGM_NCT(KEEP)                                                                             \
  if (taps == 4) { XGM_NC(KEEP, 4) } else if (taps == 3) { XGM_NC(KEEP, 3) } else { XGM_NC(KEEP, 2) }
  if (keep_norm) { XGM_NCT(true) } else { XGM_NCT(false) }
#undef XGM_NCT
#undef XGM_NC
  return 0;
}

}  // namespace xgm
