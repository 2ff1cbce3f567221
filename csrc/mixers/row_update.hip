// What follows a product in a step of single tokens, for rows of up to 8192 columns: the residual sum, its RMS norm and the short
// convolution over time that the next block begins with, in one launch.
//
//   v = alpha x + a1 y1 + a2 (y2 + y3) + bias        y1, y2: bf16 rows, or fp32 slabs of a product in parts that are added here
//   r = v / sqrt(mean(v^2) + eps) * (off + g)
//   x <- r (keep_norm) or v;  n32, nact <- r;  h <- r + sum_j cw[:, j] (inputs carried in the slot, then r), the slot moves on
//
// A workgroup per row; everything the row needs is on its way before the first use. The launches that it replaces take about
// 4.7 us each whatever they do; the rows are 8 to 24 KB of reads per slab. 64 rows of 2048 (8 slabs): 6.1 us against 4.8 + 4.8
// and 4 us less in the product; one row of 4096 (two products of 4 slabs): 6.5 us against 7.7 + 4.6.
#include "mixers_common.h"

namespace xgm {

struct RowSource {      // n = 0: bf16 rows of stride ld; n > 0: n fp32 slabs of rows of stride ld, `slab` apart; p nullptr: none
  const void* p;
  int64_t ld, slab;
  int n;
};

struct RowUpdateArgs {
  float* x;
  RowSource y1, y2;
  const float *y3, *a1, *a2, *bias, *g, *cw;
  float alpha, off, eps;
  float* state;           // [slots][TAPS - 1][W]
  const int32_t *token_seq, *seq_lens, *slots;
  float* n32;
  bf16 *nact, *h;
  int W, keep_norm;
};

__device__ __forceinline__ void row_source(const RowSource& y, int t, int c, float (&v)[4]) {
  if (y.n == 0) {
    ld4((const bf16*)y.p + (int64_t)t * y.ld + c, v);
    return;
  }
  const float* p = (const float*)y.p + (int64_t)t * y.ld + c;
  ld4(p, v);
  add_slabs(p, y.slab, y.n, v);
}

template <int NV, int TAPS>
__global__ __launch_bounds__(512) void row_update_kernel(const RowUpdateArgs a) {
  constexpr int NH = TAPS - 1;
  __shared__ float red[8];
  const int t = blockIdx.x;
  const int s = a.h ? a.token_seq[t] : -1, slot = s >= 0 ? a.slots[s] : -1, ctx = slot >= 0 ? a.seq_lens[s] - 1 : 0;
  float v[NV][4], g[NV][4];
  Raw4<float> old[NV][NH > 0 ? NH : 1], wt[NV][TAPS];
  float* st = a.state + (int64_t)max(slot, 0) * NH * a.W;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = 4 * (threadIdx.x + 512 * j);
    if (c >= a.W) continue;
    if (slot >= 0) {
#pragma unroll
      for (int k = 0; k < TAPS; ++k) wt[j][k].load(a.cw + (int64_t)c * TAPS + 4 * k);
#pragma unroll
      for (int k = 0; k < NH; ++k) {
        old[j][k].zero();
        if (ctx - NH + k >= 0) old[j][k].load(st + (int64_t)k * a.W + c);
      }
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = 4 * (threadIdx.x + 512 * j);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[j][e] = g[j][e] = 0.f;
    if (c >= a.W) continue;
    float x[4], y[4] = {0.f, 0.f, 0.f, 0.f}, z[4] = {0.f, 0.f, 0.f, 0.f}, z3[4] = {0.f, 0.f, 0.f, 0.f};
    float s1[4] = {1.f, 1.f, 1.f, 1.f}, s2[4] = {1.f, 1.f, 1.f, 1.f}, b[4] = {0.f, 0.f, 0.f, 0.f};
    ld4(a.x + (int64_t)t * a.W + c, x);
    ld4(a.g + c, g[j]);
    if (a.a1) ld4(a.a1 + c, s1);
    if (a.a2) ld4(a.a2 + c, s2);
    if (a.bias) ld4(a.bias + c, b);
    if (a.y3) ld4(a.y3 + (int64_t)t * a.W + c, z3);
    if (a.y1.p) row_source(a.y1, t, c, y);
    if (a.y2.p) row_source(a.y2, t, c, z);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[j][e] = a.alpha * x[e] + s1[e] * y[e] + s2[e] * (z[e] + z3[e]) + b[e];
      ss += v[j][e] * v[j][e];
    }
  }
  const float r = 1.f / sqrtf(block_sum(ss, red) / (float)a.W + a.eps);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = 4 * (threadIdx.x + 512 * j);
    if (c >= a.W) continue;
    float n[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) n[e] = v[j][e] * r * (a.off + g[j][e]);
    const int64_t at = (int64_t)t * a.W + c;
    st4(a.x + at, a.keep_norm ? n : v[j]);
    if (a.n32) st4(a.n32 + at, n);
    if (a.nact) st4(a.nact + at, n);
    if (slot < 0) continue;
    float w[4 * TAPS], hist[TAPS][4], o[4];
#pragma unroll
    for (int k = 0; k < TAPS; ++k) {
      float f[4];
      wt[j][k].get(f);
#pragma unroll
      for (int e = 0; e < 4; ++e) w[4 * k + e] = f[e];
      if (k < NH) old[j][k < NH ? k : 0].get(hist[k]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      hist[NH][e] = n[e], o[e] = n[e];
#pragma unroll
      for (int k = 0; k < TAPS; ++k) o[e] += w[TAPS * e + k] * hist[k][e];
    }
#pragma unroll
    for (int k = 0; k < NH; ++k) st4(st + (int64_t)k * a.W + c, hist[k + 1]);
    st4(a.h + at, o);
  }
}

// Row t is the single token of sequence token_seq[t] (no two rows share a sequence); h, with conv weights cw [W][taps] of 2 to 4
// taps, is not written for rows without a slot. Returns -1 for sizes or alignments outside this contract.
int row_update(float* x, const void* y1, int64_t ld1, int64_t slab1, int n1, const void* y2, int64_t ld2, int64_t slab2, int n2,
               const float* y3, const float* a1, const float* a2, const float* bias, float alpha, const float* g, float off,
               float eps, bool keep_norm, float* n32, void* nact, const float* cw, int taps, float* state,
               const int32_t* token_seq, const int32_t* seq_lens, const int32_t* slots, void* h, int T_, int W,
               hipStream_t st) {
  if (T_ <= 0) return 0;
  auto rows_ok = [](const void* p, int64_t ld, int64_t slab, int n) {
    return !p || (n >= 0 && ld % 4 == 0 && slab % 4 == 0 && (uintptr_t)p % (n ? 16 : 8) == 0);
  };
  if (W < 4 || W > 8192 || W % 4 || !rows_ok(y1, ld1, slab1, n1) || !rows_ok(y2, ld2, slab2, n2) || (y3 && (uintptr_t)y3 % 16) ||
      (h && (taps < 2 || taps > 4 || !cw || !state || !token_seq)) ||
      (((uintptr_t)x | (uintptr_t)a1 | (uintptr_t)a2 | (uintptr_t)bias | (uintptr_t)g | (uintptr_t)n32 | (uintptr_t)cw |
        (uintptr_t)state) & 15) || (((uintptr_t)nact | (uintptr_t)h) & 7))
    return -1;
  const RowUpdateArgs a = {x, {y1, ld1, slab1, n1}, {y2, ld2, slab2, n2}, y3, a1, a2, bias, g, cw, alpha, off, eps, state,
                           token_seq, seq_lens, slots, n32, (bf16*)nact, (bf16*)h, W, keep_norm ? 1 : 0};
#define XGM_RU(TAPS)                                                         \
  if (W <= 2048) row_update_kernel<1, TAPS><<<T_, 512, 0, st>>>(a);          \
  else if (W <= 4096) row_update_kernel<2, TAPS><<<T_, 512, 0, st>>>(a);     \
  else row_update_kernel<4, TAPS><<<T_, 512, 0, st>>>(a);
  if (!h || taps == 4) {
    XGM_RU(4)
  } else if (taps == 3) {
    XGM_RU(3)
  } else {
    XGM_RU(2)
  }
#undef XGM_RU
  return 0;
}

}  // namespace xgm
