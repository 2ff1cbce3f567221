// One token of a matrix-valued recurrence per sequence (decode steps): the state is read once, updated and written once, and
// everything else that the token needs is formed in the same workgroup.
//
//   gla_step     gated linear recurrence (gla.hip) of one token:  S <- diag(f) S + k v^T,  o = S^T q
//   ssm_step     selective state space (ssm.hip) of one token, the same kernel:  f = exp(-exp(A_log) dt), k = dt B, q = C, v = x,
//                o = S^T q + D x with dt = softplus(dt_raw + dt_bias)
//   delta_step   generalized delta rule of one token, from the fused projection row to the mixer's gated output:
//                  w = exp(-e^(-1/2) sigmoid(W2 tanh(z) + w0)),  a = sigmoid(z_a + a_bias),  u = k / sqrt(|k|^2 + 1e-6)
//                  S <- diag(w) S - (a u)(u^T S) + k v^T,  o = S^T r,  y = o / rms(o) * norm * sigmoid(gate)
//
// Bound by the states' bytes: a workgroup takes one (sequence, head), a thread four neighbouring columns of every RG-th row,
// all of its rows in flight while the row vectors are formed in LDS. The scans that serve longer portions give a lane one
// column (4-byte accesses) and stage tiles of tokens.
//   gla_step, 17 sequences x 32 heads x 64 x 128 (36 MB in and out): 10.1 us against 34.6
//   ssm_step, 64 sequences x 64 heads x 128 x 64 (268 MB): 59.7 us against 93.6 (one sequence of 128 heads: 6.6 against 6.7)
//   delta_step, 64 sequences x 32 heads x 64 x 64 (67 MB): 17.1 us against 40.1 in five launches (tanh 5.0, W2 4.9, row
//   vectors 5.0, scan 20.4, output norm 4.8)
#include "mixers_common.h"

namespace xgm {

struct GlaStepArgs {
  const float *q, *f, *k;            // fp32 [T, H dk]; raw: nullptr
  const void* raw;                   // fused rows: q = silu(raw[off_q ..]), f = l + (1 - l) sigmoid(raw[off_f ..] + f_bias)
  const float *f_bias, *lower, *decay, *bonus;
  const void* v;
  float *state, *o;
  const int32_t *qsl, *seq_lens, *slots;
  int64_t ld_raw, ld_v;
  int off_q, off_f, H, dk, dv;
  const void* dt_raw;                // state space: v = raw rows [x (H dv) | B (G dk) | C (G dk)], a row's dt inputs
  const float *dt_bias, *A_log, *D;
  int64_t ld_dt;
  int G;
};

// NR: rows of a thread; QC = dv / 4 threads side by side, RG = 256 / QC rows at a time
template <typename T, int NR>
__global__ __launch_bounds__(256) void gla_step_kernel(const GlaStepArgs a) {
  __shared__ float fs[256], ks[256], qs[256];
  __shared__ __attribute__((aligned(16))) float part[1024];   // [RG][dv]
  const int h = blockIdx.x, s = blockIdx.y, t = a.qsl[s], slot = a.slots[s];
  if (slot < 0 || a.qsl[s + 1] <= t) return;
  const int QC = a.dv / 4, RG = 256 / QC, rg = threadIdx.x / QC, c = 4 * (threadIdx.x % QC), n = a.H * a.dk;
  const bool on = rg < RG, old = a.seq_lens[s] > 1;
  float* st = a.state + ((int64_t)slot * a.H + h) * a.dk * a.dv + c;
  Raw4<float> sr[NR];
  Raw4<T> vr;
  vr.zero();
  if (on) vr.load((const T*)a.v + (int64_t)t * a.ld_v + h * a.dv + c);
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    sr[i].zero();
    if (on && old && rg + RG * i < a.dk) sr[i].load(st + (int64_t)(rg + RG * i) * a.dv);
  }
  const int d = threadIdx.x;
  float skip = 0.f;
  if (a.dt_raw) {
    const float dt = softplusf(ldf((const T*)a.dt_raw + (int64_t)t * a.ld_dt + h) + a.dt_bias[h]);
    if (d < a.dk) {
      const T* row = (const T*)a.v + (int64_t)t * a.ld_v + a.H * a.dv + h / (a.H / a.G) * a.dk + d;
      fs[d] = expf(-expf(a.A_log[h]) * dt), ks[d] = dt * ldf(row), qs[d] = ldf(row + a.G * a.dk);
    }
    if (d < a.dv) skip = a.D[h] * ldf((const T*)a.v + (int64_t)t * a.ld_v + h * a.dv + d);
  } else if (d < a.dk) {
    if (a.raw) {
      const T* row = (const T*)a.raw + (int64_t)t * a.ld_raw + h * a.dk + d;
      const float l = a.lower[h * a.dk + d];
      const float f = l + (1.f - l) * sigmoidf(ldf(row + a.off_f) + (a.f_bias ? a.f_bias[h * a.dk + d] : 0.f));
      fs[d] = f, ks[d] = 1.f - f, qs[d] = siluf(ldf(row + a.off_q));
    } else {
      const int64_t i = (int64_t)t * n + h * a.dk + d;
      const float f = a.decay ? a.decay[h] : a.f[i];
      fs[d] = f, ks[d] = a.k ? a.k[i] : 1.f - f, qs[d] = a.q[i];
    }
  }
  __syncthreads();
  float v[4], o[4] = {0.f, 0.f, 0.f, 0.f};
  vr.get(v);
  if (on) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int r = rg + RG * i;
      if (r >= a.dk) continue;
      float S[4];
      sr[i].get(S);
      const float f = fs[r], k = ks[r], q = qs[r], u = a.bonus ? a.bonus[h * a.dk + r] : 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float kv = k * v[e];
        if (a.bonus) o[e] += q * (S[e] + u * kv);
        S[e] = a.raw ? fmaf(f, S[e] - v[e], v[e]) : fmaf(f, S[e], kv);
        if (!a.bonus) o[e] += q * S[e];
      }
      st4(st + (int64_t)r * a.dv, S);
    }
    st4(part + rg * a.dv + c, o);
  }
  __syncthreads();
  if (d < a.dv) {
    float x = skip;
    for (int g = 0; g < RG; ++g) x += part[g * a.dv + d];
    a.o[((int64_t)t * a.H + h) * a.dv + d] = x;
  }
}

struct DeltaStepArgs {
  const bf16 *proj, *w2;
  const float *a_bias, *w0, *norm;
  float* state;
  bf16* out;
  const int32_t *qsl, *seq_lens, *slots;
  int64_t ld;
  int off_r, off_k, off_v, off_g, off_a, off_z, lr, H;
  float eps;
};

template <int D>
__global__ __launch_bounds__(256) void delta_step_kernel(const DeltaStepArgs a) {
  constexpr int QC = D / 4, RG = 256 / QC, NR = D / RG, TR = 256 / D;   // TR: threads per row of W2
  static_assert(D >= 32 && D <= 128 && NR * RG == D && TR * D == 256, "delta_step head size");
  __shared__ float ws[D], aus[D], us[D], kk[D], rs[D], th[256], redk[4], redo[4];
  __shared__ __attribute__((aligned(16))) float part[2][4][D];
  const int h = blockIdx.x, s = blockIdx.y, t = a.qsl[s], slot = a.slots[s], tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (slot < 0 || a.qsl[s + 1] <= t) return;
  const int rg = tid / QC, c = 4 * (tid % QC), hd = h * D;
  const bool old = a.seq_lens[s] > 1;
  const bf16* row = a.proj + (int64_t)t * a.ld;
  float* st = a.state + ((int64_t)slot * a.H + h) * D * D + c;
  Raw4<float> sr[NR];
  Raw4<bf16> vr;
  vr.load(row + a.off_v + hd + c);
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    sr[i].zero();
    if (old) sr[i].load(st + (int64_t)(rg + RG * i) * D);
  }
  // row vectors: thread d < D; W2's row d by the TR threads d TR ..
  const int d = tid, wr = tid / TR, wp = tid % TR;
  float kd = 0.f, rd = 0.f, ad = 0.f, gd = 0.f, nd = 0.f;
  if (d < D) {
    kd = bf2f(row[a.off_k + hd + d]), rd = bf2f(row[a.off_r + hd + d]);
    ad = bf2f(row[a.off_a + hd + d]) + a.a_bias[hd + d];
    gd = bf2f(row[a.off_g + hd + d]), nd = a.norm[hd + d];
  }
  const float w0 = a.w0[hd + wr];
  if (tid < a.lr) th[tid] = tanhf(bf2f(row[a.off_z + tid]));
  const float ksq = wave_sum(kd * kd);
  if (lane == 0) redk[wave] = ksq;
  __syncthreads();
  float z = 0.f;
  for (int j = 8 * wp; j < a.lr; j += 8 * TR) {
    const uint4 w = xgk::ld16(a.w2 + (int64_t)(hd + wr) * a.lr + j);
    const uint32_t p[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int e = 0; e < 4; ++e)
      z += __uint_as_float(p[e] << 16) * th[j + 2 * e] + __uint_as_float(p[e] & 0xFFFF0000u) * th[j + 2 * e + 1];
  }
  z = seg_sum(z, TR);
  if (wp == 0) ws[wr] = expf(-0.6065306597126334f * sigmoidf(z + w0));
  if (d < D) {
    const float u = kd / sqrtf(redk[0] + (D > 64 ? redk[1] : 0.f) + 1e-6f);
    us[d] = u, aus[d] = sigmoidf(ad) * u, kk[d] = kd, rs[d] = rd;
  }
  __syncthreads();
  // u^T S: this thread's rows, the wave's row groups by shuffles, the waves in LDS
  float S[NR][4], p[4] = {0.f, 0.f, 0.f, 0.f}, v[4];
  vr.get(v);
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    sr[i].get(S[i]);
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] += us[rg + RG * i] * S[i][e];
  }
#pragma unroll
  for (int o = QC; o < 64; o <<= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] += __shfl_xor(p[e], o, 64);
  if (lane < QC) st4(&part[0][wave][c], p);
  __syncthreads();
  float us4[4] = {0.f, 0.f, 0.f, 0.f}, o4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    float x[4];
    ld4(&part[0][w][c], x);
#pragma unroll
    for (int e = 0; e < 4; ++e) us4[e] += x[e];
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int r = rg + RG * i;
    const float w = ws[r], au = aus[r], k = kk[r], q = rs[r];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      S[i][e] = w * S[i][e] - au * us4[e] + k * v[e];
      o4[e] += q * S[i][e];
    }
    st4(st + (int64_t)r * D, S[i]);
  }
#pragma unroll
  for (int o = QC; o < 64; o <<= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) o4[e] += __shfl_xor(o4[e], o, 64);
  if (lane < QC) st4(&part[1][wave][c], o4);
  __syncthreads();
  const float od = d < D ? part[1][0][d] + part[1][1][d] + part[1][2][d] + part[1][3][d] : 0.f;
  const float osq = wave_sum_products(od, od);
  if (D > 64) {
    if (lane == 0) redo[wave] = osq;
    __syncthreads();
  }
  if (d >= D) return;
  const float ss = D > 64 ? redo[0] + redo[1] : osq;
  a.out[((int64_t)t * a.H + h) * D + d] = f2bf(od / sqrtf(ss / (float)D + a.eps) * nd * sigmoidf(gd));
}

// Rows of a [dk, dv] state that a thread of gla_step_kernel holds, 0 for a state that it does not take: dv a multiple of 4 up to
// 256, dk up to 256, at most 16 rows (a thread's loads in flight). Where dv / 4 does not divide 256 some threads have no
// column, so the area alone does not bound the rows: 128 x 128 takes 16, 88 x 176 would take 18.
int gla_step_rows(int dk, int dv) {
  if (dk < 1 || dk > 256 || dv < 4 || dv > 256 || dv % 4) return 0;
  const int RG = 256 / (dv / 4), nr = (dk + RG - 1) / RG;
  return nr <= 16 ? nr : 0;
}

static int launch_gla_step(const GlaStepArgs& a, bool v_f32, int ns, hipStream_t st) {
  const int nr = gla_step_rows(a.dk, a.dv);
#define XGM_GS(NR) XGM_DISPATCH_T(v_f32, gla_step_kernel<T, NR><<<dim3(a.H, ns), 256, 0, st>>>(a);)
  if (nr <= 2) { XGM_GS(2) } else if (nr <= 4) { XGM_GS(4) } else if (nr <= 8) { XGM_GS(8) } else { XGM_GS(16) }
#undef XGM_GS
  return 0;
}

// One token per sequence (max_q == 1). Return -1 for states outside gla_step_rows and for rows or states that are not aligned.
int gla_step(const float* q, const float* f, const float* k, const void* raw, int64_t ld_raw, int off_q, int off_f,
             const float* f_bias, const float* lower, const void* v, bool v_f32, int64_t ld_v, float* state, const int32_t* qsl,
             const int32_t* seq_lens, const int32_t* slots, float* o, int ns, int H, int dk, int dv, const float* decay,
             const float* bonus, hipStream_t st) {
  if (ns <= 0) return 0;
  if (H < 1 || !gla_step_rows(dk, dv) || ns > 65535 || ld_v % 4 ||
      (uintptr_t)v % (v_f32 ? 16 : 8) || (uintptr_t)state % 16 || (raw ? (!lower || decay || bonus) : (!q || (!f && !decay))) ||
      ((decay || bonus) && !k))
    return -1;
  const GlaStepArgs a = {q, f, k, raw, f_bias, lower, decay, bonus, v, state, o, qsl, seq_lens, slots, ld_raw, ld_v,
                         off_q, off_f, H, dk, dv, nullptr, nullptr, nullptr, nullptr, 0, 1};
  return launch_gla_step(a, v_f32, ns, st);
}

int ssm_step(const void* xbc, bool f32, int64_t ld_x, const void* dt_raw, int64_t ld_dt, const float* dt_bias, const float* A_log,
             const float* D, float* state, const int32_t* qsl, const int32_t* seq_lens, const int32_t* slots, float* y, int ns,
             int H, int G, int N, int P, hipStream_t st) {
  if (ns <= 0) return 0;
  if (H < 1 || G < 1 || H % G || !gla_step_rows(N, P) || ns > 65535 || ld_x % 4 ||
      (uintptr_t)xbc % (f32 ? 16 : 8) || (uintptr_t)state % 16 || !dt_raw)
    return -1;
  GlaStepArgs a = {};
  a.v = xbc, a.ld_v = ld_x, a.state = state, a.o = y, a.qsl = qsl, a.seq_lens = seq_lens, a.slots = slots, a.H = H, a.dk = N, a.dv = P;
  a.dt_raw = dt_raw, a.ld_dt = ld_dt, a.dt_bias = dt_bias, a.A_log = A_log, a.D = D, a.G = G;
  return launch_gla_step(a, f32, ns, st);
}

// One token per sequence, bf16. D 32, 64 or 128, lr (rank of W2 [H D, lr]) a multiple of 8 up to 256; columns of the projection
// row: off_r, off_k, off_v, off_g (gate), off_a, off_z (lr low-rank entries).
int delta_step(const void* proj, int64_t ld, int off_r, int off_k, int off_v, int off_g, int off_a, int off_z, int lr, const void* w2,
               const float* a_bias, const float* w0, const float* norm, float eps, float* state, const int32_t* qsl,
               const int32_t* seq_lens, const int32_t* slots, void* out, int ns, int H, int D, hipStream_t st) {
  if (ns <= 0) return 0;
  if (H < 1 || ns > 65535 || lr < 8 || lr > 256 || lr % 8 || (uintptr_t)w2 % 16 || (uintptr_t)proj % 8 || ld % 4 || off_v % 4 ||
      (uintptr_t)state % 16)
    return -1;
  const DeltaStepArgs a = {(const bf16*)proj, (const bf16*)w2, a_bias, w0, norm, state, (bf16*)out, qsl, seq_lens, slots, ld,
                           off_r, off_k, off_v, off_g, off_a, off_z, lr, H, eps};
  if (D == 32) delta_step_kernel<32><<<dim3(H, ns), 256, 0, st>>>(a);
  else if (D == 64) delta_step_kernel<64><<<dim3(H, ns), 256, 0, st>>>(a);
  else if (D == 128) delta_step_kernel<128><<<dim3(H, ns), 256, 0, st>>>(a);
  else return -1;
  return 0;
}

}  // namespace xgm
