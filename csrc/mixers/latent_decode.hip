// Latent attention of a step of single tokens (bf16; one token per sequence):
//
//   latent_query_kernel    the heads' W_uk folded into their queries: qabs[h][t] = q[t][h] . W_uk[h]
//   latent_decode_kernel   attention over the cached latents for 32 heads of one sequence and one share of its window
//   latent_out_kernel      the shares of a (token, head) merged, gated, and expanded by the head's W_uv into the output row
//
// All heads of a sequence read the same cached rows [latent (R) | rotated key (rd)], so a step cannot do without one pass over
// the windows' rows; the products are small beside it. A workgroup takes 32 heads (two tiles of 16) and walks its share 64
// keys at a time: two waves per tile of heads, 32 keys each, with their own running maximum and sum, merged in LDS at the end.
// Rows come in by LDS-DMA into two slots, the next 64 keys on their way while these are used; the share's page table is read
// into LDS first, so no address waits for memory inside the loop. A slot is 4 groups of 16 rows x R + rd columns, cut into
// blocks of 16 rows x 32 columns (1 KB, one DMA instruction) whose 16-byte granules are permuted by row / 4: the fragment
// reads (S^T = K Q^T) and the transposed ones (O^T += V^T P^T) both spread over all banks.
//
// 64 sequences of 1024 keys, 32 heads, R = 256, rd = 32: 16.0 us (37.7 MB of rows) and 7.8 us against 30.6 and, for merge,
// expansion product and transpose in three launches, 25.7. The kernel before had one 64-key tile to a workgroup (16 shares),
// nothing in flight behind it, 33 MB of fp32 shares written and read back, and half of its waves without heads. (R = 512, rd = 64: 29.8
// where every tile rescaled its 128 accumulators, 27.5 where only those that raise the maximum do. Four slots, or two tiles at a
// time on eight waves: no faster, one tile takes 7.5 us, most of it one memory latency behind the other.)
#include "attention_common.h"
#include "glds.h"

namespace xgm {
using xgk::as_frag;
using xgk::bf16x8_t;
using xgk::f32x4_t;
using xgk::mfma16x16x32;

constexpr int kLatentPages = 2048;   // page table entries of a share in LDS

// qabs[h][t][r] = sum_d q[t][h][d] uk[h][d][r], transposed: a wave has 16 columns r of a head for up to 16 MT tokens, dn = 32 NK. Latency
// alone (64 rows, 32 heads, dn = 64, R = 256: 2 MB in all), so no LDS and no exchange: every load is on its way at once, W_uk's entry by
// entry, as its rows run along r, 16 lanes to 32 bytes.
// The library's batched product took 7.7 us there, a step of 64 (four of them) 701 us with it and 685 with this.
template <int NK, int MT>
__global__ __launch_bounds__(256) void latent_query_kernel(const bf16* __restrict__ q, int dq, const bf16* __restrict__ uk,
                                                           bf16* __restrict__ qabs, int T, int H, int R) {
  const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4, h = blockIdx.y, t0 = 16 * MT * blockIdx.z;
  const int r0 = 64 * blockIdx.x + 16 * (threadIdx.x >> 6);   // (R is a multiple of 64)
  const bf16* w = uk + (int64_t)(h * 32 * NK + 8 * g) * R + r0 + li;
  bf16 wr[NK][8];
  uint4 x[MT][NK];
#pragma unroll
  for (int k = 0; k < NK; ++k)
#pragma unroll
    for (int e = 0; e < 8; ++e) wr[k][e] = w[(int64_t)(32 * k + e) * R];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int k = 0; k < NK; ++k)
      x[m][k] = xgk::ld16(q + ((int64_t)min(t0 + 16 * m + li, T - 1) * H + h) * dq + 32 * k + 8 * g);
  bf16x8_t wf[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k)
#pragma unroll
    for (int e = 0; e < 8; ++e) wf[k][e] = (short)wr[k][e];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NK; ++k) acc = mfma16x16x32(wf[k], as_frag(x[m][k]), acc);
    const int t = t0 + 16 * m + li;   // lane: columns 4 g .. of token li
    if (t < T) *reinterpret_cast<uint2*>(qabs + ((int64_t)h * T + t) * R + r0 + 4 * g) =
        make_uint2(xgk::pack2(acc[0], acc[1]), xgk::pack2(acc[2], acc[3]));
  }
}

struct LatentDecodeArgs {
  const bf16 *qabs, *q, *cache;
  const int32_t *block_tables, *qsl, *seq_lens, *slots;
  const float* rot;
  float *part_o, *part_ml;   // [share][H][T][R], [share][H][T][2]: unnormalised sums, (maximum, sum of weights)
  int dq, dn, bt_width, bs, rot_dims, T, H, window, shares;
  float scale;
};

// maximum over the four lanes that share a column
__device__ __forceinline__ float column_max(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
#endif
  return x;
}

template <int NR, int ND>
__global__ __launch_bounds__(256, 1) void latent_decode_kernel(const LatentDecodeArgs a) {
  constexpr int R = 32 * NR, DK = 32 * (NR + ND), NKK = NR + ND, NMT = 2 * NR, SLOT = 4 * NKK * 1024;
  static_assert(2 * SLOT >= (32 * R + 128) * 4 && 2 * SLOT + kLatentPages * 4 <= 160 * 1024, "latent_decode LDS");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * SLOT + kLatentPages * 4];
  int32_t* pages = reinterpret_cast<int32_t*>(lds + 2 * SLOT);
  const int s = blockIdx.y, share = blockIdx.x, lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ht = wave & 1, kg = wave >> 1;
  const int head = blockIdx.z * 32 + 16 * ht + li, t = a.qsl[s];   // the sequence's row (sequences without a token have none)
  if (a.slots[s] < 0 || a.qsl[s + 1] - t <= 0) return;
  const int pos = a.seq_lens[s] - 1, first = max(0, pos - a.window + 1);
  const int tiles_all = (pos - first + 64) / 64, per = (tiles_all + a.shares - 1) / a.shares;
  const int k0 = first + 64 * per * share, k1 = min(pos, k0 + 64 * per - 1);   // this share's keys [k0, k1]
  const int64_t row = ((int64_t)share * a.H + head) * a.T + t;
  if (k0 > pos) {   // an empty share
    if (kg == 0 && g == 0 && head < a.H) a.part_ml[2 * row] = -INFINITY, a.part_ml[2 * row + 1] = 0.f;
    return;
  }
  const int32_t* bt = a.block_tables + (int64_t)s * a.bt_width;
  const int p0 = k0 / a.bs, np = k1 / a.bs - p0 + 1;
  for (int i = threadIdx.x; i < np; i += 256) pages[i] = bt[p0 + i];
  __syncthreads();
  const int ntile = (k1 - k0 + 64) / 64;
  // rows past the share read its last row (scored -inf below)
  auto issue = [&](int c) {
    const int r16 = lane >> 2, k = min(k0 + 64 * min(c, ntile - 1) + 16 * wave + r16, k1);
    const bf16* src = a.cache + ((int64_t)pages[k / a.bs - p0] * a.bs + k % a.bs) * DK + 8 * ((lane & 3) ^ (r16 >> 2));
    uint8_t* dst = lds + (c & 1) * SLOT + wave * NKK * 1024;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) xgk::glds16(src + 32 * kk, dst + kk * 1024);
  };
  issue(0);
  // the head's query as B fragments: [W_uk^T q (R) | rotated q (rd)], 8 columns at 32 kk + 8 g
  const int hq = min(head, a.H - 1), half = a.rot_dims >> 1;
  uint4 qr[NKK];
#pragma unroll
  for (int kk = 0; kk < NR; ++kk) qr[kk] = xgk::ld16(a.qabs + ((int64_t)hq * a.T + t) * R + 32 * kk + 8 * g);
#pragma unroll
  for (int kk = 0; kk < ND; ++kk) {
    const int i0 = 32 * kk + 8 * g;
    const bf16* src = a.q + ((int64_t)t * a.H + hq) * a.dq + a.dn + i0;
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const float u = bf2f(src[e]), v = bf2f(src[e + 1]);
      f[e] = u, f[e + 1] = v;
      if (i0 + e < a.rot_dims) {
        const float* cs = a.rot + ((int64_t)pos * half + ((i0 + e) >> 1)) * 2;
        f[e] = u * cs[0] - v * cs[1];
        f[e + 1] = v * cs[0] + u * cs[1];
      }
    }
    qr[NR + kk] = xgk::pack8(f);
  }
  f32x4_t o[NMT];
#pragma unroll
  for (int mt = 0; mt < NMT; ++mt) o[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;   // the column's reference; this lane's share of its sum
  // the queries have to be here before the second tile is asked for: the wait for them would cover it too
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) asm volatile("" : "+v"(qr[kk].x), "+v"(qr[kk].y), "+v"(qr[kk].z), "+v"(qr[kk].w));
  const int koff = li * 64 + ((g ^ (li >> 2)) << 4);                 // this lane's granule of a K fragment
  const int qq = li >> 2, pp = li & 3;
  const int voff0 = (4 * g + qq) * 64 + (((pp >> 1) ^ g) << 4) + (pp & 1) * 8;         // columns 16 mt + 4 pp, mt even
  const int voff1 = (4 * g + qq) * 64 + (((2 + (pp >> 1)) ^ g) << 4) + (pp & 1) * 8;   // ... odd
  for (int c = 0; c < ntile; ++c) {
    issue(c + 1);
    xgk::wait_vmcnt<NKK>();
    xgk::raw_barrier();
    const uint8_t* t0 = lds + (c & 1) * SLOT + 2 * kg * NKK * 1024;
    f32x4_t sc[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      sc[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk)
        sc[n] = mfma16x16x32(as_frag(*reinterpret_cast<const uint4*>(t0 + (n * NKK + kk) * 1024 + koff)), as_frag(qr[kk]), sc[n]);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = k0 + 64 * c + 32 * kg + 16 * n + 4 * g + r;
        sc[n][r] = k > k1 ? -INFINITY : sc[n][r] * a.scale;
        mx = fmaxf(mx, sc[n][r]);
      }
    mx = column_max(mx);
    // (no column of the wave has a new maximum: nothing to rescale. The reference is the maximum itself: the largest weight, 1, is exact in bf16)
    if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {
      const float mn = fmaxf(m, mx), alpha = m == -INFINITY ? 0.f : __expf(m - mn);
      l *= alpha, m = mn;
#pragma unroll
      for (int mt = 0; mt < NMT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[mt][r] *= alpha;
    }
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sc[n][r] = m == -INFINITY ? 0.f : __expf(sc[n][r] - m);
        l += sc[n][r];
      }
    uint4 pb;
    pb.x = xgk::pack2(sc[0][0], sc[0][1]), pb.y = xgk::pack2(sc[0][2], sc[0][3]);
    pb.z = xgk::pack2(sc[1][0], sc[1][1]), pb.w = xgk::pack2(sc[1][2], sc[1][3]);
#pragma unroll
    for (int mt = 0; mt < NMT; ++mt) {
      // keys in the order that the score accumulators hold them: 4 g + r of both 16-key groups
      const uint8_t* v = t0 + (mt >> 1) * 1024 + (mt & 1 ? voff1 : voff0);
      const xgk::bf16x4_t a0 = xgk::lds_read_tr16(reinterpret_cast<const uint16_t*>(v));
      const xgk::bf16x4_t a1 = xgk::lds_read_tr16(reinterpret_cast<const uint16_t*>(v + NKK * 1024));
      const xgk::bf16x8_t vf = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
      o[mt] = mfma16x16x32(vf, as_frag(pb), o[mt]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    xgk::raw_barrier();
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  xgk::wait_vmcnt<0>();
  __syncthreads();   // (a slower wave's last rows are still on their way into a slot)
  // the second half of the keys joins the first
  float* mo = reinterpret_cast<float*>(lds);   // [2][NMT][64][4], then [2][16][2]
  float* mm = mo + 32 * R;
  if (kg == 1) {
#pragma unroll
    for (int mt = 0; mt < NMT; ++mt) *reinterpret_cast<f32x4_t*>(mo + ((ht * NMT + mt) * 64 + lane) * 4) = o[mt];
    if (g == 0) mm[(ht * 16 + li) * 2] = m, mm[(ht * 16 + li) * 2 + 1] = l;
  }
  __syncthreads();
  if (kg == 1 || head >= a.H) return;
  const float m2 = mm[(ht * 16 + li) * 2], l2 = mm[(ht * 16 + li) * 2 + 1];
  const float M = fmaxf(m, m2);   // (the first half holds a key: finite unless a score is not)
  const float e1 = m == -INFINITY ? 0.f : __expf(m - M), e2 = m2 == -INFINITY ? 0.f : __expf(m2 - M);
  if (g == 0) a.part_ml[2 * row] = M, a.part_ml[2 * row + 1] = l * e1 + l2 * e2;
#pragma unroll
  for (int mt = 0; mt < NMT; ++mt) {
    const f32x4_t u = *reinterpret_cast<const f32x4_t*>(mo + ((ht * NMT + mt) * 64 + lane) * 4);
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = o[mt][r] * e1 + u[r] * e2;
    st4(a.part_o + row * R + 16 * mt + 4 * g, v);
  }
}

// Workgroup = (head, TOK tokens): out[t][h dv + j] = sum_d lat[t][d] W_uv[h dv + j][d], lat the merged and gated latent sum, rounded
// to bf16. The columns of a 16-token product beyond TOK repeat them (more workgroups; the products cost nothing here): so few tokens
// that about a workgroup per compute unit runs (32 heads, 8 tokens each / as here, us: 9 tokens, 16 shares, R = 512 26.9 / 8.8, one token,
// 10 shares 12.2 / 7.0, 17 tokens, 15 shares, R = 256 10.4 / 7.1).
template <int NR, int TOK>
__global__ __launch_bounds__(256) void latent_out_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                         const bf16* __restrict__ gate, int64_t gate_stride,
                                                         const bf16* __restrict__ uv, const int32_t* __restrict__ slots,
                                                         const int32_t* __restrict__ qsl,
                                                         const int32_t* __restrict__ token_seq, bf16* __restrict__ out, int T,
                                                         int H, int dv, int shares) {
  constexpr int R = 32 * NR, LD = R + 8;
  __shared__ __attribute__((aligned(16))) uint16_t lat[TOK * LD];
  __shared__ float wt[TOK][64];   // a share's weight: e^(m_s - M) gate / L (shares <= 64)
  const int h = blockIdx.x, t0 = blockIdx.y * TOK, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, g = lane >> 4;
  const bool has = 16 * wave < dv;
  uint4 w[NR];   // this wave's first 16 rows of W_uv: on their way while the shares are merged
#pragma unroll
  for (int kk = 0; kk < NR; ++kk)
    w[kk] = xgk::ld16(uv + ((int64_t)h * dv + (has ? 16 * wave : 0) + li) * R + 32 * kk + 8 * g);
#pragma unroll
  for (int i = wave; i < TOK; i += 4) {
    const int t = t0 + i;
    float x = 0.f;
    const int s = t < T ? token_seq[t] : -1;
    if (s >= 0 && s < T && slots[s] >= 0 && qsl[s] == t && qsl[s + 1] > t) {   // (T sequences)
      const int64_t r = 2 * (((int64_t)min(lane, shares - 1) * H + h) * T + t);
      const float m = lane < shares ? part_ml[r] : -INFINITY, l = part_ml[r + 1];
      const float M = wave_max(m), e = m == -INFINITY ? 0.f : __expf(m - M);
      const float L = wave_sum(m == -INFINITY ? 0.f : e * l);
      x = e * (sigmoidf(bf2f(gate[(int64_t)t * gate_stride + h])) * (L > 0.f ? 1.f / L : 0.f));
      // (a maximum or sum that is not a number makes the row so, as the softmax does)
      if (!(L > 0.f) && L != 0.f) x = L;
    }
    wt[i][lane] = x;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < TOK * R / 4; i += 256) {
    const int k = i / (R / 4), d = 4 * (i % (R / 4)), t = min(t0 + k, T - 1);
    const float* src = part_o + ((int64_t)h * T + t) * R + d;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int sh = 0; sh < shares; ++sh) {
      const float c = wt[k][sh];
      float u[4];
      ld4(src + (int64_t)sh * H * T * R, u);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += c == 0.f ? 0.f : c * u[e];   // (an empty share's sums are not written)
    }
    st4(lat + k * LD + d, v);
  }
  __syncthreads();
  uint4 b[NR];
#pragma unroll
  for (int kk = 0; kk < NR; ++kk) b[kk] = *reinterpret_cast<const uint4*>(lat + (li & (TOK - 1)) * LD + 32 * kk + 8 * g);
  for (int j = wave; 16 * j < dv; j += 4) {
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < NR; ++kk) acc = mfma16x16x32(as_frag(w[kk]), as_frag(b[kk]), acc);
    if (li < TOK && t0 + li < T) {
      const float v[4] = {acc[0], acc[1], acc[2], acc[3]};
      st4(out + ((int64_t)(t0 + li) * H + h) * dv + 16 * j + 4 * g, v);
    }
    if (16 * (j + 4) < dv) {
#pragma unroll
      for (int kk = 0; kk < NR; ++kk) w[kk] = xgk::ld16(uv + ((int64_t)h * dv + 16 * (j + 4) + li) * R + 32 * kk + 8 * g);
    }
  }
}

// At most one token per sequence, as many rows as sequences (rows behind the last token are zero). Returns 0, or -1 for sizes that it does not take: R 64, 128, 256 or 512, rd 32 or
// 64, dv a multiple of 16, 1 to 64 shares, a share's keys within kLatentPages pages.
int latent_decode(const void* qabs, const void* q, int dq, int dn, const void* gate, int64_t gate_stride, const void* cache,
                  const int32_t* bt, int bt_width, int bs, const int32_t* qsl, const int32_t* seq_lens, const int32_t* slots,
                  const int32_t* token_seq, const float* rot, int rot_dims, const void* uv, void* out, int T, int H, int R, int dv, int window, float scale,
                  int shares, float* part_o, float* part_ml, hipStream_t st) {
  if (T <= 0) return 0;
  const int rd = dq - dn, nr = R / 32;
  const int64_t keys = std::min<int64_t>(window, (int64_t)bt_width * bs), tiles = (keys + 63) / 64;
  if (R % 32 || (rd != 32 && rd != 64) || dv < 16 || dv % 16 || shares < 1 || shares > 64 || H < 1 || bs < 1 || window < 1 ||
      rot_dims % 2 || rot_dims > rd || ((tiles + shares - 1) / shares * 64 + bs - 1) / bs + 1 > kLatentPages || T > 65535 ||
      (((uintptr_t)qabs | (uintptr_t)cache | (uintptr_t)uv | (uintptr_t)part_o) & 15) || ((uintptr_t)out & 7))
    return -1;
  const LatentDecodeArgs a = {(const bf16*)qabs, (const bf16*)q, (const bf16*)cache, bt, qsl, seq_lens, slots, rot, part_o, part_ml,
                              dq, dn, bt_width, bs, rot_dims, T, H, window, shares, scale};
  const dim3 grid(shares, T, (H + 31) / 32);
#define XGM_LO(NR, TOK)                                                                                                     \
  {                                                                                                                         \
    latent_out_kernel<NR, TOK><<<dim3(H, (T + TOK - 1) / TOK), 256, 0, st>>>(part_o, part_ml, (const bf16*)gate, gate_stride, \
                                                                             (const bf16*)uv, slots, qsl, token_seq,        \
                                                                             (bf16*)out, T, H, dv, shares);                 \
  }
#define XGM_LD(NR)                                                                                                          \
  if (nr == NR) {                                                                                                           \
    if (rd == 32) latent_decode_kernel<NR, 1><<<grid, 256, 0, st>>>(a);                                                     \
    else latent_decode_kernel<NR, 2><<<grid, 256, 0, st>>>(a);                                                              \
    if (H * T > 1024) XGM_LO(NR, 8) else if (H * T > 512) XGM_LO(NR, 4) else if (H * T > 256) XGM_LO(NR, 2) else XGM_LO(NR, 1) \
    return 0;                                                                                                               \
  }
  XGM_LD(2)
  XGM_LD(4)
  XGM_LD(8)
  XGM_LD(16)
#undef XGM_LD
#undef XGM_LO
  return -1;
}

// q: [T, H, dq] rows whose first dn entries are the unrotated ones. Returns -1 for sizes or alignments outside this contract.
int latent_query(const void* q, int dq, int dn, const void* uk, void* qabs, int T, int H, int R, hipStream_t st) {
  if (T < 1 || H < 1 || H > 65535 || dq < dn || dq % 8 || (dn != 32 && dn != 64 && dn != 128) || R < 64 || R % 64 || T > 65535 ||
      ((uintptr_t)q & 15) || ((uintptr_t)uk & 1) || ((uintptr_t)qabs & 7))
    return -1;
  const int mt = T <= 16 ? 1 : T <= 32 ? 2 : 4;
  const dim3 grid(R / 64, H, (T + 16 * mt - 1) / (16 * mt));
#define XGM_LQ(NK, MT) latent_query_kernel<NK, MT><<<grid, 256, 0, st>>>((const bf16*)q, dq, (const bf16*)uk, (bf16*)qabs, T, H, R);
#define XGM_LQM(NK) \
  if (mt == 1) { XGM_LQ(NK, 1) } else if (mt == 2) { XGM_LQ(NK, 2) } else { XGM_LQ(NK, 4) }
  if (dn == 32) { XGM_LQM(1) } else if (dn == 64) { XGM_LQM(2) } else { XGM_LQM(4) }
#undef XGM_LQM
#undef XGM_LQ
  return 0;
}
}  // namespace xgm
