// Attention of prompt portions on the matrix cores, bf16: 32 query rows per wave on v_mfma_f32_32x32x16_bf16.
//
// A workgroup of 8 waves = GH query heads of one key/value head x 8 / GH blocks of 32 rows, over 64-key tiles of K and V
// that LDS-DMA brings into a ring NSLOT - 1 tiles ahead (no staging registers, counted vmcnt waits, one raw barrier per
// tile). S^T = K Q^T leaves a lane with 32 scores of ONE query row; packed to bf16 they are the B operand of
// O^T += V^T P^T, whose A operand is a transposed LDS read. A row of DK = 64 / 128 entries is 8 / 16 chunks of 16 bytes;
// chunk c of row r lies at chunk c ^ xsw(r), applied to the DMA's source address, so that both the row reads of K and the
// transposed reads of V touch every bank once.
//
// Visibility, scores, weights and gates are those of chunk_attention.hip. Keys are walked in whole tiles: first the tiles
// that hold kept first keys (when the window starts behind them), then from the window's first key, rounded down to 16, to
// the last row's own; a tile (or a wave's part of it) that lies wholly inside every row's view skips the per-key tests, one
// that no row of the wave sees is passed over. 16 keys in a row share a page (block sizes are multiples of 16), so the page
// index of a wave's DMA rows is one scalar load.
//
// LAT: multi-head attention over expanded latents. Every head has keys and values of its own in dense rows: [kn (dn) | the
// rotated key shared by all heads (rd, read from the latent rows)] and v; key `lo` + i of sequence s is row koff[s] + i, lo the
// first key its first query row sees. The rotary part of a query is rotated while it is loaded. In latent space (latent_attention)
// a (query, key) pair costs 2 (2 R + rd) operations per head, here 2 (dn + rd + dv): 3.4 times less at R = 256 and heads of 64,
// against one product per key row that expands it (4 x 2048 tokens, 32 heads of 64 + 32, window 1024: 950 -> 205 us with the
// gather and both expansions, the attention 155 of them, since then 127; heads of 128 + 64, window 4096: 3857 -> 395). Rows of 96 and 192 entries have 12 and 24 chunks: the permutation there
// stays inside groups of 4 and 8.
//
// Vector work and matrix instructions bound it together: 4001 tokens, 32 heads of 64 + 64, took 275 vector instructions a tile and
// wave beside 16 matrix ones (156 and 64 of 266 thousand clocks), 125 us. Scores that stay products up to the exponential, masks by
// edge (compares and selects, no branches), addresses as a uniform base and a lane's constant: 113 us; 16 heads of 64 + 128 with a
// distance penalty 131 -> 121, 2 x 1800 tokens of 32 heads of 128 + 128 97 -> 93, expanded latents (64 + 32) + 64 of 4 x 2048 tokens
// 154 -> 127, (128 + 64) + 128 of 2 x 1300 96 -> 84. A distance penalty in units of products (no product with the scale in front of it),
// and heads of 128 with one block of 32 keys behind the other: 4001 tokens of 32 heads of 128 + 128 with a penalty 229 -> 214, of 16 of
// 64 + 64 105 -> 101; heads of 128 + 64 with bounded scores 116 -> 111, of 128 + 128 without either 187 -> 182.
// (Heads of 64: both blocks of 32 keys in turn, so that two chains of matrix instructions run; waves' priorities and two sums for l change nothing.)
#include "attention_common.h"
#include "glds.h"

namespace xgm {

constexpr int kPT = 64;   // keys per tile

typedef xgk::f32x16_t f32x16_t;

__device__ __forceinline__ f32x16_t mfma32x32x16(xgk::bf16x8_t a, xgk::bf16x8_t b, f32x16_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
#else
  return c;
#endif
}

__device__ __forceinline__ float xor32_max(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
#else
  return x;
#endif
}

__device__ __forceinline__ void sched_fence() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_sched_barrier(0);
#endif
}

// chunk permutation of a row: 16 consecutive rows hit all 16-byte slots of the banks for one chunk, and 4 rows x 4
// neighbouring chunks do too
template <int D>
__device__ __forceinline__ int xsw(int r) {
  return D == 96 ? (r >> 2) & 3 : D == 192 ? (r >> 1) & 7 : D == 128 ? ((r & 3) << 2) | ((r >> 2) & 3) : (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
}

template <int DK, int DV, int GH, int NSLOT, int WFN, bool LAT>
__global__ __launch_bounds__(512, DK == 64 && DV == 64 ? 4 : 2) void prompt_attention_kernel(
    const AttnArgs a, const int32_t* __restrict__ block_tables, const bf16* __restrict__ kcache,
    const bf16* __restrict__ vcache, int tiles_per_seq, int n_hg, const LatentRows lr) {
  constexpr bool sig = WFN == kWeightsSigmoid, capped = WFN == kWeightsBounded || WFN == kWeightsCapped;
  constexpr bool bounded = WFN == kWeightsBounded;
  constexpr int NW = 8, RBLK = NW / GH;
  constexpr int KROW = DK * 2, VROW = DV * 2;            // bytes of a row
  constexpr int KT = kPT * KROW, SLOT = KT + kPT * VROW;  // bytes of a K tile, of a ring slot [K | V]
  constexpr int KD = (DK + 63) / 64, VD = DV / 64;        // DMA instructions per wave and tile (8 rows per wave)
  static_assert(LAT || DK % 64 == 0, "rows of 96 and 192 entries: dense form only");
  __shared__ __attribute__((aligned(1024))) char lds[NSLOT * SLOT];

  const int bid = blockIdx.x;
  const int hg = bid % n_hg, rest = bid / n_hg;           // head groups fastest: an XCD streams few key/value heads
  const int s = rest % a.ns;
  const int q0 = a.qsl[s], qn = a.qsl[s + 1] - q0;
  if (a.slots[s] < 0 || qn <= 0) return;
  const int ctx = a.seq_lens[s] - qn;
  const int rep = a.H / a.G, hb = rep / GH;
  const int g = hg / hb;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int head = g * rep + (hg % hb) * GH + w % GH;
  const int rb = w / GH;
  const int r = lane & 31, hf = lane >> 5;
  const int voff = a.vmode == kValuesAll ? 0 : (a.vmode >= 0 ? a.vmode : g) * a.dv_head;
  const int64_t krow = (int64_t)a.G * DK, vrow = (int64_t)a.G * a.dv_head;   // elements between two cached rows
  // The workgroup's blocks of 32 rows, lowest and highest, and the wave's own (nblk: none). Where every row sees its keys from the
  // same first one on, a late row has up to all of them to walk and an early one few: half of a workgroup's blocks come from the
  // front and half from the back, an early and a late wave on each SIMD, so all workgroups have the same work (rows of the same
  // place together, 4001 tokens: 179 us for 16 heads of 64 + 128 with a distance penalty, 122 for 32 of 64 + 64; so 138, 118).
  const int nblk = (qn + 31) / 32, wg = rest / a.ns;
  int low, top, blk;
  if (RBLK > 1 && first_visible(a.mask, a.size, ctx + qn - 1) == first_visible(a.mask, a.size, ctx)) {
    constexpr int HALF = RBLK > 1 ? RBLK / 2 : 1;
    const int front = (nblk + 1) / 2, back = nblk - front, at = wg * HALF;   // blocks [0, front) and, from the end, `back` more
    if (at >= front) return;
    low = at, top = at < back ? nblk - 1 - at : min(front, at + HALF) - 1;
    blk = rb < HALF ? (at + rb < front ? at + rb : nblk) : (at + rb - HALF < back ? nblk - 1 - (at + rb - HALF) : nblk);
  } else {
    low = (tiles_per_seq - 1 - wg) * RBLK;   // late row tiles see the most keys: first
    if (low >= nblk) return;
    top = min(nblk, low + RBLK) - 1, blk = low + rb;
  }
  const int my_row = blk * 32 + r;
  const int pos_q = ctx + my_row;
  const int lo_q = first_visible(a.mask, a.size, pos_q);
  const int pos_lo = ctx + blk * 32, pos_hi = ctx + min(qn, blk * 32 + 32) - 1;   // the wave's rows (uniform)
  const int lo_lo = first_visible(a.mask, a.size, pos_lo), lo_hi = first_visible(a.mask, a.size, pos_hi);
  // tiles of the workgroup: `kt` tiles from key 0 on, then from key `kfirst` on (kt = 0: no kept keys behind a gap)
  const int last = ctx + min(qn, top * 32 + 32) - 1;
  int kfirst = first_visible(a.mask, a.size, ctx + low * 32) & ~15;
  int kt = (a.keep + kPT - 1) / kPT;
  if (kfirst <= kt * kPT) kfirst = a.keep > 0 ? 0 : kfirst, kt = 0;
  const int ntiles = kt + (last - kfirst + kPT) / kPT;
  const int32_t* bt = block_tables + (int64_t)s * a.bt_width;
  auto tile_key = [&](int t) { return t < kt ? t * kPT : kfirst + (t - kt) * kPT; };

  const bool pages_pow2 = (a.bs & (a.bs - 1)) == 0;
  const int page_shift = __builtin_ctz(a.bs);
  const int lat_lo = first_visible(a.mask, a.size, ctx);   // the sequence's first dense key row
  const int64_t lat_row = LAT ? (int64_t)lr.koff[s] - lat_lo : 0;
  // what a lane's DMA loads add to the tile's first row of the wave (elements); LAT: the address for key 0 and the bytes of a key's row
  uint32_t k_off[KD], v_off[VD], k_row[LAT ? KD : 1];
  const bf16* k_from[LAT ? KD : 1];
#pragma unroll
  for (int i = 0; i < KD; ++i) {
    if constexpr (LAT) {
      const int idx = min(64 * i + lane, DK - 1), rr = idx / (DK / 8), d = ((idx % (DK / 8)) ^ xsw<DK>(8 * w + rr)) * 8;
      k_off[i] = rr, k_row[i] = 2 * (d < lr.dn ? a.H * lr.dn : lr.R + lr.rd);
      k_from[i] = d < lr.dn ? lr.kn + (lat_row * a.H + head) * lr.dn + d : lr.lat + lat_row * (lr.R + lr.rd) + lr.R + d - lr.dn;
    } else {
      const int rr = KD == 2 ? 4 * i + (lane >> 4) : lane >> 3;
      k_off[i] = rr * (uint32_t)krow + g * DK + 8 * ((KD == 2 ? lane & 15 : lane & 7) ^ xsw<DK>(8 * w + rr));
    }
  }
#pragma unroll
  for (int i = 0; i < VD; ++i) {
    const int rr = VD == 2 ? 4 * i + (lane >> 4) : lane >> 3, ch = (VD == 2 ? lane & 15 : lane & 7) ^ xsw<DV>(8 * w + rr);
    v_off[i] = LAT ? rr * (uint32_t)(a.H * DV) + ch * 8 : rr * (uint32_t)vrow + voff + ch * 8;
  }
  auto issue = [&](int t) {
    char* dst = lds + (t % NSLOT) * SLOT;
    const int k1 = tile_key(t) + 8 * w;   // the wave's 8 rows: inside one aligned run of 16 keys
    const bool whole = k1 + 7 <= last;    // (else the last row again)
    if constexpr (LAT) {   // (keys in front of the first row are masked: any row will do)
      const bool in = whole && k1 >= lat_lo;
#pragma unroll
      for (int i = 0; i < KD; ++i) {
        const uint32_t key = in ? k1 + k_off[i] : max(min(k1 + (int)k_off[i], last), lat_lo);
        if (64 * i + lane < DK)   // (8 rows of DK / 8 chunks)
          xgk::glds16(reinterpret_cast<const char*>(k_from[i]) + (uint64_t)key * k_row[i], dst + 8 * w * KROW + i * 1024);
      }
      const bf16* vp = lr.v + ((lat_row + k1) * a.H + head) * DV;
#pragma unroll
      for (int i = 0; i < VD; ++i) {
        const int rr = VD == 2 ? 4 * i + (lane >> 4) : lane >> 3;
        const int64_t at = in ? v_off[i] : (int64_t)v_off[i] + (int64_t)(max(min(k1 + rr, last), lat_lo) - k1 - rr) * (a.H * DV);
        xgk::glds16(vp + at, dst + KT + (8 * w) * VROW + i * 1024);
      }
      return;
    }
    const int key0 = min(k1, last), pidx = pages_pow2 ? key0 >> page_shift : key0 / a.bs;
    const int64_t row = (int64_t)bt[pidx] * a.bs - (int64_t)pidx * a.bs + k1;
    const bf16 *kp = kcache + row * krow, *vp = vcache + row * vrow;
#pragma unroll
    for (int i = 0; i < KD; ++i) {
      const int rr = KD == 2 ? 4 * i + (lane >> 4) : lane >> 3;
      xgk::glds16(kp + (whole ? (int64_t)k_off[i] : k_off[i] + (min(k1 + rr, last) - k1 - rr) * krow), dst + (8 * w) * KROW + i * 1024);
    }
#pragma unroll
    for (int i = 0; i < VD; ++i) {
      const int rr = VD == 2 ? 4 * i + (lane >> 4) : lane >> 3;
      xgk::glds16(vp + (whole ? (int64_t)v_off[i] : v_off[i] + (min(k1 + rr, last) - k1 - rr) * vrow), dst + KT + (8 * w) * VROW + i * 1024);
    }
  };

  // Q^T (B operand): lane holds Q[row r][16 ks + 8 hf + 0..7]
  xgk::bf16x8_t qf[DK / 16];
  {
    const bf16* qp = a.q + ((int64_t)(q0 + min(my_row, qn - 1)) * a.H + head) * DK + 8 * hf;
#pragma unroll
    for (int ks = 0; ks < DK / 16; ++ks) {
      uint4 x = xgk::ld16(qp + 16 * ks);
      const int i0 = 16 * ks + 8 * hf - lr.dn;   // LAT: pairs (i0, i0 + 1), .. of the rotary part turn by the row's angles
      if (LAT && i0 >= 0 && i0 < lr.rot_dims) {
        float f[8];
        xgk::unpack8(x, f);
        const float* cs = lr.rot + ((int64_t)min(pos_q, ctx + qn - 1) * (lr.rot_dims >> 1) + (i0 >> 1)) * 2;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          if (i0 + e < lr.rot_dims) {
            const float c = cs[e], sn = cs[e + 1], u = f[e], v = f[e + 1];
            f[e] = u * c - v * sn;
            f[e + 1] = v * c + u * sn;
          }
        }
        x = xgk::pack8(f);
      }
      qf[ks] = xgk::as_frag(x);
    }
  }
  const float cap2 = capped ? a.softcap * kLog2e : 0.f;
  auto uniform = [](float x) {   // (the same in all lanes: a scalar register)
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x)));
  };
  float sc_h = a.scale * (a.temp ? a.temp[head] : 1.f) * (capped ? 2.f / a.softcap : 1.f) * kLog2e;
  const float pen1 = uniform(a.r1 ? a.r1[head] : 0.f), pen2 = uniform(a.r1 ? a.r2[head] : 0.f);
  const float sbias = uniform((sig && a.hbias) ? a.hbias[head] * kLog2e : 0.f);
  // Scores stay products until they are exponentials: one multiply-add takes them to their distance from the row's reference m (sc1;
  // 1 where a bound has made them scores already, or a penalty that in units of products would leave fp32). The sign of the scale is the
  // query's, so that the largest product is the largest score; a scale of 0 is the smallest number instead (0 would make a masked one not
  // a number).
  const float pen_f = pen1 / fabsf(sc_h);   // the penalty in units of products
  const bool scaled = capped || sig || (a.r1 && !(fabsf(pen_f) < 1e30f && fabsf(sc_h) > 1e-30f));
  const uint32_t flip = !scaled && sc_h < 0.f ? 0x80008000u : 0u;
  sc_h = uniform(scaled ? sc_h : sc_h == 0.f ? 1.1754944e-38f : fabsf(sc_h));
  const float sc1 = scaled ? 1.f : sc_h;
  const float pen = uniform(scaled ? pen1 : pen_f);
  float m = bounded ? 0.f : a.sink ? a.sink[head] * kLog2e : -INFINITY;
  float l = (a.sink && hf == 0) ? 1.f : 0.f;   // each half of a row's two lanes sums its own keys
  f32x16_t o[DV / 32];
#pragma unroll
  for (int db = 0; db < DV / 32; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[db][e] = 0.f;
  // everything loaded so far is complete before the first DMA: from here on vmcnt counts the DMAs alone
#pragma unroll
  for (int ks = 0; ks < DK / 16; ++ks) {
    uint4 x = __builtin_bit_cast(uint4, qf[ks]);
    x.x ^= flip, x.y ^= flip, x.z ^= flip, x.w ^= flip;
    qf[ks] = xgk::as_frag(x);
    asm volatile("" : "+v"(qf[ks]));
  }
  asm volatile("" : "+v"(m));
  xgk::wait_vmcnt<0>();
#pragma unroll
  for (int p = 0; p < NSLOT - 1; ++p)
    if (p < ntiles) issue(p);

  const int tg = lane >> 4, tq = (lane & 15) >> 2, tp = lane & 3;
  const bool wave_on = pos_lo <= pos_hi;
  for (int j = 0; j < ntiles; ++j) {
    if constexpr (NSLOT == 3) {
      if (j + 1 < ntiles) xgk::wait_vmcnt<KD + VD>();
      else xgk::wait_vmcnt<0>();
    } else {
      xgk::wait_vmcnt<0>();
    }
    xgk::raw_barrier();
    if (j + NSLOT - 1 < ntiles) issue(j + NSLOT - 1);
    const int base = tile_key(j);
    // (wave-uniform) nothing of this tile is visible to the wave's rows
    if (!wave_on || base > pos_hi || (base + kPT - 1 < lo_lo && base >= a.keep)) continue;
    const uint32_t slot = (j % NSLOT) * SLOT;
    // chunk 2 ks + hf of row r: KROW a power of two, one xor of the whole address; else xor inside 4 (8) chunks, added on
    constexpr bool POW2 = DK == 64 || DK == 128;
    constexpr int KG = DK == 192 ? 4 : 2;   // (pairs of chunks per permuted group)
    const uint32_t k_lane = POW2 ? (slot + r * KROW) ^ ((uint32_t)(hf ^ xsw<DK>(r)) << 4)
                                 : slot + r * KROW + ((uint32_t)((hf ^ xsw<DK>(r)) & 1) << 4);
    uint32_t k_pair[KG];
#pragma unroll
    for (int i = 0; i < KG; ++i) k_pair[i] = (uint32_t)(i ^ (xsw<DK>(r) >> 1)) << 5;
    auto k_at = [&](int ks) { return POW2 ? k_lane ^ (ks << 5) : k_lane + k_pair[ks % KG] + (ks / KG) * (32 * KG); };
    const uint32_t v_row = slot + KT + (4 * hf + tq) * VROW + 8 * (tp & 1);
    const uint32_t v_hi = (uint32_t)(DV == 128 ? tq : tq >> 1) << 6, v_lo = 2 * (tg & 1) + (tp >> 1);
    const uint32_t v_lane0 = (v_row + ((v_lo ^ hf) << 4)) | v_hi;
    const uint32_t v_lane1 = (v_row + 8 * VROW + ((v_lo ^ (hf + 2)) << 4)) | v_hi;

    f32x16_t sacc[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) sacc[kb][e] = 0.f;
    if constexpr (DK == 128) {   // (turns as below: as fast without a bound or penalty, 2 to 5 % slower with)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int ks = 0; ks < DK / 16; ++ks)
          sacc[kb] = mfma32x32x16(xgk::as_frag(xgk::ld16(lds + (k_at(ks) + kb * 32 * KROW))), qf[ks], sacc[kb]);
        sched_fence();   // bound the hoisted fragment reads
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < DK / 16; ++ks) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
          sacc[kb] = mfma32x32x16(xgk::as_frag(xgk::ld16(lds + (k_at(ks) + kb * 32 * KROW))), qf[ks], sacc[kb]);
        if (ks % 2) sched_fence();
      }
    }
    // scores in units of ln 2; register e of block kb is key base + 32 kb + 4 hf + (e & 3) + 8 (e >> 2)
    const bool full = base + kPT - 1 <= pos_lo && (base >= lo_hi || base + kPT <= a.keep);
    const int vis_hi = pos_q - base - 4 * hf, vis_lo = lo_q - base - 4 * hf, vis_keep = a.keep - base - 4 * hf;
    if (scaled) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          float v = sacc[kb][e] * sc_h;
          if constexpr (capped) v = cap2 - 2.f * cap2 * rcp_fast(1.f + exp2_fast(v));
          sacc[kb][e] = v;
        }
    }
    if (a.r1) {
      // (distances are exact in fp32; those of keys behind the query may have no logarithm and are masked below; 138 -> 130 us
      // against an integer distance and the general logarithm)
      const float dist = (float)vis_hi;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          sacc[kb][e] -= pen * log2_fast(fmaf(pen2, dist - (float)(kb * 32 + (e & 3) + 8 * (e >> 2)), 1.f));
    }
    if (!full) {   // (wave-uniform: a tile mostly has one of the two edges)
      if (base + kPT - 1 > pos_lo) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int e = 0; e < 16; ++e) sacc[kb][e] = kb * 32 + (e & 3) + 8 * (e >> 2) > vis_hi ? -INFINITY : sacc[kb][e];
      }
      if (base < lo_hi && base + kPT > a.keep) {   // keys from vis_keep on, up to vis_lo
        const uint32_t hidden = max(vis_lo - vis_keep, 0);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int c = kb * 32 + (e & 3) + 8 * (e >> 2);
            const bool out = DK == 128 ? (uint32_t)(c - vis_keep) < hidden : (bool)((int)(c < vis_lo) & (int)(c >= vis_keep));
            sacc[kb][e] = out ? -INFINITY : sacc[kb][e];
          }
      }
    }
    if constexpr (sig) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e) sacc[kb][e] = rcp_fast(1.f + exp2_fast(-(sacc[kb][e] + sbias)));
    } else {
      float nm = 0.f;
      if constexpr (!bounded) {
        float mx = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sacc[kb][e]);
        mx = xor32_max(mx) * sc1;
        // (none of the wave's rows has a new maximum: nothing to rescale. A reference that lags behind the maximum by up to 2^8 is 2 to 4 %
        // faster, but the largest weight is then not 1, which bf16 holds exactly: 2 to 20 % more error at scores of spread 1 to 3)
        if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {
          const float m_new = fmaxf(m, mx), alpha = m == -INFINITY ? 0.f : exp2_fast(m - m_new);
          l *= alpha;
#pragma unroll
          for (int db = 0; db < DV / 32; ++db)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[db][e] *= alpha;
          m = m_new;
        }
        nm = m == -INFINITY ? 0.f : -m;
      }
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float p = exp2_fast(bounded ? sacc[kb][e] : fmaf(sacc[kb][e], sc1, nm));
          sacc[kb][e] = p;
          l += p;
        }
    }
    // O^T += V^T P^T: step (kb, ss) takes score registers 8 ss .. 8 ss + 7 (keys 32 kb + 16 ss + ..)
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int ss = 0; ss < 2; ++ss) {
        uint4 pb;
        pb.x = xgk::pack2(sacc[kb][8 * ss + 0], sacc[kb][8 * ss + 1]);
        pb.y = xgk::pack2(sacc[kb][8 * ss + 2], sacc[kb][8 * ss + 3]);
        pb.z = xgk::pack2(sacc[kb][8 * ss + 4], sacc[kb][8 * ss + 5]);
        pb.w = xgk::pack2(sacc[kb][8 * ss + 6], sacc[kb][8 * ss + 7]);
        const xgk::bf16x8_t pf = xgk::as_frag(pb);
        const uint32_t ro = (kb * 32 + 16 * ss) * VROW;
#pragma unroll
        for (int db = 0; db < DV / 32; ++db) {
          const xgk::bf16x4_t a0 = xgk::lds_read_tr16(reinterpret_cast<const uint16_t*>(lds + ((v_lane0 ^ (db << 6)) + ro)));
          const xgk::bf16x4_t a1 = xgk::lds_read_tr16(reinterpret_cast<const uint16_t*>(lds + ((v_lane1 ^ (db << 6)) + ro)));
          const xgk::bf16x8_t vf = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
          o[db] = mfma32x32x16(vf, pf, o[db]);
        }
        if (ss) sched_fence();
      }
  }
  l += __shfl_xor(l, 32, 64);
  // lane holds O[row r][32 db + 8 t + 4 hf + 0..3] in registers 4 t .. 4 t + 3
  if (my_row < qn) {
    const int64_t row = q0 + my_row;
    float inv = sig ? 1.f : (l > 0.f ? 1.f / l : 0.f);
    if (a.gate && !a.gate_elem) inv *= sigmoidf(bf2f(a.gate[row * a.ld_gate + head]));
    bf16* op = a.out + (row * a.H + head) * DV + 4 * hf;
    const bf16* ge = (a.gate && a.gate_elem) ? a.gate + row * a.ld_gate + (int64_t)head * DV + 4 * hf : nullptr;
#pragma unroll
    for (int db = 0; db < DV / 32; ++db)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        float e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          e[i] = o[db][4 * t + i] * inv;
          if (ge) e[i] *= sigmoidf(bf2f(ge[32 * db + 8 * t + i]));
        }
        *reinterpret_cast<uint2*>(op + 32 * db + 8 * t) = make_uint2(xgk::pack2(e[0], e[1]), xgk::pack2(e[2], e[3]));
      }
  }
}

bool prompt_attention(const AttnArgs& a, int max_q, int wfn, hipStream_t st) {
  const int dv = a.vmode == kValuesAll ? a.G * a.dv_head : a.dv_head;
  const int rep = a.H / a.G;
  if (a.bs % 16 != 0 || (a.dk != 64 && a.dk != 128) || (dv != 64 && dv != 128) || (uintptr_t)a.kcache % 16 != 0 ||
      (uintptr_t)a.vcache % 16 != 0 || (a.G * a.dv_head) % 8 != 0 || a.dv_head % 8 != 0)
    return false;
  const int gh = rep % 4 == 0 ? 4 : rep % 2 == 0 ? 2 : 1, bm = 32 * 8 / gh;
  const int tps = (max_q + bm - 1) / bm, n_hg = a.G * rep / gh;
  const int grid = n_hg * a.ns * tps;
#define XGM_PA3(DK, DV, GH, WFN)                                                                                      \
  prompt_attention_kernel<DK, DV, GH, 3, WFN, false><<<grid, 512, 0, st>>>(a, a.block_tables, a.kcache, a.vcache, tps, n_hg, \
                                                                          LatentRows{})
#define XGM_PA2(DK, DV, GH)                                  \
  switch (wfn) {                                             \
    case kWeightsSigmoid:                                    \
      XGM_PA3(DK, DV, GH, kWeightsSigmoid);                  \
      break;                                                 \
    case kWeightsBounded:                                    \
      XGM_PA3(DK, DV, GH, kWeightsBounded);                  \
      break;                                                 \
    case kWeightsCapped:                                     \
      XGM_PA3(DK, DV, GH, kWeightsCapped);                   \
      break;                                                 \
    default:                                                 \
      XGM_PA3(DK, DV, GH, kWeightsSoftmax);                  \
      break;                                                 \
  }
#define XGM_PA1(DK, DV)        \
  if (gh == 4) {               \
    XGM_PA2(DK, DV, 4)         \
  } else if (gh == 2) {        \
    XGM_PA2(DK, DV, 2)         \
  } else {                     \
    XGM_PA2(DK, DV, 1)         \
  }
  if (a.dk == 64 && dv == 64) {
    XGM_PA1(64, 64)
  } else if (a.dk == 128 && dv == 128) {
    XGM_PA1(128, 128)
  } else if (a.dk == 64) {
    XGM_PA1(64, 128)
  } else {
    XGM_PA1(128, 64)
  }
#undef XGM_PA1
#undef XGM_PA2
#undef XGM_PA3
  return true;
}

// ---- dense latent rows of a step's keys: per sequence the cached rows from the first key that its first new token sees to its
// last; koff[s] = first row of sequence s. One workgroup copies 16 rows.
constexpr int kGatherRows = 16;

__global__ __launch_bounds__(256) void latent_gather_kernel(const bf16* __restrict__ cache, const int32_t* __restrict__ block_tables,
                                                            int bt_width, int bs, const int32_t* __restrict__ qsl,
                                                            const int32_t* __restrict__ seq_lens,
                                                            const int32_t* __restrict__ slots, int ns, int window, int W8,
                                                            bf16* __restrict__ rows, int32_t* __restrict__ koff, int nk) {
  __shared__ int first_s, first_i;
  const int r0 = blockIdx.x * kGatherRows;
  if (threadIdx.x == 0) first_s = ns, first_i = 0;
  __syncthreads();
  if (threadIdx.x < 64) {   // key counts of 64 sequences at a time, summed up over the wave
    int before = 0;
    for (int s0 = 0; s0 < ns; s0 += 64) {
      const int s = s0 + threadIdx.x;
      int n = 0;
      if (s < ns) {
        const int q = qsl[s + 1] - qsl[s], len = seq_lens[s];
        n = slots[s] < 0 || q <= 0 ? 0 : len - max(0, len - q - window + 1);
      }
      int upto = n;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int up = __shfl_up(upto, o, 64);
        if (threadIdx.x >= o) upto += up;
      }
      const int at = before + upto - n;
      if (s < ns && blockIdx.x == 0) koff[s] = min(at, nk);
      if (r0 >= at && r0 < at + n) first_s = s, first_i = r0 - at;
      before += __shfl(upto, 63, 64);
    }
  }
  __syncthreads();
  int s = first_s, i = first_i;   // row r0 = key i of sequence s; the rows behind it follow
  for (int r = r0; r < min(r0 + kGatherRows, nk); ++r, ++i) {
    int lo = 0, len = 0;
    for (; s < ns; ++s, i = 0) {
      const int q = qsl[s + 1] - qsl[s];
      len = seq_lens[s], lo = max(0, len - q - window + 1);
      if (slots[s] >= 0 && q > 0 && i < len - lo) break;
    }
    if (s >= ns) break;
    const int key = lo + i;
    const uint4* src = reinterpret_cast<const uint4*>(cache) +
                       ((int64_t)block_tables[(int64_t)s * bt_width + key / bs] * bs + key % bs) * W8;
    for (int c = threadIdx.x; c < W8; c += 256) reinterpret_cast<uint4*>(rows)[(int64_t)r * W8 + c] = src[c];
  }
}

void latent_gather(const void* cache, const int32_t* bt, int bt_width, int bs, const int32_t* qsl, const int32_t* seq_lens,
                   const int32_t* slots, int ns, int window, int width, void* rows, int32_t* koff, int nk, hipStream_t st) {
  if (ns <= 0 || nk <= 0) return;
  latent_gather_kernel<<<(nk + kGatherRows - 1) / kGatherRows, 256, 0, st>>>(
      (const bf16*)cache, bt, bt_width, bs, qsl, seq_lens, slots, ns, window, width / 8, (bf16*)rows, koff, nk);
}

// q [T][H][dn + rd], out [T][H][dv]; kn [rows][H][dn], v [rows][H][dv], lat [rows][R + rd], koff of latent_gather
int latent_prompt_attention(const void* q, int dn, int rd, int dv, const void* kn, const void* v, const void* lat, int R,
                            const int32_t* koff, const void* gate, int64_t ld_gate, const float* rot, int rot_dims,
                            const int32_t* qsl, const int32_t* seq_lens, const int32_t* slots, void* out, int T_, int ns,
                            int max_q, int H, int window, float scale, hipStream_t st) {
  if (ns <= 0 || max_q <= 0) return 0;
  const int dk = dn + rd;
  if (dn % 8 || rd % 8 || R % 8 || H < 1 || window < 1 || rot_dims % 2 || rot_dims > rd || !((dk == 96 && dv == 64) ||
      (dk == 192 && dv == 128)))
    return -1;
  AttnArgs a = {};
  a.q = (const bf16*)q, a.qsl = qsl, a.seq_lens = seq_lens, a.slots = slots, a.out = (bf16*)out;
  a.T = T_, a.ns = ns, a.H = H, a.G = H, a.dk = dk, a.dv_head = dv, a.mask = kMaskWindow, a.size = window, a.scale = scale;
  a.gate = (const bf16*)gate, a.ld_gate = ld_gate, a.vmode = kValuesOwn, a.bs = 16;
  const LatentRows lr = {(const bf16*)kn, (const bf16*)v, (const bf16*)lat, koff, rot, dn, R, rd, rot_dims};
  const int tps = (max_q + 255) / 256, grid = H * ns * tps;
  if (dk == 96)
    prompt_attention_kernel<96, 64, 1, 3, kWeightsSoftmax, true><<<grid, 512, 0, st>>>(a, nullptr, nullptr, nullptr, tps, H, lr);
  else
    prompt_attention_kernel<192, 128, 1, 3, kWeightsSoftmax, true><<<grid, 512, 0, st>>>(a, nullptr, nullptr, nullptr, tps, H, lr);
  return 0;
}

}  // namespace xgm
