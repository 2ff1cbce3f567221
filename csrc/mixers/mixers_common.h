// Helpers shared by the sequence-mixer translation units (csrc/mixers/*.hip): loads / stores of
// activations that are float or bf16 (raw uint16_t), and the host-side dtype dispatch.
#pragma once

#include "common.h"

namespace xgm {
using xgk::bf2f;
using xgk::block_sum;
using xgk::f2bf;
using xgk::wave_max;
using xgk::wave_sum;
using xgk::wave_sum_products;
typedef uint16_t bf16;

template <typename T> __device__ __forceinline__ float ldf(const T* p);
template <> __device__ __forceinline__ float ldf<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float ldf<bf16>(const bf16* p) { return bf2f(*p); }
template <typename T> __device__ __forceinline__ void stf(T* p, float v);
template <> __device__ __forceinline__ void stf<float>(float* p, float v) { *p = v; }
template <> __device__ __forceinline__ void stf<bf16>(bf16* p, float v) { *p = f2bf(v); }

__device__ __forceinline__ float sigmoidf(float x) { return 1.f / (1.f + expf(-x)); }

// 4 consecutive elements (16-byte / 8-byte aligned)
__device__ __forceinline__ void ld4(const float* p, float (&f)[4]) {
  const float4 v = *reinterpret_cast<const float4*>(p);
  f[0] = v.x, f[1] = v.y, f[2] = v.z, f[3] = v.w;
}
__device__ __forceinline__ void ld4(const bf16* p, float (&f)[4]) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  f[0] = __uint_as_float(v.x << 16), f[1] = __uint_as_float(v.x & 0xFFFF0000u);
  f[2] = __uint_as_float(v.y << 16), f[3] = __uint_as_float(v.y & 0xFFFF0000u);
}
__device__ __forceinline__ void st4(float* p, const float (&f)[4]) {
  *reinterpret_cast<float4*>(p) = make_float4(f[0], f[1], f[2], f[3]);
}
__device__ __forceinline__ void st4(bf16* p, const float (&f)[4]) {
  *reinterpret_cast<uint2*>(p) = make_uint2(xgk::pack2(f[0], f[1]), xgk::pack2(f[2], f[3]));
}

// four elements as they lie in memory: loads of a batch are issued before the first conversion waits for one
template <typename T> struct Raw4;
template <> struct Raw4<float> {
  float4 v;
  __device__ __forceinline__ void load(const float* p) { v = *reinterpret_cast<const float4*>(p); }
  __device__ __forceinline__ void zero() { v = make_float4(0.f, 0.f, 0.f, 0.f); }
  __device__ __forceinline__ void get(float (&f)[4]) const { f[0] = v.x, f[1] = v.y, f[2] = v.z, f[3] = v.w; }
};
template <> struct Raw4<bf16> {
  uint2 v;
  __device__ __forceinline__ void load(const bf16* p) { v = *reinterpret_cast<const uint2*>(p); }
  __device__ __forceinline__ void zero() { v = make_uint2(0, 0); }
  __device__ __forceinline__ void get(float (&f)[4]) const {
    f[0] = __uint_as_float(v.x << 16), f[1] = __uint_as_float(v.x & 0xFFFF0000u);
    f[2] = __uint_as_float(v.y << 16), f[3] = __uint_as_float(v.y & 0xFFFF0000u);
  }
};

// v += the N - 1 slabs behind the first, all of them in flight
template <int N>
__device__ __forceinline__ void add_slabs_n(const float* p, int64_t slab, float (&v)[4]) {
  float u[N - 1][4];
#pragma unroll
  for (int s = 1; s < N; ++s) ld4(p + s * slab, u[s - 1]);
#pragma unroll
  for (int s = 1; s < N; ++s)
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += u[s - 1][e];
}
// ... of n (1, 2, 4 or 8 parts are what the products have)
__device__ __forceinline__ void add_slabs(const float* p, int64_t slab, int n, float (&v)[4]) {
  if (n == 4) add_slabs_n<4>(p, slab, v);
  else if (n == 8) add_slabs_n<8>(p, slab, v);
  else if (n == 2) add_slabs_n<2>(p, slab, v);
  else
    for (int s = 1; s < n; ++s) {
      float u[4];
      ld4(p + s * slab, u);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += u[e];
    }
}

// sum over the L lanes (a power of two, the same for all) of an aligned segment of the wave, whose lanes all take part: lanes ^ L / 2, ..,
// 1 joined in turn by register moves, as wave_sum does it
template <int CTRL>
__device__ __forceinline__ float lane_dpp(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
#else
  return v;
#endif
}
__device__ __forceinline__ float seg_sum(float v, int L) {
#if defined(__HIP_DEVICE_COMPILE__)
  if (L > 32) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  }
  if (L > 16) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  }
#endif
  if (L > 8) v += lane_dpp<0x128>(v);                    // row_ror:8
  if (L > 4) v += lane_dpp<0x1B>(lane_dpp<0x141>(v));    // half rows mirrored (^ 7), quads mirrored (^ 3)
  if (L > 2) v += lane_dpp<0x4E>(v);
  if (L > 1) v += lane_dpp<0xB1>(v);
  return v;
}

// e^z - 1 - z for z <= 0. Above -1, z^2 times the polynomial that interpolates the quotient at the 7 Chebyshev points of [-1, 0]
// (1e-8 of it off), which spares the difference of close numbers; else the exponential itself (the difference is above 1/3).
__device__ __forceinline__ float exp_tail(float z) {
  float p = fmaf(z, 1.6928126569837332e-05f, 0.00018832476052921265f);
  p = fmaf(z, p, 0.0013822416076436639f);
  p = fmaf(z, p, 0.008331050164997578f);
  p = fmaf(z, p, 0.041666291654109955f);
  p = fmaf(z, p, 0.166666641831398f);
  p = fmaf(z, p, 0.5f);
#if defined(__HIP_DEVICE_COMPILE__)
  const float e = __builtin_amdgcn_exp2f(z * 1.44269504f);
#else
  const float e = expf(z);
#endif
  return z > -1.f ? z * z * p : (e - 1.f) - z;
}

// xIELU: sp z^2 + z / 2 for z > 0, cn (e^z - 1 - z) + z / 2 else. z / 2 is exact, so it joins in the last multiply-add.
// Error of the fp32 result against fp64 (2-norm over a range of z; in brackets with expm1f and every operation rounded): above
// -1/2 3.4e-8 (1.0e-7), -1 to -1/2 1.2e-7 (1.8e-7), -2 to -1 1.8e-7 (2.1e-7), 0 to 5 3.3e-8 (4.0e-8).
__device__ __forceinline__ float xieluf(float z, float sp, float cn) {
  return fmaf(z > 0.f ? sp * z : cn, z > 0.f ? z : exp_tail(z), 0.5f * z);
}

// The workgroup of row kernels with `lanes` threads a row: a row's own (256 of its threads, or whole waves), and below a wave as many rows
// as 256 threads hold. us, a wave a row / now: head norms with gates, 8192 rows of one head of 64 4.8 / 2.9, group norms with
// gates of 8192 x 64 4.9 / 3.1.
inline dim3 row_block(int lanes) {
  return lanes >= 64 ? dim3(lanes > 256 ? 256 : (lanes + 63) / 64 * 64) : dim3(max(1, lanes), 256 / max(1, lanes));
}

// max(z, 0)^2; a NaN stays one (fmaxf would make it 0)
__device__ __forceinline__ float relu2f(float z) {
  const float r = z < 0.f ? 0.f : z;
  return r * r;
}
__device__ __forceinline__ float siluf(float x) { return x / (1.f + expf(-x)); }
__device__ __forceinline__ float softplusf(float x) { return x > 20.f ? x : log1pf(expf(x)); }

}  // namespace xgm

#define XGM_DISPATCH_T(f32, ...)      \
  if (f32) {                          \
    using T = float;                  \
    __VA_ARGS__                       \
  } else {                            \
    using T = bf16;                   \
    __VA_ARGS__                       \
  }
