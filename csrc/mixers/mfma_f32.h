// Pieces shared by the chunked fp32 recurrences (chunk_scan.hip, delta_chunk.hip).
//
// v_mfma_f32_16x16x4_f32: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and D[4 (l / 16) + r][l % 16], r = 0..3. The
// contraction may run in any order as long as both operands agree: with step r of lane group g standing for index 4 g + r, a D
// tile is the B operand of the next product as it lies, and D of a transposed product is its A operand.
#pragma once

#include "attention_common.h"

namespace xgm {

using xgk::f32x4_t;

__device__ __forceinline__ f32x4_t mfma_f32(float a, float b, f32x4_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
#else
  return c;
#endif
}

// A chunk's tokens lie at these positions of its 16 rows (an involution), so that the four matrix steps of the state's update, which
// take rows t, 4 + t, 8 + t and 12 + t, take tokens 4 t .. 4 t + 3: the terms join in the order of the token loop (ascending where
// decays are strong; the other order costs the state 16 % of error at decays around 1/2).
__device__ __forceinline__ constexpr int tok_pos(int t) { return (t & 3) << 2 | t >> 2; }

// inputs past 2^28, infinities and NaN: a chunk that holds one runs token by token (a masked 0 times infinity would reach
// the tokens before it)
constexpr float kChunkMaxIn = 268435456.f;
__device__ __forceinline__ bool out_of_range(float x) { return !(fabsf(x) < kChunkMaxIn); }

// A running product of decays as the sum of two floats: the rounding of every factor is kept, so that a chunk's 16 steps cost the
// state one rounding instead of 16. (A sum of logarithms is rounded to 2^-24 of its own size, which is an error of the decay
// itself: at decays around 1/2 the state's was 5 to 9 times the token loop's.)
struct Prod {
  float h, l;
};
__device__ __forceinline__ Prod prod_mul(Prod a, float f) {
  const float h = a.h * f;
  return {h, fmaf(a.l, f, fmaf(a.h, f, -h))};
}
__device__ __forceinline__ Prod prod_mul(Prod a, Prod b) {
  const float h = a.h * b.h;
  return {h, fmaf(a.h, b.l, fmaf(a.l, b.h, fmaf(a.h, b.h, -h)))};
}
__device__ __forceinline__ float prod_times(Prod p, float x) { return fmaf(p.h, x, p.l * x); }
// a + b and what its rounding left out
__device__ __forceinline__ Prod two_sum(float a, float b) {
  const float s = a + b, bb = s - a;
  return {s, (a - (s - bb)) + (b - bb)};
}
// x / p and 1 / p: the reciprocal instruction and one Newton step
__device__ __forceinline__ float prod_div(float x, Prod p) {
  const float r = rcp_fast(p.h), t = x * r;
  return fmaf(fmaf(-p.l, t, fmaf(-p.h, t, x)), r, t);
}
__device__ __forceinline__ float prod_rcp(Prod p) {
  const float r = rcp_fast(p.h);
  return fmaf(r, fmaf(-p.l, r, fmaf(-p.h, r, 1.f)), r);
}

}  // namespace xgm
