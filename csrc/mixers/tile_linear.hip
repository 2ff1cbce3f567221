// Products of many activation rows: the plain ones, and the sum of K's parts. The kernel is tile_linear.h's.
#include "tile_linear.h"

namespace xgm {
template <bool PAIR>
__global__ __launch_bounds__(256) void tile_linear_sum_kernel(const TileArgs a) {
  const int cols = (PAIR ? a.N / 2 : a.N) / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, slab = (int64_t)a.M * a.N;
  if (i >= (int64_t)a.M * cols) return;
  const int64_t row = i / cols;
  const int col = 4 * (int)(i - row * cols);
  const float* at = a.part + row * a.N + col;
  float v[4];
  ld4(at, v);
  add_slabs(at, slab, a.S, v);
  float up[4], b[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (PAIR) {
    ld4(at + a.N / 2, up);
    add_slabs(at + a.N / 2, slab, a.S, up);
  } else if (a.bias) {
    tile_bias(a, col, b);
  }
  tile_by_act<PAIR>(a, [&](auto act_c) __attribute__((always_inline)) {
    constexpr int ACT = decltype(act_c)::value;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = PAIR ? tile_glu<ACT>(a, v[e], up[e]) : tile_act<ACT>(a, v[e] + b[e]);
  });
  st4(a.out + row * (PAIR ? a.N / 2 : a.N) + col, v);
}

int tile_linear(const void* x, int64_t ld_x, const void* w, const void* bias, bool bias_f32, float* part, void* out, int M,
                int N, int K, int S, int act, int pairs, float p0, float p1, int fm, int fn, int cus, hipStream_t st) {
  const bool gated = act >= kTileGlu;
  if (M < 1 || N < 8 || N % 8 || K < 64 || K % 64 || ld_x < K || ld_x % 8 || S < 1 || S > K / 64 || act < 0 || gated != (pairs != 0) ||
      (gated && !xgk::glu_known(act - kTileGlu)) || cus < 1 || pairs < 0 || pairs > 2 || (gated && (bias || N % (pairs == kPairBlocks ? 32 : 8))) || (S > 1 && !part) ||
      (!out && (S == 1 || act != kTileNone || bias)) ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)bias | (uintptr_t)part | (uintptr_t)out) & 15) ||
      N >= kTileColumns || (int64_t)N * K * 2 >= (1LL << 32) || 256 * ld_x * 2 >= (1LL << 32))
    return -1;
  TileArgs a = {(const bf16*)x, (const bf16*)w, bias, S > 1 ? part : nullptr, (bf16*)out, ld_x, M, N, K, S, act, pairs, p0, p1, bias_f32,
                nullptr, nullptr, 0, 1, 0, M <= kRotateRows ? 32 * fn : 0};
  if (gated ? tile_launch_gated(a, fm, fn, cus, st) : tile_launch_size<false>(a, fm, fn, cus, st)) return -1;
  if (S > 1 && out) {   // (without a result the slabs are it: the next kernel adds them)
    const int64_t n = (int64_t)M * (gated ? N / 2 : N) / 4;
    if (gated) tile_linear_sum_kernel<true><<<(unsigned)((n + 255) / 256), 256, 0, st>>>(a);
    else tile_linear_sum_kernel<false><<<(unsigned)((n + 255) / 256), 256, 0, st>>>(a);
  }
  return 0;
}
}  // namespace xgm
