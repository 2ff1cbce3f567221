// The tile and the parts of K of a product on tile_linear.h: every form of the kernel is priced, the cheapest wins (the first of
// equals). Prompt steps rarely have the row count of the one before, so the search runs for every product of nearly every step: in
// Python it took 20 to 140 us a product, here 2 with the call; a step of a new row count, Dofivik "1b", 80 to 130 rows, 1886 -> 1733 us
// until its end, Loluzen 1216 -> 1177, Vizonex 1142 -> 1027. The prices and the rules around them are ops/tile_linear.py's.
#include <cmath>
#include <cstdint>

namespace xgm {

struct TilePrices {   // ops/tile_linear.py's, in this order
  double x_read, w_read, small, sum, part, part_bytes, out_bytes, split_k, split_tiles;
};

static int64_t up(int64_t a, int64_t b) { return (a + b - 1) / b; }

// tiles: n rows of {rows / 32, columns / 32, us per 64 of K, us per tile}; splits: ascending. best: {rows / 32, columns / 32, parts}
int tile_plan(const double* tiles, int n, const int* splits, int n_splits, const double* prices, int64_t M, int64_t N, int64_t K, int cus,
              int* best) {
  const TilePrices& p = *reinterpret_cast<const TilePrices*>(prices);
  double least = INFINITY;
  if (M < 1 || N < 1 || K < 64 || cus < 1) return -1;
  for (int i = 0; i < n; ++i) {
    const int fm = (int)tiles[4 * i], fn = (int)tiles[4 * i + 1];
    const int64_t rows = up(M, 32 * fm), count = rows * up(N, 32 * fn);
    if (32 * fm >= 2 * M + 64) continue;
    const double read = p.x_read * fm + p.w_read * fn / std::sqrt(std::sqrt((double)rows)) + (fm == 3 && fn == 2 ? p.small : 0);
    const double kt = std::fmax(tiles[4 * i + 2], read), per = tiles[4 * i + 3];
    for (int j = 0; j < n_splits; ++j) {
      const int64_t S = splits[j];
      if (S > 1 && (K / S < (int64_t)p.split_k || count * S > (int64_t)p.split_tiles)) break;
      double t = up(count * S, cus) * (up(K / 64, S) * kt + per);
      t += S > 1 ? p.sum + p.part * S + 4 * M * N * S / p.part_bytes : 2 * M * N / p.out_bytes;
      if (t < least) least = t, best[0] = fm, best[1] = fn, best[2] = (int)S;
    }
  }
  return least < INFINITY ? 0 : -2;
}

// `pairs` rows among E experts' [N, K] weights: the tiles counted at n_q quantiles of an expert's rows, avg (1 + quantile)
int grouped_plan(const double* tiles, int n, const double* quantiles, int n_q, int64_t pairs, int64_t E, int64_t N, int64_t K, int cus,
                 int* best) {
  double least = INFINITY;
  if (pairs < 1 || E < 1 || N < 1 || K < 64 || cus < 1) return -1;
  const double avg = (double)pairs / E;
  for (int i = 0; i < n; ++i) {
    const int fm = (int)tiles[4 * i], fn = (int)tiles[4 * i + 1];
    double high = 0;
    for (int j = 0; j < n_q; ++j) high += std::ceil(std::fmax(1.0, avg + quantiles[j] * avg) / (32 * fm));
    const double count = E * high / n_q * up(N, 32 * fn);
    const double t = std::ceil(count / cus) * (K / 64.0 * tiles[4 * i + 2] + tiles[4 * i + 3]);
    if (t < least) least = t, best[0] = fm, best[1] = fn;
  }
  return least < INFINITY ? 0 : -2;
}

}  // namespace xgm
