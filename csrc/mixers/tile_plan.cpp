// The tile and the parts of K of a product on tile_linear.hip: every form of the kernel is priced, the cheapest wins (the first of
// equals). Prompt steps rarely have the row count of the one before, so the search runs for every product of nearly every step: in
// Python it took 20 to 140 us a product, here 2 with the call; a step of a new row count, Dofivik "1b", 80 to 130 rows, 1886 -> 1733 us
// until its end, Loluzen 1216 -> 1177, Vizonex 1142 -> 1027. The prices and the rules around them are ops/tile_linear.py's.
#include <cmath>
#include <cstdint>

namespace xgm {

struct TilePrices {   // ops/tile_linear.py's, in this order
  double launch, sum, w_bytes, part_bytes, out_bytes, overlap, split_k, split_tiles;
};

static int64_t up(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The shorter of products and weight stream stays visible in part.
static double overlapped(const TilePrices& p, double work, double load) {
  return work > load ? work + p.overlap * load : load + p.overlap * work;
}

// tiles: n rows of {rows / 32, columns / 32, us per 64 of K, us per tile}; splits: ascending. best: {rows / 32, columns / 32, parts}
int tile_plan(const double* tiles, int n, const int* splits, int n_splits, const double* prices, int64_t M, int64_t N, int64_t K, int cus,
              int* best) {
  const TilePrices& p = *reinterpret_cast<const TilePrices*>(prices);
  double least = INFINITY;
  if (M < 1 || N < 1 || K < 64 || cus < 1) return -1;
  for (int i = 0; i < n; ++i) {
    const int fm = (int)tiles[4 * i], fn = (int)tiles[4 * i + 1];
    const double kt = tiles[4 * i + 2], per = tiles[4 * i + 3];
    // (many small tiles read the weights and rows more often than this counts: those of 64 columns only while the chip holds
    // them all, 512 x 2048 x 2048 11.7 us against 15.6 with 128 columns)
    const int64_t count = up(M, 32 * fm) * up(N, 32 * fn);
    if (32 * fm >= 2 * M + 64 || (fn == 2 && M > 400 && count > cus) || (fm <= 4 && fn == 4 && M > 2600)) continue;
    for (int j = 0; j < n_splits; ++j) {
      const int64_t S = splits[j];
      if (S > 1 && (K / S < (int64_t)p.split_k || count * S > (int64_t)p.split_tiles)) break;
      const double work = up(count * S, cus) * (up(K / 64, S) * kt + per), load = 2 * N * K / p.w_bytes;
      double t = p.launch + overlapped(p, work, load);
      t += S > 1 ? p.sum + 4 * M * N * S / p.part_bytes : 2 * M * N / p.out_bytes;
      if (t < least) least = t, best[0] = fm, best[1] = fn, best[2] = (int)S;
    }
  }
  return least < INFINITY ? 0 : -2;
}

// `pairs` rows among E experts' [N, K] weights: the tiles counted at n_q quantiles of an expert's rows, avg (1 + quantile)
int grouped_plan(const double* tiles, int n, const double* quantiles, int n_q, const double* prices, int64_t pairs, int64_t E, int64_t N,
                 int64_t K, int cus, int* best) {
  const TilePrices& p = *reinterpret_cast<const TilePrices*>(prices);
  double least = INFINITY;
  if (pairs < 1 || E < 1 || N < 1 || K < 64 || cus < 1) return -1;
  const double avg = (double)pairs / E;
  for (int i = 0; i < n; ++i) {
    const int fm = (int)tiles[4 * i], fn = (int)tiles[4 * i + 1];
    double high = 0;
    for (int j = 0; j < n_q; ++j) high += std::ceil(std::fmax(1.0, avg + quantiles[j] * avg) / (32 * fm));
    const double count = E * high / n_q * up(N, 32 * fn);
    const double work = std::ceil(count / cus) * (K / 64.0 * tiles[4 * i + 2] + tiles[4 * i + 3]), load = 2 * E * N * K / p.w_bytes;
    const double t = overlapped(p, work, load);
    if (t < least) least = t, best[0] = fm, best[1] = fn;
  }
  return least < INFINITY ? 0 : -2;
}

}  // namespace xgm
