// The rules by which a step's operations choose their kernels: how many slices of K, how many keys a wave, how many
// ranges of keys a tile.  The same rules as the Python wrappers of the kernels (allpaca_amd/kernels/tuned.py), where
// each is explained with what was measured; tests/test_dispatch_rules.py holds the two against each other.
#pragma once
#include <algorithm>
#include <cmath>

namespace apc_rules {

constexpr int SKINNY_MAX_ROWS = 16;
constexpr int ROWS_MAX = 64;        // the kernel that finishes in one launch
constexpr int SPLITK_MAX_ROWS = 128;
constexpr int MANY_ROWS_SPLIT_MAX = 1024;
constexpr int WHOLE_WAVES = 4;
constexpr int CHIP_UNITS = 256;     // compute units the rules below were measured on

inline long cdiv(long a, long b) { return (a + b - 1) / b; }

inline int k_split(int M, int N, int K) {  // 17..128 rows: about 240 blocks in all
  const long blocks = cdiv(N, 128) * cdiv(M, 128);
  const int s = (int)std::max(1L, std::min(12L, (long)std::nearbyint(240.0 / (double)blocks)));  // half to even
  return std::max(1, std::min(s, K / 256));
}

inline int k_split_many_rows(int M, int N, int K) {  // 129..1024 rows
  const long blocks = cdiv(N, 128) * cdiv(M, 128);
  int s;
  if (blocks <= 56) s = 5;
  else if (blocks <= 68) s = 4;
  else if (blocks <= 88) s = 3;
  else if (blocks <= 208 && !(blocks >= 150 && N > K)) s = 2;
  else s = 1;
  return std::max(1, std::min(s, K / 256));
}

// gemm_direct_bf16.hip with K in slices, up to 1,024 rows: the bands of 16 outputs that a wave takes, and the microseconds
// of 4,096 columns of K a slice.  A tile's slices all go to one XCD of 32 compute units, so a launch has as many rounds as the
// busiest XCD: 896 rows into 6,144 outputs in three slices are 252 blocks of 8 bands, but 33 on an XCD, which take two
// rounds; 504 blocks of 4 bands fill the two (K 5,376: 111 and 78 us).  A round that is not full takes less, its blocks
// share the L2 with fewer.  Against 2,700 products of 257 to 1,024 rows the time is off by 5.5 % (root mean square).
struct DirectSlices {
  int bands;
  double us;
};
inline DirectSlices direct_slices(int M, int N, int k_split) {
  DirectSlices best{0, 0.0};
  for (int nf : {3, 4, 5, 6, 8}) {
    const long tiles = cdiv(M, 128) * cdiv(N, 64 * nf), rounds = cdiv(cdiv(tiles, 8) * k_split, CHIP_UNITS / 8);
    const double us = rounds * (12.0 + nf * (7.5 + 3.8 * (double)(tiles * k_split) / (double)(rounds * CHIP_UNITS)));
    if (!best.bands || us <= best.us) best = {nf, us};
  }
  return best;
}

// 129..1024 rows: slices of K, and whether the kernel without weights in LDS takes them (tuned._slices_many_rows says what
// it rests on).  Expected microseconds:
struct Slices {
  int k_split;
  bool direct;
};
constexpr int DIRECT_SLICES_MIN_ROWS = 257, DIRECT_MIN_ROWS = 1024;
inline double outputs_us(int M, int N) { return (double)M * N / 1048576.0; }
inline double direct_slices_us(int M, int N, int K, int s) {
  return direct_slices(M, N, s).us * (K / (4096.0 * s)) + 8.0 + (1.5 * s + 0.7) * outputs_us(M, N);
}
inline double tiled_slices_us(int M, int N, int K, int s) {
  const long columns = cdiv(N, 128), blocks = cdiv(M, 128) * columns * s, full = (blocks - 1) / 512, rest = blocks - 512 * full;
  const double first = (double)std::min(rest, (long)CHIP_UNITS) / CHIP_UNITS;
  double us = 64.5 * full + (rest > CHIP_UNITS ? 48.7 : 27.3) + 12.6 * first;
  if (columns % 8) us *= 1.0 + 0.23 * std::min(blocks, (long)CHIP_UNITS) / CHIP_UNITS;
  return us * (K / (4096.0 * s)) + 8.6 + (1.6 * s + 0.3) * outputs_us(M, N);
}
inline double whole_us(int M, int N, int K) {
  const long tiles = cdiv(M, 128) * cdiv(N, 128);
  if (M < DIRECT_MIN_ROWS && tiles <= CHIP_UNITS) return 11.0 + (30.5 + 9.0 * tiles / CHIP_UNITS) * (K / 4096.0);
  return 12.0 + direct_slices(M, N, 1).us * (K / 4096.0);
}
inline Slices slices_many_rows(int M, int N, int K) {
  Slices best{k_split_many_rows(M, N, K), false};
  if (M < DIRECT_SLICES_MIN_ROWS || M > MANY_ROWS_SPLIT_MAX || K % 128 || N % 4) return best;
  double least = 0.96 * (best.k_split == 1 ? whole_us(M, N, K) : tiled_slices_us(M, N, K, best.k_split));
  if (best.k_split > 1 && whole_us(M, N, K) < least) best = {1, false}, least = whole_us(M, N, K);
  for (int s : {2, 3, 4, 6, 8}) {
    if (K % (128 * s) || K < 256 * s) continue;
    const double us = direct_slices_us(M, N, K, s);
    if (us < least) best = {s, true}, least = us;
  }
  return best;
}

inline int tiled_k_split(int M, int N, int K, bool gated = false) {
  if (M <= SPLITK_MAX_ROWS) return k_split(M, N, K);
  if (M > MANY_ROWS_SPLIT_MAX) return 1;
  return gated ? k_split_many_rows(M, N, K) : slices_many_rows(M, N, K).k_split;
}

// Products of 17 to 64 rows: bands of 16 outputs a block of gemm_rows_bf16.hip takes, or 0 where the tiled kernel is expected
// to be faster.  Microseconds, N the width of each matrix of a gated product.  Fitted to 6,134 products (17 to 64 rows, K 1,024
// to 14,336, 320 to 32,000 columns; off by 6 to 8 %, root mean square): of 1,988 sizes what is chosen takes 0.86 of the tiled
// kernel's time in the mean and 1.07 at worst.
//  * gemm_rows_bf16.hip: every block reads its bands' weights and all activations, and a round has a fixed part.  32 rows,
//    K 8,192, q, k and v of 640 columns are 20 blocks that each read a megabyte: 22 us, and 13 in slices on the tiled kernel.
//  * The tiled kernel: steps of 64 columns, two blocks a unit, the slices through memory and a second kernel.  With columns
//    enough it needs neither slices nor that kernel: 64 rows, K 1,024, SwiGLU of 14,336 15 us there, 19 in two rounds here.
enum RowsKind : int { ROWS_PLAIN = 0, ROWS_GATED = 1, ROWS_QKV = 2 };
inline double rows_us(int M, int N, int K, int bands, int kind, long* rounds) {
  const long blocks = cdiv(N / 16, kind == ROWS_GATED ? bands / 2 : bands), r = cdiv(blocks, CHIP_UNITS);
  const double fill = (double)blocks / (double)(r * CHIP_UNITS), tiles = M / 16.0;
  *rounds = r;
  return 3.8 + 3.0 * (r - 1) + r * (K / 1024.0) * (bands * (0.56 + 0.58 * fill) + 0.5 * tiles - (bands == 1 ? 0.37 : 0.25)) +
         (kind == ROWS_QKV ? 0.58 : 0.1) * tiles;
}
inline double tiled_rows_us(int M, int N, int K, int kind) {
  const int columns = kind == ROWS_GATED ? 2 * N : N, s = k_split(M, columns, K);
  const double steps = (double)cdiv(K / 64, s), full = (double)(cdiv(columns, 128) * s) / CHIP_UNITS;
  double us = 4.5 + steps * (0.33 + 0.32 * full + (full > 1.0 ? 0.33 : 0.0));
  if (s > 1) us += 3.2 + 2.0e-6 * s * M * (double)columns;
  if (kind == ROWS_GATED) us += 0.5;
  if (kind == ROWS_QKV) us += s > 1 ? 0.4 : 9.0;   // K whole: rotation and cache write in a kernel of their own
  return us;
}
inline int rows_bands(int M, int N, int K, int kind) {
  if (cdiv(M, 16) * 16 * (long)K > 1L << 18) return 0;   // beyond, 17 rows, K 11,008 into 320 to 1,280 columns: up to 1.27 of the tiled kernel's time
  int best = 0;
  double least = tiled_rows_us(M, N, K, kind);
  for (int bands : {1, 2, 4}) {
    if ((kind == ROWS_GATED && bands == 1) || (kind == ROWS_QKV && bands != 2)) continue;
    long rounds;
    const double us = rows_us(M, N, K, bands, kind, &rounds);
    // rounds further on overlap less than expected: 17 rows, K 4,096 into 32,000 columns 53 us, tiled 47
    if (us < least && (rounds == 1 || rounds * K <= (kind == ROWS_PLAIN ? 4096 : 2048))) best = bands, least = us;
  }
  return best;
}

// sums of x^2 a row that the products behind a norm take
inline int ss_parts_max(int M) { return M <= ROWS_MAX ? 1024 : 256; }

// ranges that the decode kernel cuts every row's keys into (the kernel sizes them from the row's own length)
inline int decode_parts(long pairs, int span) {
  const long per_pair = std::max(1L, (long)CHIP_UNITS / std::max(1L, pairs));
  return (int)std::max(1L, std::min((long)WHOLE_WAVES * per_pair, cdiv(span, 64)));
}

// whether a decode step's rows go to the kernel that may share out their work over all waves: enough pairs that no pair
// would be cut for its own sake (where a block has no room for a pair of its own: so many that shares are sure to pay), no
// more than there are counters for, and a longest row that could be far longer than the others
constexpr int EVEN_MAX_PAIRS = 4096, EVEN_ALONE_MIN_PAIRS = 1024;
inline bool decode_even(long pairs, int span, bool pair_fits, int min_pairs, int min_span) {
  return pairs >= (pair_fits ? min_pairs : std::max(min_pairs, EVEN_ALONE_MIN_PAIRS)) && pairs <= EVEN_MAX_PAIRS && span > min_span;
}

// Whether shares beat a block a pair for the lengths at hand (tuned._even_pays says what it rests on).  steps: of 32 keys,
// over all rows; longest: of the longest row
inline bool even_pays(long long steps, int longest, int n_rows, int tiles, int window) {
  if (window) {
    const int most = window / 32 + 1;
    longest = std::min(longest, most);
    steps = std::min(steps, (long long)n_rows * most);
  }
  const int waves = std::max(1, CHIP_UNITS / tiles) * WHOLE_WAVES;
  const double units = (double)n_rows * WHOLE_WAVES / waves, share = (double)(steps + 2LL * n_rows) / waves;
  const double whole = std::max(1.03 * share + 2.5 + 1.1 * units, 4.1 + 0.245 * longest * std::min(std::ceil(units), 2.8));
  return 7.3 + std::max(share, 8.3) + 0.05 * (n_rows / 64.0) < whole;
}

// Whether a step's decoded rows go into the launch of its tiles of prompt rows (attn_prefill_wide_kernel), behind them.  There a
// decode block has a unit of its own where two share one in a launch of their own (heads of 128; two and four with heads of 64), which
// matters once they are many, and where the tiles fill whole rounds a round of them only waits.  tile_blocks: the tiles' blocks; pairs:
// (row, kv head) pairs with a block each, or `last`: blocks for ranges of their keys, a round of the chip at most.  One layer, two launches /
// one, us, 32 heads over 8 of 128: 504 rows behind 1,544 beside 32 rows of 1,000 keys 63 / 41, 128 of 1,000 125 / 107, 256 of 100 68 / 60;
// 1,024 rows (a whole round) beside 8 of 2,000 (last) 45 / 42, 32 of 2,000 72 / 75, 64 112 / 117, 256 of 100 55 / 65; 70 rows beside 64 of 1,000
// 59 / 53, 256 of 100 40 / 44.  Over 1,976 steps (70 to 1,900 prompt rows beside 1 to 256, five pairs of heads) what is chosen takes 0.797 of
// the two launches' time in the mean and 1.008 at worst (always one 0.792 and 1.17, the better of the two 0.791).
inline bool decode_beside_tiles(long tile_blocks, int d, long pairs, bool last) {
  const long round = CHIP_UNITS * (d <= 64 ? 2 : 1), free = (round - tile_blocks % round) % round;
  return last || pairs < CHIP_UNITS || (pairs <= 1024 && free * 16 > round);
}

// ranges of keys that the 128-row attention kernel cuts every tile of a step into; `keys`: of the longest prompt
inline int key_splits(int n_tiles, int n_heads, int keys, int window, int splits_max, int range_min) {
  const long blocks = (long)n_tiles * n_heads;
  if (!splits_max || blocks <= 0 || keys <= 0) return 1;
  if (window) keys = std::min(keys, window + 128);
  const long few = std::min((long)keys / std::max(1, range_min / 2), (long)(CHIP_UNITS / 2) / blocks);
  const long s = std::min({(long)splits_max, (long)CHIP_UNITS / blocks, std::max((long)keys / range_min, few)});
  return (int)std::max(1L, s);
}

// the same from a model of the launch's time (tuned._key_splits_by_time says what it rests on).  passes: of 64 keys, over
// all tiles; rows: of the step
constexpr double KEY_PARTS_MAX = 268435456.0;   // bytes of partial results
inline int key_splits_by_time(int n_tiles, int rows, int n_heads, int d, long long passes, int window, int splits_max) {
  const long blocks = (long)n_tiles * n_heads;
  double mean = (double)passes / n_tiles;
  if (window) mean = std::min(mean, (double)(cdiv(window, 64) + 2));
  int best = 1;
  double best_us = 1e30;
  for (int s = 1; s <= std::max(1, splits_max); ++s) {
    if (s > 1 && (double)s * rows * n_heads * (d + 2) * 4.0 > KEY_PARTS_MAX) break;
    const long unit = cdiv(blocks * s, CHIP_UNITS);   // blocks of the busiest compute unit
    const double q = mean / s;
    double us = d <= 64 ? (unit / 2) * (6.0 + 1.15 * q) + (unit % 2) * (6.0 + 0.66 * q) : unit * (12.5 + 0.8 * q);
    if (s > 1) us += (d <= 64 ? 5.0 : 12.0) + (double)s * rows * n_heads * (d + 2) * 8.0 / 6e6;
    if (s == 1) best_us = 0.97 * us;                  // (cut only where it is worth something)
    else if (us < best_us) best = s, best_us = us;
  }
  return best;
}

}  // namespace apc_rules
