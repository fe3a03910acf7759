// Which kernel a projection's product goes to, in which tiles and pieces: rules on its kind, sizes and row pitches alone.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>
#include <utility>

#include "../../include/picotron_amd.h"

namespace {

// row-major products: a @ b^T, a @ b, a^T @ b
enum class Product { NT, NN, TN };
struct ProductSizes {
  int64_t M, N, K, lda, ldb;   // lda, ldb: elements between the rows of a and b as they lie in memory
};

// How much of the GPU's 256 CUs a product keeps busy, over the library's tile shapes (256 x 256 and narrower ones, which run
// at the given share of its rate): output / (waves of workgroups x tile).
double tile_fit(int64_t M, int64_t N) {
  double best = 0;
  for (auto [side, rate] : {std::pair<int64_t, double>(256, 1.0), {192, 0.97}, {160, 0.95}, {128, 0.85}})
    for (auto [m, n] : {std::pair<int64_t, int64_t>(side, 256), {256, side}}) {
      const int64_t waves = (((M + m - 1) / m) * ((N + n - 1) / n) + 255) / 256;
      best = std::max(best, rate * M * N / (256.0 * waves * m * n));
    }
  return best;
}

// Into how many pieces the contraction is cut (1: not at all).  The library works on output tiles and walks the whole
// contraction in each, so a product of few tiles and a long contraction -- the input gradient of the vocabulary projection
// or of gate / up, weight gradients of a small model -- leaves most of the GPU idle: [512 x 49152] @ [49152 x 576] took
// 143 us and takes 53 us in 16 pieces, [2048 x 21760] @ [21760 x 4096] 447 and 291 us in two.  The pieces cost 8 bytes of
// fp32 traffic per output element each, hence the lower bound on a piece's length and, as output grows, on its ratio to
// the number of tiles.  The lines lie where sweeps over 100 .. 8192 rows, 192 .. 4096 columns and contractions of 4096 ..
// 49152 crossed, on the side where no class loses: of 2400 drawn products the 548 that are cut took 0.54 (NN), 0.82 (NT) and
// 0.74 (TN) of the library's time in the geometric mean, four over 1.06 (1.25 at most: [1076 x 49152] @ [49152 x 3072]).
// Products of the forward's layout (NT), the library's best, gain only from 8192 on; up to 32 tiles in pieces of 1024 ([128 x
// 2048] of 8192 17.2 us whole, 22.1 in two, 14.9 in eight), up to 56 of 2048, and at 57 .. 64 not where the library's own
// split fills the GPU ([512 x 2048] of 8192 27 us, 28.7 in two; [256 x 4096] of 10880 1.23 times).
// More than 256 tiles and a contraction from 16384 on (NN): the library is fast where one of its tile shapes fills the CUs
// evenly ([5120 x 49152] @ [49152 x 2048]: 1200 TFLOP/s) and at half that rate elsewhere ([4500 x 49152]: 620, in four
// pieces 1150).  Contractions under 24576 are never faster in four pieces than in two, and two of 129 .. 192 tiles fill two waves of
// workgroups badly ([5465 x 16384] @ [16384 x 2048] 286 us, in two 316, in four 440; [4096 x 16384] @ [16384 x 2048] 255 and 230);
// two of a longer one have to fill the GPU well ([3200 x 32000] @ [32000 x 2048] 395, in two 522, in four 376).
int64_t contraction_parts(Product kind, int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
  if ((M * N) % 8) return 1;   // (pico_sum_parts moves 8 elements at a time)
  auto cuts = [&](int64_t parts) { return K % parts == 0 && (K / parts) % 32 == 0; };
  int64_t most = 1, piece = 0;
  if (kind == Product::NN && tiles > 256) {
    if (K < 16384 || tile_fit(M, N) >= 0.88) return 1;
    const int64_t t256 = ((M + 255) / 256) * ((N + 255) / 256);
    if (K < 24576) return cuts(2) && (t256 <= 128 || t256 > 192) ? 2 : 1;
    int64_t best = 1;
    double least = 1.8;   // (of the ideal time)
    for (int64_t parts : {2, 4}) {
      if (!cuts(parts)) continue;
      const int64_t waves = (t256 * parts + 255) / 256;
      const double cost = waves * 256.0 * 65536 / (static_cast<double>(M) * N * parts) + 1040.0 * parts / K;
      if (cost < least && (parts > 2 || cost < 1.28)) {   // (two half-filled waves: 956 us at [6145 x 32000], 792 in four pieces)
        least = cost;
        best = parts;
      }
    }
    return best;
  }
  if (kind == Product::NN && K >= 5120) {
    // (narrow outputs of the vocabulary's contraction: [4608 x 49152] @ [49152 x 768] 432 us, in four 540, in eight 346)
    most = std::min<int64_t>(16, (N < 1024 && N % 256 == 0 && K >= 40000 && tiles > 128 ? 2048 : 1024) / tiles);
    piece = std::max<int64_t>(1280, 16 * tiles);
  } else if (kind == Product::TN && K >= 4096) {
    most = tiles < 256 ? std::min<int64_t>(K >= 16384 ? 4 : 2, 512 / tiles) : 1;
    piece = 2048;
  } else if (kind == Product::NT && K >= 8192) {
    const bool whole = K < 10240 || (M % 256 == 0 && K < 12288);   // (57 .. 64 tiles)
    most = tiles <= 32 ? 8 : tiles <= 56 || (tiles <= 64 && !whole) ? 4 : tiles > 64 && tiles <= 128 ? 2 : 1;
    piece = tiles <= 32 ? 1024 : tiles <= 56 ? 2048 : 4096;
  }
  int64_t parts = 1;
  while (2 * parts <= most && cuts(2 * parts) && K / (2 * parts) >= piece) parts *= 2;
  return parts;
}

// Which operand of a weight gradient (a^T b, both with the contraction as their slow axis) is transposed first, 1: a, 2: b, 0:
// none.  The library runs the product at 1000 - 1100 TFLOP/s as it is and 13 % faster where one operand has the contraction
// as its fast axis, and the narrower operand is small beside the work: [4096 x 49152]^T [4096 x 2048] 732 -> 616 us, the
// transposition included, [4096 x 16384]^T [4096 x 2048] 227 -> 202, [4096 x 49152]^T [4096 x 576] 289 -> 229.  The gain is
// proportional to the wider side and to the narrower operand's size, the transposition to the latter plus a launch: the line
// lies where a sweep over contractions of 512 .. 8192 crossed ([4096 x 6144]^T [4096 x 2048]: 88 and 89 us).  Under 1024 rows
// the product is bound by writing the result unless the narrower side leaves the library's tiles half empty.
// (Transposing the wider operand too costs more than the second 13 %.)
// The library runs the transposed layout in tiles of 256 x 256.  With fewer than 384 of them its gain depends on how they fill
// the GPU, unless one side is the vocabulary's: over 330 its other layout has better tiles ([4096 x 10880]^T [4096 x 2048] 172
// us, transposed 273), up to 330 it wins outside 1152 .. 2048 rows ([1280 x 12288]^T [1280 x 1536] 64, 73; from 4096 rows 166,
// 159), up to 256 from 1536 rows on ([4096 x 8192]^T [4096 x 2048] 124, 112), up to 230 with longer contractions and a side of
// 8192 at least ([3266 x 9216]^T [3266 x 1152] 0.82 times, [2944 x 8192]^T [2944 x 1024] 1.03).  Short contractions that are no
// multiple of its step of 64 lose ([1262 x 12288]^T [1262 x 4096] 1.06 times).  Of 212 drawn products that are transposed ten took
// over 1.04 of the library's time and none over 1.13, 0.91 in the geometric mean.
int64_t turned_operand(Product kind, const ProductSizes& n) {
  if (kind != Product::TN) return 0;
  const auto [M, N, K, lda, ldb] = n;
  const int64_t narrow = std::min(M, N), wide = std::max(M, N);
  if (narrow % 8 || (M < N ? lda : ldb) % 8 || (K < 1024 && (K < 768 || narrow >= 1024))) return 0;
  if (wide <= 5000 + 1e10 / (static_cast<double>(K) * narrow)) return 0;
  const int64_t t256 = ((M + 255) / 256) * ((N + 255) / 256);
  const bool vocabulary = wide >= 24576;
  if (K % 64 && K < 1408 && t256 < 1024) return 0;
  if (t256 <= 230 && !vocabulary && (wide < 8192 || K < (t256 > 160 ? 3072 : 4800))) return 0;
  if (t256 > 230 && t256 <= 256 && !vocabulary && K < (K % 64 ? 2048 : 1536)) return 0;
  if (t256 > 256 && t256 <= 330 && K > 1152 && K < 2048) return 0;
  if (t256 > 330 && t256 < 384 && !vocabulary && K > 1024) return 0;
  return M < N ? 1 : 2;
}
// Whether a product goes to the package's own kernel (pico_product), with tiles of which side and how many groups of waves
// (0: no).  It wins where the library's tiles leave most CUs idle, until either there are more tiles than CUs -- the
// library's larger ones then do more per byte -- or the walk along the contraction is so long that its steps, and not its
// start, are the time.  Weight gradients (TN, the library's slowest layout) stay with it longest.  Library and own kernel, us:
//   TN, tiles of 64 while they are at most 256, or 512 and the walk short: [512 x 960]^T [512 x 576] 9.2, 6.0;
//      [2331 x 1024]^T [2331 x 1024] 24, 15; [3072 x 576] from 1024 rows 14.2, 13.1, from 4096 35, 37;
//   TN, up to 256 tiles of 128, two groups: [2048 x 2048] from 512 rows 13.6, 11.3, from 4096 49, 42; [3072 x 1024] from 2630
//      41, 27; [1024 x 2688] from 4096 41, 40, from 8192 70, 76;
//   TN, more tiles of 128: few rows.  [49152 x 576] from 512 69, 48 (pico_product_large 40), from 1024 93, 89.  The library runs an even number of
//      its tiles side by side best and a ragged contraction a quarter slower: [32000 x 1024] from 512 46, 48, but [32000 x
//      1152] 61, 50 and [8192 x 1024] from 443 20, 14;
//   NN: [512 x 1024] @ [1024 x 1024] 9.2, 7.4; [512 x 3072] @ [3072 x 576] 17.0, 14.2; [512 x 2048] @ [2048 x 2048] 15, 12;
//      tiles of 128: [4096 x 1536] @ [1536 x 1024] 21, 19, but with 512 of them [4096 x 2048] @ [2048 x 2048] 37, 41;
//   NT, its best: [512 x 1024] @ [1024 x 1024]^T 8.4, 6.8; [512 x 1536] @ [1536 x 576]^T 8.4, 8.8.
// Over 2400 drawn products of 100 .. 8192 rows, 192 .. 49152 columns and contractions of 100 .. 49152 the time over the
// library's was, where these lines choose the kernel, 0.75 (NN, 211 products), 0.81 (NT, 115) and 0.70 (TN, 316) in the geometric
// mean and 1.04 at most.  Half of them go to pico_product_mid or pico_product_large, see their rules.
struct OwnProduct {
  int64_t groups, tile;
};
OwnProduct own_product(Product kind, int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64), wide_tiles = ((M + 127) / 128) * ((N + 127) / 128), narrow = std::min(M, N);
  constexpr OwnProduct no = {0, 64};
  if (N % 8 || (kind == Product::TN ? M : K) % 8) return no;
  if (kind == Product::TN) {
    if (tiles <= 256) return K <= 384 ? OwnProduct{1, 64} : K <= 4096 ? OwnProduct{2, 64} : no;
    if (wide_tiles <= 128) return K <= 2560 ? OwnProduct{1, 64} : no;
    if (wide_tiles <= 256) return K <= 384 ? OwnProduct{1, 128} : K <= (wide_tiles >= 230 ? 8192 : 4096) ? OwnProduct{2, 128} : no;
    const int64_t most = narrow % 512 ? (K % 64 ? 1000 : 768) : (K % 64 ? 576 : 320);
    return K <= most && wide_tiles <= 3500 ? OwnProduct{1, 128} : no;
  }
  if (tiles > 512) {
    if (wide_tiles > 256) return no;
    return K <= 600 ? OwnProduct{1, 128} : kind == Product::NN && K <= 4096 ? OwnProduct{2, 128} : no;
  }
  if (tiles > 256) return K <= 600 ? OwnProduct{1, 64} : no;
  if (kind == Product::NN) return K <= (tiles <= 32 ? 1088 : tiles <= 64 ? 2112 : 4096) ? OwnProduct{2, 64} : no;
  return K <= (tiles > 128 ? 3072 : tiles > 60 ? 1088 : 0) ? OwnProduct{2, 64} : no;
}

double last_round(double walk, double end, double used, double walk_idle, double end_idle) {   // (idle: of the time, where few CUs are busy)
  return used > 0 ? walk * (walk_idle + (1 - walk_idle) * used) + end * (end_idle + (1 - end_idle) * used) : 0;
}
// `work` us of products beside a walk through the operands and the result at `rate` TB/s: the longer one, and more where both are long
double with_memory(double work, int64_t M, int64_t N, int64_t K, double rate) {
  const double memory = 2e-6 / rate * (static_cast<double>(M) * K + static_cast<double>(N) * K + static_cast<double>(M) * N);
  return std::sqrt(std::sqrt(work * work * work * work + memory * memory * memory * memory));
}
double own_time(Product kind, OwnProduct own, int64_t M, int64_t N, int64_t K) {
  struct Form {
    int64_t tile, groups;
    double start, trip, end, walk_idle, end_idle;
  };
  static constexpr Form forms[] = {{64, 1, 3.07, 0.26, 0.16, 0.84, 0.00}, {64, 2, 2.12, 0.54, 1.18, 0.86, 0.84},
                                   {128, 1, 3.69, 0.52, 1.36, 1.00, 0.08}, {128, 2, 3.01, 1.14, 2.73, 0.78, 0.30}};
  for (const Form& f : forms) {
    if (f.tile != own.tile || f.groups != own.groups) continue;
    const int64_t tiles = ((M + f.tile - 1) / f.tile) * ((N + f.tile - 1) / f.tile), steps = (K + 63) / 64;
    const double walk = (steps + f.groups - 1) / f.groups * f.trip;
    const double t = f.start + tiles / 256 * (walk + f.end) + last_round(walk, f.end, tiles % 256 / 256.0, f.walk_idle, f.end_idle);
    const double layout = kind == Product::TN ? 1.04 : f.tile == 64 ? (kind == Product::NT ? 0.93 : 1.04) : f.groups == 1 ? 0.95 : 1.0;
    return with_memory(layout * t, M, N, K, 5.3);
  }
  return 0;
}
// The time of pico_product_large, the package's kernel for products that fill the GPU, and the tiles and pieces of the contraction that
// take least.
//
// It follows from the rounds: 256 workgroups take a tile each, a step of 64 of contraction costs 1.1 .. 1.4 us (less while part of the
// GPU idles), a tile's end 2 .. 5 us; and from what is read and written, at 4.4 TB/s.  Unit of all estimates here: a timed call, the
// geometric mean of one with operands from memory and one with operands in the caches, over 1.07, less 3 us that any call shows.
// Over 2900 timed (shape, tiles, pieces) the estimate has an error of 6 % (standard deviation).
struct LargeProduct {
  int64_t tile_m = 0, tile_n = 0, parts = 0;
};
double large_time(int64_t M, int64_t N, int64_t K, LargeProduct& best) {
  struct Form {
    int64_t m, n;
    double step, end;
  };
  static constexpr Form forms[] = {{256, 256, 1.44, 4.6}, {256, 192, 1.31, 4.6}, {192, 256, 1.27, 2.9}, {256, 128, 1.13, 2.7}, {128, 256, 1.09, 1.9}};
  const int64_t steps = (K + 63) / 64;
  double least = 1e30;
  for (const Form& f : forms) {
    const int64_t tiles = ((M + f.m - 1) / f.m) * ((N + f.n - 1) / f.n);
    for (int64_t parts : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32}) {
      if (parts > 1 && (tiles * parts > 300 || steps < 8 * parts)) break;
      const int64_t full = tiles * parts / 256, rest = tiles * parts % 256, length = (steps + parts - 1) / parts;
      const double used = rest / 256.0;   // of the GPU, in the last round
      double t = 3.6 + full * (length * f.step + f.end);
      if (rest) t += length * f.step * (0.7 + 0.3 * used) + f.end * (0.45 + 0.55 * used);
      if (parts > 1) t += 5 + 1e-6 * M * N * (0.84 * parts - 0.4);   // the pieces in fp32, and their sum
      if (t < least) {
        least = t;
        best = {f.m, f.n, parts};
      }
    }
  }
  return with_memory(least, M, N, K, 4.4);
}
// The library's at its best: hardly ever less, 1.0 .. 1.9 times this in the mean of a class of sizes, see library_cost
double other_time(Product kind, int64_t M, int64_t N, int64_t K) {
  struct Form {
    int64_t m, n;
    double step[3];   // NT, NN, TN
  };
  static constexpr Form forms[] = {{256, 256, {1.37, 1.45, 3.0}}, {256, 192, {1.16, 1.2, 2.0}}, {192, 256, {1.16, 1.2, 2.0}}, {256, 128, {0.72, 0.83, 1.7}},
                                   {128, 256, {0.72, 0.83, 1.7}}, {128, 128, {0.41, 0.51, 0.88}}, {64, 128, {0.22, 0.19, 0.27}}, {128, 64, {0.22, 0.19, 0.27}}};
  static constexpr double start[3] = {-1.6, 8.6, 2.2}, end[3] = {8.8, 2.3, 2.4};
  const int k = static_cast<int>(kind);
  double least = 1e30;
  for (const Form& f : forms) {
    const int64_t rounds = (((M + f.m - 1) / f.m) * ((N + f.n - 1) / f.n) + 255) / 256;
    least = std::min(least, rounds * (K / 64.0 * f.step[k] + end[k]));
  }
  return start[k] + least;
}
// (the library takes its largest tiles where their pieces fill the GPU)
bool fills(int64_t M, int64_t N, int64_t parts) { return ((M + 255) / 256) * ((N + 255) / 256) * parts >= 256; }
// The library's time for an input gradient that it would get in `parts` pieces (contraction_parts), at its best: whole tiles of a
// contraction that divides evenly.
double cut_time(int64_t M, int64_t N, int64_t K, int64_t parts) {
  struct Form {
    int64_t m, n;
    double step;
  };
  static constexpr Form forms[] = {{256, 256, 1.44}, {256, 128, 0.71}, {128, 256, 0.71}, {128, 128, 0.35}};
  const bool full = fills(M, N, parts);
  double least = 1e30;
  for (const Form& f : forms) {
    const int64_t rounds = (((M + f.m - 1) / f.m) * ((N + f.n - 1) / f.n) * parts + 255) / 256;
    if (f.m * f.n < 65536 && full) continue;
    least = std::min(least, rounds * (K / 64.0 / parts * f.step + 1.6));
  }
  return 2 + with_memory(least, M, N, K, 6.8) + 1.53e-6 * M * N * parts;
}
// own_product's choice where the kernel takes the operands as they lie in memory; the library takes any row pitch
OwnProduct own_product(Product kind, const ProductSizes& n) {
  const OwnProduct own = own_product(kind, n.M, n.N, n.K);
  if (own.groups > 0 && !pico_product_takes(n.M, n.N, n.K, n.lda, n.ldb, kind == Product::TN, kind != Product::NT)) return {0, 64};
  return own;
}

// The time of pico_product_mid and the tiles that take least (tile_m 0: none).
//
// It follows from the rounds: 256 workgroups take a tile each, a trip (64 of contraction for each group of waves) costs `trip`,
// a tile's start and end `end`, and in the last round both depend on how much of the GPU is busy; reading and writing go on beside, at 4.8 TB/s.
// Over 7000 timed (shape, tiles) the estimate has an error of 4 .. 10 % (standard deviation), small tiles the larger one.
struct MidProduct {
  int64_t tile_m = 0, tile_n = 0, parts = 1;
};
double mid_time(Product kind, int64_t M, int64_t N, int64_t K, MidProduct& best) {
  struct Form {
    int64_t m, n, groups;
    double start, trip[3], end, walk_idle, end_idle;   // (trip: NT, NN, TN)
  };
  static constexpr Form forms[] = {
      {32, 32, 4, 1.89, {0.67, 0.69, 0.87}, 1.14, 0.47, 1.12}, {32, 64, 4, 1.72, {0.83, 0.88, 1.01}, 1.39, 0.64, 1.09},
      {64, 32, 4, 1.71, {0.90, 1.20, 1.12}, 1.33, 0.58, 1.15}, {64, 64, 2, 1.86, {0.52, 0.57, 0.56}, 1.54, 0.80, 0.83},
      {64, 96, 2, 1.84, {0.66, 0.71, 0.68}, 1.76, 0.78, 0.81}, {96, 64, 2, 1.89, {0.73, 0.67, 0.68}, 1.79, 0.82, 0.75},
      {96, 96, 2, 1.84, {0.83, 0.85, 0.88}, 2.18, 0.82, 0.75}, {64, 128, 2, 1.88, {0.81, 0.83, 0.80}, 1.98, 0.84, 0.73},
      {128, 64, 2, 1.94, {0.82, 0.80, 0.87}, 2.01, 0.86, 0.70}, {128, 96, 2, 1.66, {1.20, 1.28, 1.21}, 2.21, 0.71, 0.79},
      {128, 128, 2, 1.98, {1.35, 1.36, 1.23}, 2.68, 0.84, 0.60}, {128, 192, 1, 2.24, {0.79, 0.77, 0.77}, 3.06, 0.90, 0.45},
      {192, 128, 1, 2.52, {0.88, 0.83, 0.84}, 2.85, 0.90, 0.37}, {128, 256, 1, 2.52, {1.03, 0.92, 0.96}, 3.53, 0.89, 0.36}};
  const int64_t steps = (K + 63) / 64;
  double least = 1e30;
  for (const Form& f : forms) {
    const int64_t tiles = ((M + f.m - 1) / f.m) * ((N + f.n - 1) / f.n);
    // (long walks along a slow axis in rows of 64 bytes take up to twice that: [4819 x 232]^T [4819 x 184] 36 us in tiles of 64 x 32, 14 in pieces)
    if (tiles > 1024 || (f.m == 32 && f.n == 32 && steps > 48) || (std::min(f.m, f.n) == 32 && kind != Product::NT && steps > 64)) continue;
    const double walk = (steps + f.groups - 1) / f.groups * f.trip[static_cast<int>(kind)];
    const double t = f.start + tiles / 256 * (walk + f.end) + last_round(walk, f.end, tiles % 256 / 256.0, f.walk_idle, f.end_idle);
    if (t < least) {
      least = t;
      best = {f.m, f.n, 1};
    }
  }
  return with_memory(least, M, N, K, 4.8);
}
// The same for a contraction that is cut into pieces, one round of workgroups of one piece each, and the pieces' sum: 6 .. 7 % error over
// 2100 timed (shape, tiles, pieces).  (1.5 us of it are for the second launch, which costs more where the operands are in the caches.)
double mid_parts_time(int64_t M, int64_t N, int64_t K, MidProduct& best) {
  struct Form {
    int64_t m, n, groups;
    double start, trip, end, walk_idle, end_idle;
  };
  static constexpr Form forms[] = {
      {64, 96, 2, 5.19, 0.69, 2.25, 0.78, 0.81}, {64, 128, 2, 5.23, 0.82, 2.54, 0.84, 0.73}, {96, 96, 2, 5.19, 0.85, 2.80, 0.82, 0.75},
      {128, 128, 2, 5.33, 1.27, 3.43, 0.84, 0.60}, {128, 192, 1, 5.59, 0.72, 3.92, 0.90, 0.45}, {192, 128, 1, 5.87, 0.70, 3.66, 0.90, 0.37},
      {128, 256, 1, 5.87, 0.83, 4.53, 0.89, 0.36}};
  const int64_t steps = (K + 63) / 64;
  double least = 1e30;
  for (const Form& f : forms) {
    const int64_t tiles = ((M + f.m - 1) / f.m) * ((N + f.n - 1) / f.n), most = 256 / tiles;
    for (const int64_t wanted : {most, 2 * most / 3, most / 2}) {
      const int64_t parts = std::min<int64_t>({wanted, 64, steps / 2});
      if (parts < 2) continue;
      const double walk = ((steps + parts - 1) / parts + f.groups - 1) / f.groups * f.trip;
      const double t = f.start + last_round(walk, f.end, tiles * parts / 256.0, f.walk_idle, f.end_idle) + 1e-6 * M * N * (1.82 * parts - 1.13);
      if (t < least) {
        least = t;
        best = {f.m, f.n, parts};
      }
    }
  }
  return with_memory(least, M, N, K, 4.6);
}
// The route of a product: the library whole or in `parts` pieces of the contraction, with operand `turn` (1: a, 2: b) transposed first;
// pico_product (a square tile, groups), pico_product_mid or pico_product_large (tiles, pieces).
struct ProductRoute {
  enum Kernel { Library, Own, Mid, Large } kernel = Library;
  int64_t tile_m = 0, tile_n = 0, groups = 0, parts = 1, turn = 0;
};
// What the library promises for a product: what it took, over its time at its best, where the package's kernels were as fast, by classes of sizes.  Its
// choice of tiles is not monotone in any size, and it has few kernels for contractions that are no multiple of 64 and for rows that are no whole lines
// (over other_time: NN 1.0 and 1.3, NT 1.0 and 1.35; in pieces, over cut_time, 1.3 and 1.9), so a class spreads over 12 .. 28 %.  Forward products with much
// work are its best: there the line is on its side ([4096 x 4096] @ [4096 x 4096]^T 93 us, pico_product_large 103; [4096 x 2048] @ [16384 x 2048]^T 192, 206),
// but for short contractions ([3832 x 512] @ [49152 x 512]^T 315, 218).  A vocabulary's logits of up to 768 columns leave always ([680 x 576] @ [32000 x
// 576]^T 57 -> 29), unless they are short (256) and their rows no whole lines ([6912 x 192] @ [73448 x 192]^T 433, 523).  Weight gradients are its slowest
// layout, unless an operand is transposed first.
double library_cost(Product kind, const ProductSizes& n, int64_t parts, int64_t turn) {
  const auto [M, N, K, lda, ldb] = n;
  const bool odd_k = K % 64 != 0, odd_n = N % 64 != 0;
  if (parts > 1 && kind == Product::NN) {
    const bool few = ((M + 127) / 128) * ((N + 127) / 128) * parts <= 256;
    return (K / parts % 64 != 0 ? 1.6 : odd_n ? 1.55 : N % 256 != 0 ? 1.45 : few ? 1.6 : fills(M, N, parts) ? 1.0 : 1.15) * cut_time(M, N, K, parts);
  }
  const double whole = other_time(kind, M, N, K);
  if (kind == Product::TN && turn != 0) return (odd_k ? 1.15 : odd_n ? 1.1 : std::min(M, N) < 256 ? 1.1 : 0.75) * whole;
  if (kind == Product::TN) return 1.5 * whole;
  const double gflop = 2e-9 * M * N * K;
  if (kind == Product::NT && N >= 24576 && K <= 768) return (odd_n && K <= 256 ? 0.65 : 2) * whole;
  if (kind == Product::NT) return (odd_k ? (gflop >= 40 ? 1.25 : 1.5) : K <= 800 && gflop >= 16 ? 1.2 : odd_n ? (gflop >= 40 ? 1.05 : 1.2) : gflop >= 40 ? 0.9 : 1.0) * whole;
  return (odd_k ? 1.45 : odd_n ? 1.35 : K % 1024 != 0 ? 1.25 : 1.2) * (K >= 24576 ? 1.25 : 1.0) * whole;
}
// The kernel that promises least.  (Lines that compared the kernels in pairs, with a margin each, sent products past kernels that the next pair would have
// taken: [1025 x 32000] @ [32000 x 336] 54 us in pico_product_large, 104 in the library's pieces.)  Of 4958 products of drawn
// layers (64 .. 8192 rows, 64 .. 4096 columns, up to 22016 on the other side, four vocabularies) the choice takes 1.019 of the fastest kernel's time in the
// geometric mean and 0.823 of the time without pico_product_mid and pico_product_large; 100 are over 1.05 of that, 1.22 at most.  With and without, us:
//   NT: 0.81 of the library's time in pico_product_large, 0.71 in pico_product_mid ([2331 x 1536] @ [576 x 1536]^T 12.0 -> 9.5);
//   NN: 0.81 in pico_product_large ([2242 x 10880] @ [10880 x 4096] 248 -> 178; in pieces [4096 x 49152] @ [49152 x 2048] 663 -> 635), 0.67 in pico_product_mid ([2331
//     x 3072] @ [3072 x 576] 27.7 -> 15.8; [145 x 49152] @ [49152 x 576] 37 -> 23), 0.93 of pico_product's ([512 x 3072] @ [3072 x 576] 12.9 -> 8.7);
//   TN: 0.80 in pico_product_large ([4096 x 4096]^T [4096 x 4096] 137 -> 103), 0.63 in pico_product_mid; 0.88 of pico_product's ([451 x 9792]^T [451 x 3264] 49.7 -> 38.8; [2331 x 3072]^T [2331 x 576] 23.7 -> 15.8).
ProductRoute choose_route(Product kind, const ProductSizes& n) {
  const auto [M, N, K, lda, ldb] = n;
  const int a_slow = kind == Product::TN, b_slow = kind != Product::NT;
  const OwnProduct own = own_product(kind, n);
  ProductRoute route;
  double least;
  if (own.groups > 0) {
    route = {ProductRoute::Own, own.tile, own.tile, own.groups, 1, 0};
    least = own_time(kind, own, M, N, K);
  } else {
    route = {ProductRoute::Library, 0, 0, 0, contraction_parts(kind, M, N, K), turned_operand(kind, n)};
    least = 1.5 + library_cost(kind, n, route.parts, route.turn);   // (1.5 us: its calls take the host longer)
  }
  auto consider = [&](double cost, const ProductRoute& other) {
    if (cost >= least) return;
    least = cost;
    route = other;
  };
  if (M < 1 || N < 1 || K < 1) return route;
  // A step of many products with much work runs at the GPU's limit of power, where what moves more per product is slower than it is by itself:
  // pico_product_mid and narrow tiles ([5640 x 12288]^T [5640 x 1536] by itself 211 us in mid, 226 in large; in a training step 234 and 197).
  const double gflop = std::min(M, N) >= 512 ? 2e-9 * M * N * K : 0, narrow = gflop >= 60 ? 1.15 : gflop >= 25 ? 1.1 : 1.0, mid = gflop >= 60 ? 1.25 : 1.0;
  // (rows that start in the same memory channel: [3584 x 32768] @ [32768 x 512] 131 us in the library's pieces, 178 in this kernel's)
  const bool strided = kind == Product::NN && lda % 32768 == 0 && N <= 1024;
  LargeProduct large;
  const double large_cost = large_time(M, N, K, large);
  if (K >= 128 && std::min(M, N) >= 192 && pico_product_large_takes(M, N, K, lda, ldb, a_slow, b_slow, static_cast<int>(large.parts)))
    consider((strided ? 1.35 : large.tile_m * large.tile_n < 65536 ? narrow : 1.0) * large_cost, {ProductRoute::Large, large.tile_m, large.tile_n, 0, large.parts, 0});
  if (pico_product_mid_takes(M, N, K, lda, ldb, a_slow, b_slow)) {
    MidProduct whole, cut;
    const double whole_cost = mid * mid_time(kind, M, N, K, whole), cut_cost = mid * mid_parts_time(M, N, K, cut);
    // With few tiles the library deals out a contraction that divides evenly: [128 x 3328] @ [832 x 3328]^T 6.9 us, here 9.0; over 300 such
    // products whole walks here took 1.06 .. 1.3 of its time, and 0.6 .. 0.9 with other contractions or more tiles.
    const bool dealt = kind == Product::NT && K > 3072 && (K % 256 == 0 ? K <= 8192 : K % 128 == 0 && K <= 4352) && ((M + 31) / 32) * ((N + 63) / 64) <= 128;
    if (whole.tile_m > 0 && !dealt) consider(whole_cost, {ProductRoute::Mid, whole.tile_m, whole.tile_n, 0, 1, 0});
    if (cut.parts > 1 && !dealt) consider(cut_cost, {ProductRoute::Mid, cut.tile_m, cut.tile_n, 0, cut.parts, 0});
  }
  return route;
}

// The rules go through some thirty tiles each, 0.4 .. 1.3 us a call on the side that paces a small model's step (13 us of a two-layer
// 135M step), so what they say is kept by the numbers they were asked with: per thread, and dropped for whatever comes to the same place.
template <typename Answer>
struct RouteTable {
  struct Entry {
    int64_t key[6] = {};
    bool used = false;
    Answer answer;
  } entries[256];
  template <typename Make>
  const Answer& get(const int64_t (&key)[6], const Make& make) {
    uint64_t h = 1469598103934665603ull;
    for (const int64_t v : key) h = (h ^ static_cast<uint64_t>(v)) * 1099511628211ull;
    Entry& e = entries[(h ^ (h >> 29)) % 256];
    if (!e.used || !std::equal(key, key + 6, e.key)) {
      e.answer = make();
      std::copy(key, key + 6, e.key);
      e.used = true;
    }
    return e.answer;
  }
};
ProductRoute product_route(Product kind, const ProductSizes& n) {
  static thread_local RouteTable<ProductRoute> table;
  return table.get({static_cast<int64_t>(kind), n.M, n.N, n.K, n.lda, n.ldb}, [&] { return choose_route(kind, n); });
}
// for tests: "mid 64x96", "large 256x192 in 24", "own 64 in 2 groups", "library", "library in 4", "turned" (the library with an
// operand transposed first)
std::string route_name(const ProductRoute& r) {
  const std::string tiles = std::to_string(r.tile_m) + "x" + std::to_string(r.tile_n), pieces = r.parts > 1 ? " in " + std::to_string(r.parts) : "";
  switch (r.kernel) {
    case ProductRoute::Mid: return "mid " + tiles + pieces;
    case ProductRoute::Large: return "large " + tiles + pieces;
    case ProductRoute::Own: return "own " + std::to_string(r.tile_m) + " in " + std::to_string(r.groups) + (r.groups > 1 ? " groups" : " group");
    default: return (r.turn ? "turned" : "library") + pieces;
  }
}

struct GradientTiles {
  MidProduct dx, dw;   // (tile_m 0: apart)
};
// The time at which the last of n1 workgroups of t1 each, then n2 of t2 each, ends on 256 CUs
double workgroups_end(int64_t n1, double t1, int64_t n2, double t2) {
  const int64_t rest = n1 % 256, idle = 256 - rest;
  const double early = n1 / 256 * t1, late = early + t1, first = rest ? late : early;   // `idle` CUs are free at `early`, `rest` at `late`
  double end = 1e30;
  for (const double base : {early, late})
    for (int64_t k = 0; k <= n2 / 256 + static_cast<int64_t>(t1 / t2) + 2; ++k) {
      const double at = base + k * t2;
      const int64_t done = idle * static_cast<int64_t>((at - early) / t2 + 1e-9) + (at >= late ? rest * static_cast<int64_t>((at - late) / t2 + 1e-9) : 0);
      if (at < first || done < n2) continue;
      end = std::min(end, at);
      break;
    }
  return end;
}
GradientTiles choose_gradient_tiles(int64_t rows, int64_t out, int64_t in) {
  struct Form {
    int64_t m, n, groups;
    double trip, end;
  };
  static constexpr Form forms[] = {{32, 64, 4, 0.72, 1.93}, {64, 64, 2, 0.48, 2.15}, {64, 96, 2, 0.54, 2.50}, {64, 128, 2, 0.68, 2.69}};
  auto tiles = [](int64_t M, int64_t N, const Form& f) { return ((M + f.m - 1) / f.m) * ((N + f.n - 1) / f.n); };
  auto length = [](int64_t K, const Form& f) { return ((K + 63) / 64 + f.groups - 1) / f.groups * f.trip + f.end; };
  if (tiles(rows, in, forms[3]) + tiles(out, in, forms[3]) > 1024) return {};
  GradientTiles best;
  double least = 1e30;
  for (const Form& x : forms)
    for (const Form& w : forms) {
      const int64_t nx = tiles(rows, in, x), nw = tiles(out, in, w);
      const double tx = length(out, x), tw = length(rows, w), busy = std::min(1.0, (nx + nw) / 256.0);
      const double t = 1.02 + (0.91 + 0.09 * busy) * (rows > out ? workgroups_end(nw, tw, nx, tx) : workgroups_end(nx, tx, nw, tw));
      if (t < least) {
        least = t;
        best = {{x.m, x.n, 1}, {w.m, w.n, 1}};
      }
    }
  auto alone = [](Product kind, int64_t M, int64_t N, int64_t K) {
    MidProduct tiles;
    return std::min(mid_time(kind, M, N, K, tiles), mid_parts_time(M, N, K, tiles));
  };
  return least < 0.85 * (alone(Product::NN, rows, in, out) + alone(Product::TN, out, in, rows)) ? best : GradientTiles{};
}
GradientTiles gradient_tiles(int64_t rows, int64_t out, int64_t in) {
  static thread_local RouteTable<GradientTiles> table;
  return table.get({rows, out, in, 0, 0, 0}, [&] { return choose_gradient_tiles(rows, out, in); });
}
std::string route_name(const GradientTiles& t) {   // "32x64 64x96" (of dx, of dw) or "apart"
  auto tiles = [](const MidProduct& m) { return std::to_string(m.tile_m) + "x" + std::to_string(m.tile_n); };
  return t.dx.tile_m > 0 ? tiles(t.dx) + " " + tiles(t.dw) : "apart";
}

}  // namespace
