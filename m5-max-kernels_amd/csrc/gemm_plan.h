// Host-side choice of a GEMM's tile (no device code).
//
// Times are microseconds on MI355X as functions of the row length in bytes, fitted to INT8, FP8 and BF16
// products with a weight that the Infinity Cache holds.  Over M 1 to 2048, N 1024 to 21504 and K 1024 to
// 16384 (about 750 products a mode) four in five lie within 15% of them; with weights read from memory
// just over half do: the 64-row tiles take a fifth longer, the decode tile and K ranges about as
// modelled.  The choice costs 1% (weights from memory: 2%) over the fastest launch in the geometric
// mean, at worst 1.3 and 1.4 times.
// A round is one pass of workgroups over the CUs.
//
//   128 x 128 ring     1 workgroup per CU:   2 + r (6 + 3.6 us/KB)   1024 x 4096 x 4096 INT8 21.5 us
//                      from 3 rounds on, 15% more (8366 x 1920 x 8192 INT8, 4 rounds: 200 us)
//   64 x 64 ring       2 per CU:                 r (3.4 + 2.85)      256 x 7168 x 5376  INT8 18.7 us
//                      more rounds (L2-bound):   r (3.4 + 3.4)       553 x 7168 x 16384 INT8 131 us
//                      at most 1 per CU:         3.4 + 1.78
//   64 x 64 deep ring  1 per CU:                 r (3.85 + 1.43)     128 x 5376 x 14336 INT8 24.3 us
//   decode             r = ceil(N / 16 / CUs): 2 + r (0.62 + 0.02 M)   1 x 4096 x 4096  INT8  4.9 us
//   256-row schedules  u rounds' worth of tiles: u (13 + 10)         4096 x 4096 x 4096 INT8 54.5 us
//
// Every product streams its weight once, at about 5.2 TB/s at best; the 256-row tiles, with one stage
// ahead, at about 2 TB/s where the Infinity Cache does not hold it (402 x 14336 x 16384: 152 us), and
// at 3 TB/s where it does: the other tiles' rates are of weights that it holds, too.  With 2 TB/s for
// both, two rounds of 128 x 128 tiles were taken for one round of 256 x 128 halves (BF16 256 x 21504 x
// 4096: 70.0 us against 55.5 with one weight, 83.0 against 76.0 with weights in turn; INT8 256 x 21504 x
// 5376: 49.8 against 39.9, 59.3 against 57.8).  K ranges are weighed against the 2 TB/s.  A split
// over K adds a second launch and its 4-byte partial sums, written and read at about 6 TB/s.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace m5k {
namespace gemm {
namespace plan {

// TILE_256_HALF: 256 x 128 tiles, a form of the K ranges only.
enum Tile { TILE_256 = 0, TILE_128 = 1, TILE_64 = 2, TILE_64_DEEP = 3, TILE_DECODE = 4, TILE_256_HALF = 5 };

struct Choice {
  int tile;
  int splits;  // K ranges per tile (1: no partial sums)
  double us;
};

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

inline double split_us(int64_t m, int64_t n, int splits) {
  return splits > 1 ? 5.0 + 8.0 * splits * static_cast<double>(m) * static_cast<double>(n) / 6.0e6 : 0.0;
}

// max(a tile's own time, the weight's stream), the former breaking ties.
inline double with_stream(double us, int64_t n, int64_t kb, double bytes_per_us = 5.2e6) {
  return std::max(us, 2.0 + static_cast<double>(n) * static_cast<double>(kb) / bytes_per_us) + 0.05 * us;
}

inline double tile_us(int tile, int64_t m, int64_t n, int64_t kb, int cus, int splits) {
  const double len = static_cast<double>(ceil_div(kb, splits)) * 1e-3;
  double us = 0.0;
  switch (tile) {
    case TILE_128: {
      const int64_t r = ceil_div(ceil_div(m, 128) * ceil_div(n, 128) * splits, cus);
      us = 2.0 + static_cast<double>(r) * (r > 2 ? 1.15 : 1.0) * (6.0 + 3.6 * len);
      break;
    }
    case TILE_64: {
      const int64_t wgs = ceil_div(m, 64) * ceil_div(n, 64) * splits;
      const int64_t r = ceil_div(wgs, 2 * cus);
      us = wgs <= cus ? 3.4 + 1.78 * len : static_cast<double>(r) * (3.4 + (r > 1 ? 3.4 : 2.85) * len);
      break;
    }
    case TILE_64_DEEP: {
      const int64_t r = ceil_div(ceil_div(m, 64) * ceil_div(n, 64) * splits, cus);
      us = static_cast<double>(r) * (3.85 + 1.43 * len);
      break;
    }
    default: {
      const int64_t r = ceil_div(ceil_div(n, 16), cus);
      us = 2.0 + static_cast<double>(r) * len * (0.62 + 0.02 * static_cast<double>(m));
      break;
    }
  }
  return with_stream(us, n, kb) + split_us(m, n, splits);
}

// `units_256`: the 256-row schedules' time in 256 x 256 tile times; they stream the weight at 2 MB/us.
inline double tile256_us(double units_256, int64_t n, int64_t kb, double bytes_per_us = 2.0e6) {
  return with_stream(units_256 * (13.0 + 10.0e-3 * static_cast<double>(kb)), n, kb, bytes_per_us);
}

// The same beside other unsplit tiles: 3 MB/us for a weight that the Infinity Cache holds.
inline double unsplit256_us(double units_256, int64_t n, int64_t kb) {
  constexpr double kInfinityCache = 256.0e6;
  const double weight = static_cast<double>(n) * static_cast<double>(kb);
  return tile256_us(units_256, n, kb, weight <= kInfinityCache ? 3.0e6 : 2.0e6);
}

// The fastest tile of an [m, n] output with rows of kb bytes and min_splits to max_splits K ranges, or
// {TILE_256, 1} where none is 5% faster than `limit_us` (the 256-row schedules' time): near the line
// the predictions err either way.
// Unaligned operands have the two shallow rings only.
inline Choice choose(int64_t m, int64_t n, int64_t kb, int cus, bool aligned, int max_splits, double limit_us,
                     int min_splits = 1) {
  Choice best{TILE_256, 1, 0.95 * limit_us};
  auto offer = [&](int tile, int splits) {
    const double us = tile_us(tile, m, n, kb, cus, splits);
    if (us < best.us) best = Choice{tile, splits, us};
  };
  if (min_splits == 1) {
    offer(TILE_128, 1);
    offer(TILE_64, 1);
    if (!aligned) return best;
    offer(TILE_64_DEEP, 1);
    if (m <= 32) offer(TILE_DECODE, 1);
  }
  // K ranges of at least 1 KiB.
  for (int s = std::max(2, min_splits); s <= max_splits && kb / s >= 1024; ++s) {
    offer(TILE_128, s);
    offer(TILE_64, s);
    offer(TILE_64_DEEP, s);
  }
  return best;
}

}  // namespace plan
}  // namespace gemm
}  // namespace m5k
