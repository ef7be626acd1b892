// W8A8 / FP8 / BF16 / FP16 linear layers on gfx950 MFMA: tile schedules and launches.  Epilogues in
// gemm_epilogue.h, the small-tile kernels in gemm_ring.h and gemm_decode.h, the choice among all of
// them in gemm_plan.h.
#pragma once
#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "gemm_decode.h"
#include "gemm_plan.h"
#include "gemm_ring.h"

namespace m5k {
namespace gemm {
namespace detail {

// One 256 x G::TN output tile per workgroup.
template <int MODE, bool ALIGNED, int OUT_DT, int BIAS, int GATE, bool RAW, class G = KernelGrid>
__global__ __launch_bounds__(G::THREADS, 1) void gemm_kernel(const uint8_t* __restrict__ A,
                                                             const uint8_t* __restrict__ B, int M, int N,
                                                             int64_t Kb, EpiParams p) {
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + G::TN - 1) / G::TN;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * G::TN;
  const TileScalePrefetch<G> pre = prefetch_scales<MODE, RAW, G>(p, M, N, m0, n0);
  AccTile<MODE, G> acc;
  if constexpr (ALIGNED) mainloop_dma<MODE, G>(A, B, M, N, Kb, m0, n0, acc, 0, k_stages(Kb));
  else mainloop_staged<MODE, G>(A, B, M, N, Kb, m0, n0, acc);
  epilogue<MODE, OUT_DT, BIAS, GATE, RAW, G>(acc, M, N, m0, n0, p, pre);
}

// ---- Mixed tiles for a partial last round ---------------------------------------------------
//
// T tiles on C CUs (one workgroup per CU) take ceil(T / C) rounds; when the last round is only
// partly filled, most CUs idle through it.  The mixed launch runs the first `full` tiles of the
// raster order (a whole number of rounds) as 256 x 256 tiles and splits each remaining tile
// into two 256 x 128 halves, which take a little over half a tile's time each, so the leftover
// work runs as one shorter, better-filled round.  Each output element is still one
// workgroup's dot product over all of K: results are bit-identical to the plain launch.
// Workgroups [0, full) are the full tiles.  Workgroup full + w runs logical half
// h = xcd_logical(w), which is half h & 1 of tile full + h / 2 in the raster order.  full is
// a multiple of 8, so w keeps the hardware's XCD (w % 8 == (full + w) % 8), each XCD gets a
// contiguous run of h, and the two halves of a tile land on one XCD unless a run boundary
// falls between them.
using HalfGrid = Grid8Half;

template <int MODE, int OUT_DT, int BIAS, int GATE, bool RAW>
__global__ __launch_bounds__(KernelGrid::THREADS, 1) void gemm_mixed_kernel(const uint8_t* __restrict__ A,
                                                                            const uint8_t* __restrict__ B, int M,
                                                                            int N, int64_t Kb, int full,
                                                                            EpiParams p) {
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const int bid = static_cast<int>(blockIdx.x);
  if (bid < full) {
    using G = KernelGrid;
    int tm, tn;
    band_coords(xcd_logical(bid, full), tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const TileScalePrefetch<G> pre = prefetch_scales<MODE, RAW, G>(p, M, N, m0, n0);
    AccTile<MODE, G> acc;
    mainloop_dma<MODE, G>(A, B, M, N, Kb, m0, n0, acc, 0, k_stages(Kb));
    epilogue<MODE, OUT_DT, BIAS, GATE, RAW, G>(acc, M, N, m0, n0, p, pre);
  } else {
    using G = HalfGrid;
    const int h = xcd_logical(bid - full, 2 * (tiles_m * tiles_n - full));
    int tm, tn;
    band_coords(full + (h >> 1), tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN + (h & 1) * G::TN;
    if (n0 >= N) return;  // right half of a last tile column at most 128 wide (whole workgroup)
    const TileScalePrefetch<G> pre = prefetch_scales<MODE, RAW, G>(p, M, N, m0, n0);
    AccTile<MODE, G> acc;
    mainloop_dma<MODE, G>(A, B, M, N, Kb, m0, n0, acc, 0, k_stages(Kb));
    epilogue<MODE, OUT_DT, BIAS, GATE, RAW, G>(acc, M, N, m0, n0, p, pre);
  }
}

constexpr int XCDS = 8;
// Time of a 256 x 128 tile in units of a 256 x 256 tile's (measured: 256 half tiles of
// 2048 x 4096 x 4096 INT8 in 0.57 of the 256 full tiles of 4096 x 4096 x 4096).
constexpr double kHalfTileCost = 0.56;

// Finish time, in 256 x 256 tile times, of `full` tiles (a multiple of the CU count: whole
// rounds) followed by `half` half tiles; workgroup w runs on XCD w % 8, whose CUs take its
// workgroups in order.
inline double mixed_makespan(int64_t full, int64_t half, int cus) {
  const int64_t c = cus / XCDS;
  const int64_t per = (half + XCDS - 1) / XCDS;  // the busiest XCD's half tiles
  return static_cast<double>(full / cus) + static_cast<double>((per + c - 1) / c) * kHalfTileCost;
}

// Full tiles of the mixed launch, or -1 for the plain launch.  Candidates keep the last one
// or two rounds of tiles as halves; the mixed launch is used for a predicted gain of 5% or
// more.  The full part is always whole rounds, so the half tiles start together once every
// full tile is done.  Measured on MI355X, half tiles that overlapped a partial round of full
// tiles ran slower than such a model predicts (4-8% behind the plain launch at N = 6144 and
// 14336), while the whole-round splits matched or beat it.
// M5K_GEMM_MIXED_TILES=0 in the environment selects the plain launch (read on every call).
inline int64_t mixed_full_tiles(int64_t m, int64_t n, int cus) {
  if (cus < XCDS || cus % XCDS) return -1;
  if (const char* env = std::getenv("M5K_GEMM_MIXED_TILES"); env && env[0] == '0') return -1;
  const int64_t total = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);
  const int64_t rounds = total / cus;
  if (total % cus == 0 || rounds > 64) return -1;  // no partial round, or one that is noise
  double best = static_cast<double>(rounds + 1) * 0.95;
  int64_t pick = -1;
  for (int64_t j = rounds; j >= 0 && j + 2 >= rounds; --j) {
    const int64_t full = j * cus;
    const double t = mixed_makespan(full, 2 * (total - full), cus);
    if (t < best) {
      best = t;
      pick = full;
    }
  }
  return pick;
}

// ---- Narrow tiles for a whole number of rounds ------------------------------------------------
//
// 256 x 224 tiles (Grid8Narrow, 16 x 16 modes) do 7/8 of a full tile's MFMAs.  Where their
// count fills whole rounds and the 256-wide count does not (N = 7168: 28 full or 32 narrow
// tile columns; at M = 4096, 448 tiles = 1.75 rounds against 512 = 2 rounds), the narrow grid
// finishes in 2 x 7/8 round times instead of 2.  Bit-identical to the plain launch for the
// same reason as the mixed launch.
constexpr double kNarrowTileCost = 0.9;  // 256 x 224 tile time / 256 x 256 tile time

// Predicted time, in 256 x 256 tile times, of the plain, mixed and narrow launches; returns
// true when the narrow launch is 5% or more ahead of both others.
inline bool narrow_pays(int64_t m, int64_t n, int cus, int64_t mixed_full) {
  if (cus <= 0) return false;
  if (const char* env = std::getenv("M5K_GEMM_NARROW_TILES"); env && env[0] == '0') return false;
  const int64_t tiles_m = (m + BM - 1) / BM;
  const int64_t plain_tiles = tiles_m * ((n + BN - 1) / BN);
  const int64_t narrow_tiles = tiles_m * ((n + Grid8Narrow::TN - 1) / Grid8Narrow::TN);
  if (plain_tiles > 64 * static_cast<int64_t>(cus)) return false;
  double other = static_cast<double>((plain_tiles + cus - 1) / cus);
  if (mixed_full >= 0) other = std::min(other, mixed_makespan(mixed_full, 2 * (plain_tiles - mixed_full), cus));
  const double narrow = static_cast<double>((narrow_tiles + cus - 1) / cus) * kNarrowTileCost;
  return narrow < 0.95 * other;
}

// The direct-to-LDS main loop needs 16-byte aligned rows and bases and 256-row windows that
// fit a 32-bit buffer offset (rows of at most 2^23 bytes); other operands take the
// register-staged loop.
inline bool dma_ok(const void* a, const void* b, int64_t kb) {
  return kb % 16 == 0 && kb <= (int64_t(1) << 23) && aligned16(a) && aligned16(b);
}

// SCHED_QUAD: plain 256 x 256 tiles on Grid4 (four waves of 128 x 128, one per SIMD, 256 AGPR
// accumulators), W8A8 only.  Never planned: on the FFN-down, FFN-up and 4096^3 GEMMs it measured
// 1.10-1.15x the time of the eight-wave grid (same bits), since a lone wave per SIMD has no
// sibling to issue MFMAs while it waits on LDS reads and stage barriers.  It stays a tuner option.
enum Schedule { SCHED_PLAIN = 0, SCHED_MIXED = 1, SCHED_NARROW = 2, SCHED_QUAD = 3 };

// A schedule forced for the calls of this host thread (m5k_gemm_set_schedule: the harness tuner),
// else one named by M5K_GEMM_SCHEDULE ("plain", "mixed", "narrow", "quad"; read on every call, for
// outside tools), else -1.  A forced mixed launch keeps the planner's full-tile count when it has
// one, else runs every tile of the last (or only) round as two halves.  Narrow applies to the
// 16 x 16 modes and quad to W8A8; the other modes run plain in their place.
inline thread_local int g_thread_schedule = -1;

// The split entry points of this host thread run as many K ranges as a call names, not up to as many
// (m5k_gemm_set_exact_splits: the harness tuner, and tests of the split kernels).
inline thread_local bool g_thread_exact_splits = false;

inline int forced_schedule(bool md16, bool i8, int64_t m, int64_t n, int cus, int64_t& full) {
  int which = g_thread_schedule;
  if (which < 0) {
    const char* env = std::getenv("M5K_GEMM_SCHEDULE");
    if (env == nullptr || env[0] == '\0') return -1;
    if (std::strcmp(env, "plain") == 0) which = SCHED_PLAIN;
    else if (std::strcmp(env, "mixed") == 0) which = SCHED_MIXED;
    else if (std::strcmp(env, "narrow") == 0) which = SCHED_NARROW;
    else if (std::strcmp(env, "quad") == 0) which = SCHED_QUAD;
    else return -1;
  }
  full = -1;
  if (which == SCHED_PLAIN) return SCHED_PLAIN;
  if (which == SCHED_NARROW) return md16 ? SCHED_NARROW : SCHED_PLAIN;
  if (which == SCHED_QUAD) return i8 ? SCHED_QUAD : SCHED_PLAIN;
  if (which == SCHED_MIXED && cus >= XCDS && cus % XCDS == 0) {
    const int64_t total = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);
    full = mixed_full_tiles(m, n, cus);
    if (full < 0) full = total > cus ? (total - 1) / cus * cus : 0;
    return SCHED_MIXED;
  }
  return -1;
}

// Launch schedule of an aligned GEMM with an [m, n] output on `cus` CUs; `full` receives the
// mixed launch's full tiles (-1 otherwise).  Narrow tiles exist for the 16 x 16 modes only.
inline int plan_schedule(bool md16, bool i8, int64_t m, int64_t n, int cus, int64_t& full) {
  if (const int forced = forced_schedule(md16, i8, m, n, cus, full); forced >= 0) return forced;
  full = mixed_full_tiles(m, n, cus);
  if (md16 && narrow_pays(m, n, cus, full)) {
    full = -1;
    return SCHED_NARROW;
  }
  return full >= 0 ? SCHED_MIXED : SCHED_PLAIN;
}

// ---- Small tiles (gemm_ring.h, gemm_decode.h) ----------------------------------------------------

// Ring shapes by tile.  64 KiB of stages let two 64 x 64 workgroups share a CU; 96 KiB ("deep") keep
// one, with twice the K per barrier.  FP8 stages hold two planes, so half as many.
template <int MODE>
struct RingTiles {
  using T128 = ring::Cfg<MODE, 128, 128, MODE == F8 ? 2 : 4>;
  using T64 = ring::Cfg<MODE, 64, 64, MODE == F8 ? 2 : 4>;
  using Deep = ring::Cfg<MODE, 64, 64, 3, 2>;
  // Unaligned operands: two stage buffers, filled through registers.
  using U128 = ring::Cfg<MODE, 128, 128, 2, 1>;
  using U64 = ring::Cfg<MODE, 64, 64, 2, 1>;
};

constexpr bool small_mode(int mode) { return mode == I8 || mode == F8 || mode == BF16 || mode == F16; }

// Time of the 256-row schedules' launch in 256 x 256 tile times.
inline double units_256(bool md16, int64_t m, int64_t n, int cus) {
  const int64_t tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);
  if (cus <= 0) return static_cast<double>(tiles);
  const int64_t full = mixed_full_tiles(m, n, cus);
  if (md16 && narrow_pays(m, n, cus, full)) {
    const int64_t narrow = ((m + BM - 1) / BM) * ((n + Grid8Narrow::TN - 1) / Grid8Narrow::TN);
    return static_cast<double>((narrow + cus - 1) / cus) * kNarrowTileCost;
  }
  if (full >= 0) return 1.03 * mixed_makespan(full, 2 * (tiles - full), cus);
  return static_cast<double>((tiles + cus - 1) / cus);
}

// The tile of an [m, n] output with rows of kb bytes (no partial sums): one of gemm_plan.h's, or
// TILE_256 for the 256-row schedules.  Aligned operands under a forced schedule run that schedule.
// Aligned float rows of under 1 KiB stay there too: the smaller tiles split K over waves, and eight
// 128-byte lines leave each of them one or none.  Unaligned operands have ring tiles at any K, except
// FP8's, which keep the register-staged loop (one_stage_on_256: INT8's of one stage, over many tiles).
inline plan::Choice plan_tile(int mode, int64_t m, int64_t n, int64_t kb, int cus, bool aligned, int max_splits = 1,
                              double limit_us = 1e30) {
  const plan::Choice none{plan::TILE_256, 1, 0.0};
  const bool md16 = mode == I8 || mode == BF16 || mode == F16;
  if (!small_mode(mode) || cus <= 0 || (!aligned && mode == F8)) return none;
  if (aligned) {
    int64_t full = -1;
    if (forced_schedule(md16, mode == I8, m, n, cus, full) >= 0) return none;
    if (mode != I8 && kb < 8 * BKB) return none;
    const double units = units_256(md16, m, n, cus);
    limit_us = std::min(limit_us, max_splits > 1 ? plan::tile256_us(units, n, kb) : plan::unsplit256_us(units, n, kb));
  }
  return plan::choose(m, n, kb, cus, aligned, max_splits, limit_us);
}

// Unaligned INT8 rows of one stage (K <= 128): the byte-wise 256-row loop costs one pass there, 3 + 17.5 us
// a round, and over several rounds of small tiles `small` less than they do (4096 x 4096 x 100: 21.4 us
// against 29.2; 9000 x 1600 x 65 20.5 against 26.2).  From two stages on the small tiles are ahead (x 257:
// 34.3 us against 46.4).
inline bool one_stage_on_256(int mode, bool aligned, int64_t m, int64_t n, int64_t kb, int cus, const plan::Choice& small) {
  if (mode != I8 || aligned || kb > BKB || cus <= 0) return false;
  const int64_t rounds = plan::ceil_div(plan::ceil_div(m, BM) * plan::ceil_div(n, BN), cus);
  return 3.0 + 17.5 * static_cast<double>(rounds) < 0.95 * small.us;
}

template <class C, bool ALIGNED, int OUT_DT, int BIAS, int GATE>
int launch_ring(const uint8_t* A, const uint8_t* B, int64_t m, int64_t n, int64_t kb, const EpiParams& q,
                hipStream_t st, const char* name) {
  const int64_t wgs = ((m + C::TM - 1) / C::TM) * ((n + C::TN - 1) / C::TN);
  M5K_REQUIRE(wgs <= 0x7FFFFFFF, "%s: too many tiles", name);
  launch_kernel(ring::gemm_ring_kernel<C, ALIGNED, OUT_DT, BIAS, GATE>, dim3(static_cast<unsigned>(wgs)), dim3(512), st,
                A, B, (int)m, (int)n, kb, q);
  return launch_status(name);
}

template <int MODE, int OUT_DT, int BIAS, int GATE>
int launch_small(int tile, bool aligned, const uint8_t* A, const uint8_t* B, int64_t m, int64_t n, int64_t kb,
                 const EpiParams& q, hipStream_t st, const char* name) {
  using R = RingTiles<MODE>;
  if constexpr (MODE != F8) {
    if (!aligned)
      return tile == plan::TILE_128
                 ? launch_ring<typename R::U128, false, OUT_DT, BIAS, GATE>(A, B, m, n, kb, q, st, name)
                 : launch_ring<typename R::U64, false, OUT_DT, BIAS, GATE>(A, B, m, n, kb, q, st, name);
  }
  switch (tile) {
    case plan::TILE_128: return launch_ring<typename R::T128, true, OUT_DT, BIAS, GATE>(A, B, m, n, kb, q, st, name);
    case plan::TILE_64: return launch_ring<typename R::T64, true, OUT_DT, BIAS, GATE>(A, B, m, n, kb, q, st, name);
    case plan::TILE_64_DEEP:
      return launch_ring<typename R::Deep, true, OUT_DT, BIAS, GATE>(A, B, m, n, kb, q, st, name);
    default: break;
  }
  const dim3 wgs(static_cast<unsigned>((n + 15) / 16)), block(64 * decode::WAVES);
  if (m <= 16)
    launch_kernel(decode::gemm_decode_kernel<MODE, 1, OUT_DT, BIAS, GATE>, wgs, block, st, A, B, (int)m, (int)n, kb, q);
  else
    launch_kernel(decode::gemm_decode_kernel<MODE, 2, OUT_DT, BIAS, GATE>, wgs, block, st, A, B, (int)m, (int)n, kb, q);
  return launch_status(name);
}

template <int MODE, int OUT_DT, int BIAS, int GATE, bool RAW>
int launch(const void* a, const void* b, int64_t m, int64_t n, int64_t k, const EpiParams& p,
           hipStream_t st, const char* name) {
  const int64_t kb = k * Traits<MODE>::elem_bytes;
  const int64_t tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);
  M5K_REQUIRE(tiles <= 0x7FFFFFFF, "%s: too many tiles", name);
  // The direct-to-LDS path addresses a tile's rows through 32-bit buffer windows.
  const bool aligned = dma_ok(a, b, kb);
  const dim3 grid(static_cast<unsigned>(tiles)), block(KernelGrid::THREADS);
  auto* A = static_cast<const uint8_t*>(a);
  auto* B = static_cast<const uint8_t*>(b);
  EpiParams q = p;
  q.coalesced = n % 8 == 0 && aligned16(p.c) && (p.residual == nullptr || (aligned16(p.residual) && aligned16(p.gate)));
  if constexpr (small_mode(MODE) && !RAW) {
    const plan::Choice small = plan_tile(MODE, m, n, kb, device_cus(), aligned);
    if (small.tile != plan::TILE_256 && !one_stage_on_256(MODE, aligned, m, n, kb, device_cus(), small))
      return launch_small<MODE, OUT_DT, BIAS, GATE>(small.tile, aligned, A, B, m, n, kb, q, st, name);
  }
  if (aligned) {
    int64_t full = -1;
    // The narrow 256 x 224 tile serves the 16 x 16 modes with 16-byte fragments (INT8, BF16,
    // FP16); FP8's 32-byte fragments for its seven B blocks do not fit beside the accumulators.
    constexpr bool narrow_ok = Traits<MODE>::MD == 16 && MODE != F8;
    const int sched = plan_schedule(narrow_ok, MODE == I8, m, n, device_cus(), full);
    if constexpr (narrow_ok) {
      if (sched == SCHED_NARROW) {
        using G = Grid8Narrow;
        const int64_t wgs = ((m + BM - 1) / BM) * ((n + G::TN - 1) / G::TN);
        launch_kernel(gemm_kernel<MODE, true, OUT_DT, BIAS, GATE, RAW, G>, dim3(static_cast<unsigned>(wgs)), block, st,
                      A, B, (int)m, (int)n, kb, q);
        return launch_status(name);
      }
    }
    if constexpr (MODE == I8) {
      if (sched == SCHED_QUAD) {
        launch_kernel(gemm_kernel<MODE, true, OUT_DT, BIAS, GATE, RAW, Grid4>, grid, dim3(Grid4::THREADS), st, A, B,
                      (int)m, (int)n, kb, q);
        return launch_status(name);
      }
    }
    if (sched == SCHED_MIXED) {
      const int64_t wgs = full + 2 * (tiles - full);
      launch_kernel(gemm_mixed_kernel<MODE, OUT_DT, BIAS, GATE, RAW>, dim3(static_cast<unsigned>(wgs)), block, st, A, B,
                    (int)m, (int)n, kb, static_cast<int>(full), q);
    } else {
      launch_kernel(gemm_kernel<MODE, true, OUT_DT, BIAS, GATE, RAW>, grid, block, st, A, B, (int)m, (int)n, kb, q);
    }
  } else if constexpr (MODE == I8 || MODE == F8 || MODE == F32) {
    // INT8: one stage, no CU count, or the raw accumulators.
    launch_kernel(gemm_kernel<MODE, false, OUT_DT, BIAS, GATE, RAW>, grid, block, st, A, B, (int)m, (int)n, kb, q);
  } else {
    return launch_small<MODE, OUT_DT, BIAS, GATE>(plan::TILE_64, false, A, B, m, n, kb, q, st, name);
  }
  return launch_status(name);
}

// ---- Split-K W8A8 for short M ------------------------------------------------------------
//
// With few output tiles (M of one or two tile rows) the plain launch leaves most CUs idle
// while its few workgroups stream the whole weight.  The split form gives each tile `splits`
// workgroups, each over a contiguous range of 128-byte K stages, writing raw INT32 partial tiles to
// workspace[s][M][N]; a second kernel sums the partials in split order (exact: INT32 sums of
// a bounded dot product) and applies the same FP32 epilogue as gemm_kernel, so the output
// is bit-identical to the plain launch.  P is the partial type: INT32 for INT8, FP32 for the
// FP8 split (launch_f8_splitk).
template <int MODE, class G = KernelGrid, class P = int32_t>
__global__ __launch_bounds__(G::THREADS, 1) void gemm_splitk_kernel(const uint8_t* __restrict__ A,
                                                                    const uint8_t* __restrict__ B, int M, int N,
                                                                    int64_t Kb, int splits, int64_t stages_per_split,
                                                                    P* __restrict__ partial) {
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + G::TN - 1) / G::TN;
  const int tile = static_cast<int>(blockIdx.x) / splits, s = static_cast<int>(blockIdx.x) % splits;
  int tm, tn;
  tile_coords(tile, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * G::TN;
  const int64_t kt_total = k_stages(Kb);
  const int64_t kt0 = s * stages_per_split;
  const int64_t kt1 = kt0 + stages_per_split < kt_total ? kt0 + stages_per_split : kt_total;
  AccTile<MODE, G> acc;
  mainloop_dma<MODE, G>(A, B, M, N, Kb, m0, n0, acc, kt0, kt1 - kt0);
  P* out = partial + static_cast<int64_t>(s) * M * N;
  for_each_acc<G>(acc, m0, n0, [&](int m, int n, auto v) {
    if (m < M && n < N) out[static_cast<int64_t>(m) * N + n] = v;
  });
}

// Sums the partial tiles in split order and applies the epilogue.  VEC = 4: four consecutive columns
// per thread (N % 4 == 0 and 16-byte aligned c), one 16-byte load per split and one packed store; the
// splits' loads do not depend on each other, so a thread has them all in flight.
template <int OUT_DT, int BIAS, int GATE, class P, int VEC>
__global__ __launch_bounds__(256) void splitk_epilogue_kernel(const P* __restrict__ partial, int splits, int M, int N,
                                                              EpiParams p) {
  constexpr int MODE = std::is_same<P, float>::value ? F8 : I8;
  const int64_t total = static_cast<int64_t>(M) * N;
  for (int64_t idx = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * VEC; idx < total;
       idx += static_cast<int64_t>(gridDim.x) * 256 * VEC) {
    const int m = static_cast<int>(idx / N), n = static_cast<int>(idx - static_cast<int64_t>(m) * N);
    if constexpr (VEC == 1) {
      P v = 0;
      for (int s = 0; s < splits; ++s) v += partial[s * total + idx];
      store_elem<OUT_DT>(p.c, idx, result_value<MODE, BIAS, GATE>(p, v, m, n, N));
    } else {
      typedef P vec4 __attribute__((ext_vector_type(4)));
      vec4 v = {0, 0, 0, 0};
#pragma unroll 4
      for (int s = 0; s < splits; ++s) v += *reinterpret_cast<const vec4*>(partial + s * total + idx);
      float r[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = result_value<MODE, BIAS, GATE>(p, v[e], m, n + e, N);
      if constexpr (OUT_DT == M5K_F32) {
        *reinterpret_cast<float4*>(static_cast<float*>(p.c) + idx) = make_float4(r[0], r[1], r[2], r[3]);
      } else {
        uint2 w;
        if constexpr (OUT_DT == M5K_BF16) w = make_uint2(f32x2_to_bf16x2(r[0], r[1]), f32x2_to_bf16x2(r[2], r[3]));
        else
          w = make_uint2(f32_to_f16_bits(r[0]) | (f32_to_f16_bits(r[1]) << 16),
                         f32_to_f16_bits(r[2]) | (f32_to_f16_bits(r[3]) << 16));
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.c) + idx) = w;
      }
    }
  }
}

template <int OUT_DT, int BIAS, int GATE, class P>
int launch_splitk_epilogue(const P* workspace, int used, int64_t m, int64_t n, const EpiParams& p, hipStream_t st,
                           const char* name) {
  const bool vec = n % 4 == 0 && aligned16(p.c) && aligned16(workspace);
  const int64_t blocks = (m * n / (vec ? 4 : 1) + 255) / 256;
  const dim3 grid(static_cast<unsigned>(blocks < 65536 ? blocks : 65536));
  if (vec)
    launch_kernel(splitk_epilogue_kernel<OUT_DT, BIAS, GATE, P, 4>, grid, dim3(256), st, workspace, used, (int)m, (int)n, p);
  else
    launch_kernel(splitk_epilogue_kernel<OUT_DT, BIAS, GATE, P, 1>, grid, dim3(256), st, workspace, used, (int)m, (int)n, p);
  return launch_status(name);
}

template <class C, class P>
int launch_ring_splitk(const uint8_t* A, const uint8_t* B, int64_t m, int64_t n, int64_t kb, int splits, P* workspace,
                       int& used, hipStream_t st, const char* name) {
  const int64_t total = ring::stages<C>(kb);
  const int64_t per = (total + splits - 1) / splits;
  used = static_cast<int>((total + per - 1) / per);  // no empty split
  const int64_t wgs = ((m + C::TM - 1) / C::TM) * ((n + C::TN - 1) / C::TN) * used;
  M5K_REQUIRE(wgs <= 0x7FFFFFFF, "%s: too many workgroups", name);
  launch_kernel(ring::gemm_ring_splitk_kernel<C, P>, dim3(static_cast<unsigned>(wgs)), dim3(512), st, A, B, (int)m, (int)n,
                kb, used, per, workspace);
  return launch_status(name);
}

// K bytes of a main-loop stage: the ranges are whole stages.
constexpr int64_t stage_bytes(int mode, int tile) {
  return tile == plan::TILE_64_DEEP || (mode == F8 && (tile == plan::TILE_128 || tile == plan::TILE_64)) ? 2 * BKB : BKB;
}
template <int MODE>
constexpr bool ring_stages_agree() {
  using R = RingTiles<MODE>;
  return R::T128::STAGE_K == stage_bytes(MODE, plan::TILE_128) && R::T64::STAGE_K == stage_bytes(MODE, plan::TILE_64) &&
         R::Deep::STAGE_K == stage_bytes(MODE, plan::TILE_64_DEEP);
}
static_assert(ring_stages_agree<I8>() && ring_stages_agree<F8>(), "K ranges are counted as they are launched");

// Ranges of a row of kb bytes in at most `splits` of equally many stages: none is empty.
inline int used_ranges(int mode, int tile, int64_t kb, int splits) {
  const int64_t total = plan::ceil_div(kb, stage_bytes(mode, tile)), per = plan::ceil_div(total, splits);
  return static_cast<int>(plan::ceil_div(total, per));
}

struct SplitPlan {
  int tile;    // plan::Tile
  int splits;  // K ranges asked of the launch
  int ranges;  // and those that run; 1: the unsplit launch, with its own choice of tile
};

// The launch of a split entry point.  At most `splits` K ranges per tile, as many as the planner expects
// to pay: a tile small enough to fill the CUs needs none, and then no partial sums exist (128 x 4096 x
// 4096 INT8 with 4 ranges of 256 x 64 tiles and the epilogue pass 16.2 us; unsplit 64 x 64 tiles 9.7
// us).  The 256-row tiles serve what is left, middle M with a long K: 256 x 128 where their workgroups
// fit in one round, else 256 x 256 (M 900, N 5376, K 14336: 86.5 us with 3 ranges, 93.5 us unsplit).
// With the thread's exact setting, or under a forced schedule, the call's count itself runs (fewer only
// where ranges would be empty), on that schedule's 256-row tiles or on the best tile for that count.
inline SplitPlan plan_split(int mode, int64_t m, int64_t n, int64_t kb, int cus, int splits) {
  const bool md16 = mode != F8;  // the narrow schedule's modes
  const int used = used_ranges(mode, plan::TILE_256, kb, splits);
  const int64_t tiles_m = (m + BM - 1) / BM;
  const bool half = cus > 0 && tiles_m * ((n + HalfGrid::TN - 1) / HalfGrid::TN) * used <= static_cast<int64_t>(cus);
  const int tn = half ? HalfGrid::TN : BN;
  const int64_t wgs = tiles_m * ((n + tn - 1) / tn) * used;
  const double rounds = cus > 0 ? static_cast<double>((wgs + cus - 1) / cus) : 1.0;
  // Half tiles take a little more than in a mixed launch (768 x 5376 x 14336 in 2 ranges 69 us).
  const double split_256 =
      plan::tile256_us(rounds * (half ? 1.08 * kHalfTileCost : 1.0), n, kb / used) + plan::split_us(m, n, used);
  const SplitPlan rows_256{half ? plan::TILE_256_HALF : plan::TILE_256, splits, used};
  int64_t full = -1;
  if (forced_schedule(md16, mode == I8, m, n, cus, full) >= 0) return rows_256;
  plan::Choice c;
  if (g_thread_exact_splits) {
    if (splits == 1 || cus <= 0) return rows_256;
    c = plan::choose(m, n, kb, cus, true, splits, split_256, splits);
    if (c.tile == plan::TILE_256) return rows_256;
  } else {
    const double plain_256 = plan::tile256_us(units_256(md16, m, n, cus), n, kb);
    c = plan_tile(mode, m, n, kb, cus, true, splits, std::min(split_256, plain_256));
    if (c.tile == plan::TILE_256) return plain_256 < split_256 ? SplitPlan{plan::TILE_256, 1, 1} : rows_256;
  }
  return SplitPlan{c.tile, c.splits, used_ranges(mode, c.tile, kb, c.splits)};
}

template <int MODE, int OUT_DT, int BIAS, int GATE, class P>
int launch_splitk(const uint8_t* A, const uint8_t* B, int64_t m, int64_t n, int64_t kb, const EpiParams& p, int splits,
                  P* workspace, hipStream_t st, const char* name) {
  const SplitPlan c = plan_split(MODE, m, n, kb, device_cus(), splits);
  if (c.ranges == 1)
    return launch<MODE, OUT_DT, BIAS, GATE, false>(A, B, m, n, kb / Traits<MODE>::elem_bytes, p, st, name);
  using R = RingTiles<MODE>;
  int used = c.ranges, rc = M5K_OK;
  if (c.tile == plan::TILE_128) {
    rc = launch_ring_splitk<typename R::T128>(A, B, m, n, kb, c.splits, workspace, used, st, name);
  } else if (c.tile == plan::TILE_64) {
    rc = launch_ring_splitk<typename R::T64>(A, B, m, n, kb, c.splits, workspace, used, st, name);
  } else if (c.tile == plan::TILE_64_DEEP) {
    rc = launch_ring_splitk<typename R::Deep>(A, B, m, n, kb, c.splits, workspace, used, st, name);
  } else {
    const bool half = c.tile == plan::TILE_256_HALF;
    const int tn = half ? HalfGrid::TN : BN;
    const int64_t per = plan::ceil_div(k_stages(kb), c.splits);
    const int64_t wgs_256 = ((m + BM - 1) / BM) * ((n + tn - 1) / tn) * used;
    M5K_REQUIRE(wgs_256 <= 0x7FFFFFFF, "%s: too many workgroups", name);
    const dim3 wgs(static_cast<unsigned>(wgs_256)), block(KernelGrid::THREADS);
    if (half)
      launch_kernel(gemm_splitk_kernel<MODE, HalfGrid, P>, wgs, block, st, A, B, (int)m, (int)n, kb, used, per, workspace);
    else
      launch_kernel(gemm_splitk_kernel<MODE, KernelGrid, P>, wgs, block, st, A, B, (int)m, (int)n, kb, used, per, workspace);
    rc = launch_status(name);
  }
  if (rc) return rc;
  return launch_splitk_epilogue<OUT_DT, BIAS, GATE, P>(workspace, used, m, n, p, st, name);
}

template <int OUT_DT>
int launch_i8_splitk(const int8_t* a, const int8_t* b, int64_t m, int64_t n, int64_t k, const EpiParams& p,
                     int splits, int32_t* workspace, hipStream_t st, const char* name) {
  auto* A = reinterpret_cast<const uint8_t*>(a);
  auto* B = reinterpret_cast<const uint8_t*>(b);
  if (p.bias) {
    return p.bias_map ? launch_splitk<I8, OUT_DT, EPI_TABLE, EPI_NONE>(A, B, m, n, k, p, splits, workspace, st, name)
                      : launch_splitk<I8, OUT_DT, EPI_VECTOR, EPI_NONE>(A, B, m, n, k, p, splits, workspace, st, name);
  }
  if (p.residual) {
    return p.gate_map
               ? launch_splitk<I8, M5K_BF16, EPI_NONE, EPI_TABLE>(A, B, m, n, k, p, splits, workspace, st, name)
               : launch_splitk<I8, M5K_BF16, EPI_NONE, EPI_VECTOR>(A, B, m, n, k, p, splits, workspace, st, name);
  }
  return launch_splitk<I8, OUT_DT, EPI_NONE, EPI_NONE>(A, B, m, n, k, p, splits, workspace, st, name);
}

// FP8 split-K: FP32 partial tiles, summed in split order by the same epilogue kernel.  Each K
// range is its own FP32 accumulation, so the output can differ from the unsplit launch in the
// last bits of the FP32 sum (FP8's accumulation order is not pinned); it is deterministic.
template <int OUT_DT>
int launch_f8_splitk(const uint8_t* a, const uint8_t* b, int64_t m, int64_t n, int64_t k, const EpiParams& p,
                     int splits, float* workspace, hipStream_t st, const char* name) {
  return launch_splitk<F8, OUT_DT, EPI_NONE, EPI_NONE>(a, b, m, n, k, p, splits, workspace, st, name);
}

inline int check_shape(int64_t m, int64_t n, int64_t k, const char* name) {
  M5K_REQUIRE(m > 0 && n > 0 && k > 0, "%s: empty shape m=%lld n=%lld k=%lld", name, (long long)m,
              (long long)n, (long long)k);
  M5K_REQUIRE(m <= 0x7FFFFFFF && n <= 0x7FFFFFFF, "%s: m or n exceeds int32", name);
  return M5K_OK;
}

template <int MODE, int OUT_DT>
int launch_plain(const void* a, const void* b, int64_t m, int64_t n, int64_t k, const EpiParams& p,
                 hipStream_t st, const char* name) {
  if (p.residual) {
    return p.gate_map ? launch<MODE, M5K_BF16, EPI_NONE, EPI_TABLE, false>(a, b, m, n, k, p, st, name)
                      : launch<MODE, M5K_BF16, EPI_NONE, EPI_VECTOR, false>(a, b, m, n, k, p, st, name);
  }
  return launch<MODE, OUT_DT, EPI_NONE, EPI_NONE, false>(a, b, m, n, k, p, st, name);
}

template <int OUT_DT>
int launch_i8(const void* a, const void* b, int64_t m, int64_t n, int64_t k, const EpiParams& p,
              hipStream_t st) {
  const char* name = "m5k_gemm_i8";
  if (p.bias) {
    return p.bias_map ? launch<I8, OUT_DT, EPI_TABLE, EPI_NONE, false>(a, b, m, n, k, p, st, name)
                      : launch<I8, OUT_DT, EPI_VECTOR, EPI_NONE, false>(a, b, m, n, k, p, st, name);
  }
  return launch_plain<I8, OUT_DT>(a, b, m, n, k, p, st, name);
}

}  // namespace detail
}  // namespace gemm
}  // namespace m5k

