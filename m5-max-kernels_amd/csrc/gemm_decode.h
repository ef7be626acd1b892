// Decode-shaped GEMM: a handful of rows (M <= 32) against the whole weight.
//
// The time is the weight's stream from memory, so the kernel is all loads in flight: a workgroup
// owns 16 weight rows (output columns), its eight waves take the 128-byte lines of K in turn, and
// each lane loads MFMA fragments straight from global memory into registers, 16 bytes at a time,
// one line ahead of the MFMAs that use them.  No LDS ring and no barrier stand between a load and
// its use; the waves' sums meet once in the LDS at the end, so there are no partial outputs in
// memory and no second launch.  The activation rows come from the L2 (every workgroup reads them);
// up to two 16-row blocks that traffic stays below the weight's share of the L1 fill.  Against split-K
// over 256-row tiles and its second pass (us): 1 x 4096 x 4096 INT8 12.4 -> 4.9 (3.4 TB/s), 16 rows
// 12.7 -> 6.3; 16 x 4096 x 14336 BF16 212 -> 28.7 (4.1 TB/s), unsplit there.  Two or four lines ahead,
// at half the occupancy, measured the same to 15% slower.
//
// INT32 sums are exact in any order.  Float modes add the eight waves' FP32 chains in wave order.
#pragma once

#include <type_traits>

#include "gemm_epilogue.h"

namespace m5k {
namespace gemm {
namespace decode {

using detail::EpiParams;

constexpr int WAVES = 8;

// One line's fragments: chunks (lane >> 4) and 4 + (lane >> 4) of row (lane & 15) of each block.
template <int MODE, int FM>
struct Line {
  Frag<MODE> a[FM], b;
};

template <int MODE, int FM>
__device__ __forceinline__ void load_line(Line<MODE, FM>& f, const uint8_t* const (&ap)[FM], const uint8_t* bp, int64_t ofs) {
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    f.a[i].lo = *reinterpret_cast<const v4i*>(ap[i] + ofs);
    f.a[i].hi = *reinterpret_cast<const v4i*>(ap[i] + ofs + 64);
  }
  f.b.lo = *reinterpret_cast<const v4i*>(bp + ofs);
  f.b.hi = *reinterpret_cast<const v4i*>(bp + ofs + 64);
}

// The last line of a K that is no multiple of 128 bytes: chunks at or past K read as zero (their
// addresses are moved back into the row).
template <int MODE, int FM>
__device__ __forceinline__ void load_line_tail(Line<MODE, FM>& f, const uint8_t* const (&ap)[FM], const uint8_t* bp,
                                               int64_t ofs, int64_t left, int chunk) {
  const bool lo = chunk < left, hi = chunk + 64 < left;
  const int64_t olo = lo ? ofs : -static_cast<int64_t>(chunk), ohi = hi ? ofs + 64 : -static_cast<int64_t>(chunk);
  const v4i z = {0, 0, 0, 0};
  auto pick = [&](const uint8_t* p, Frag<MODE>& r) {
    const v4i l = *reinterpret_cast<const v4i*>(p + olo), h = *reinterpret_cast<const v4i*>(p + ohi);
    r.lo = lo ? l : z;
    r.hi = hi ? h : z;
  };
#pragma unroll
  for (int i = 0; i < FM; ++i) pick(ap[i], f.a[i]);
  pick(bp, f.b);
}

template <int MODE, int FM>
__device__ __forceinline__ void mfma_line(typename Traits<MODE>::acc_t (&acc)[FM], const Line<MODE, FM>& f) {
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    mfma<MODE>(acc[i], f.a[i], f.b);
    if constexpr (MODE != F8) mfma<MODE>(acc[i], Frag<MODE>{f.a[i].hi, {}}, Frag<MODE>{f.b.hi, {}});
  }
}

// Rows 16-byte multiples, bases 16-byte aligned, M <= 16 FM.
template <int MODE, int FM, int OUT_DT, int BIAS, int GATE>
__global__ __launch_bounds__(64 * WAVES, 4) void gemm_decode_kernel(const uint8_t* __restrict__ A,
                                                                 const uint8_t* __restrict__ B, int M, int N, int64_t Kb,
                                                                 EpiParams p) {
  using acc_t = typename Traits<MODE>::acc_t;
  using sum_t = typename std::conditional<MODE == I8, int32_t, float>::type;
  __shared__ __attribute__((aligned(16))) sum_t red[WAVES][FM][256];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 15, chunk = (lane >> 4) * 16;
  const int n0 = static_cast<int>(blockIdx.x) * 16;
  // Rows past M or N repeat the last one; their sums are never stored.
  const uint8_t* ap[FM];
#pragma unroll
  for (int i = 0; i < FM; ++i) ap[i] = A + static_cast<int64_t>(min(16 * i + frow, M - 1)) * Kb + chunk;
  const uint8_t* bp = B + static_cast<int64_t>(min(n0 + frow, N - 1)) * Kb + chunk;
  const int64_t whole = Kb / BKB;  // lines this kernel loads without a bounds check
  acc_t acc[FM];
#pragma unroll
  for (int i = 0; i < FM; ++i) acc[i] = acc_t{};
  // Wave w takes lines w, w + 8, ...: line t of this wave starts at (8 t + w) * 128.
  const int64_t mine = whole > wave ? (whole - wave + WAVES - 1) / WAVES : 0;
  Line<MODE, FM> f0, f1;
  auto load = [&](Line<MODE, FM>& d, int64_t t) { load_line(d, ap, bp, (t * WAVES + wave) * BKB); };
  if (mine > 0) load(f0, 0);
  int64_t t = 0;
  for (; t + 2 <= mine; t += 2) {
    load(f1, t + 1);
    mfma_line(acc, f0);
    if (t + 2 < mine) load(f0, t + 2);
    mfma_line(acc, f1);
  }
  if (t < mine) mfma_line(acc, f0);
  if (whole * BKB < Kb && whole % WAVES == wave) {
    Line<MODE, FM> g;
    load_line_tail(g, ap, bp, whole * BKB, Kb - whole * BKB, chunk);
    mfma_line(acc, g);
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) *reinterpret_cast<acc_t*>(&red[wave][i][lane * 4]) = acc[i];
  __syncthreads();
  // Sum e of block i: slot 4 * lane + r holds row 4 (lane >> 4) + r, column lane & 15.
  for (int e = threadIdx.x; e < FM * 256; e += 64 * WAVES) {
    const int i = e >> 8, cell = e & 255, col = cell & 15, row = cell >> 4;
    const int slot = ((row >> 2) * 16 + col) * 4 + (row & 3);
    const int m = 16 * i + row, n = n0 + col;
    if (m >= M || n >= N) continue;
    sum_t v = red[0][i][slot];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v += red[w][i][slot];
    store_elem<OUT_DT>(p.c, static_cast<int64_t>(m) * N + n, detail::result_value<MODE, BIAS, GATE>(p, v, m, n, N));
  }
}

}  // namespace decode
}  // namespace gemm
}  // namespace m5k
