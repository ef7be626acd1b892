// Small-tile MFMA GEMM for outputs whose 256 x 256 tiles would leave CUs idle (short and middle M),
// and for operands whose rows are not 16-byte multiples.
//
// A workgroup of eight waves computes a TM x TN tile (128 x 128 or 64 x 64).  The waves
// form a 2 x 2 grid of (TM/2) x (TN/2) sub-tiles in two K groups: a stage holds two sub-steps of K
// (64 bytes each; 128 for FP8, whose MFMA takes 128), and group g multiplies sub-step g of every
// stage.  A wave thus reads half of each stage, so a 128 x 128 tile moves 64 KiB of fragments per
// 32 KiB stage (8 waves of 64 x 32 over the whole K would move 96 KiB, more than the MFMAs cover)
// while two waves per SIMD hide each other's latencies.  At the end the groups exchange halves of
// their accumulators through the LDS, and each wave finishes a quarter-height strip: the geometry
// of Grid<4, 2, TN, TM>, whose epilogue runs unchanged.
//
// NST stages (2 to 4) ring through the LDS, all but the one being read in flight: 32 to 48 KiB of weights
// per CU under way against 16 KiB for the 256-row tiles' two-stage loop, which is what a short-M product,
// bound by streaming the weight, needs.  INT8, us, 256-row tiles (split over K with a second pass for
// the partial sums where that paid) against these, unsplit: 128 x 4096 x 4096 16.2 -> 9.7; 128 x 5376
// x 14336 31.1 -> 24.3; 512 x 7168 x 5376 36.1 -> 25.2; 128 x 21504 x 5376 49.7 -> 33.5; 1024 x 4096
// x 4096 29.4 -> 21.5; BF16 128 x 5376 x 5120 58.6 -> 18.7, 1024 x 4096 x 4096 52.2 -> 37.3.
//
// INT32 sums are exact in any order.  Float modes sum the two K groups' FP32 chains at the end:
// another order than one chain over K, with half as many roundings along each.  Every tile here
// gives the same bits: group g takes the same half of every 128-byte line (FP8: every other line).
#pragma once

#include "gemm_epilogue.h"

namespace m5k {
namespace gemm {
namespace ring {

using detail::EpiParams;

template <int MODE_, int TM_, int TN_, int NST_, int PLANES_ = (MODE_ == F8 ? 2 : 1)>
struct Cfg {
  static constexpr int MODE = MODE_, TM = TM_, TN = TN_, NST = NST_;
  static constexpr int PLANES = PLANES_;  // 128-byte row planes per stage
  static constexpr int ROWS = TM + TN;
  static constexpr int PLANE_BYTES = ROWS * BKB;
  static constexpr int STAGE = PLANES * PLANE_BYTES;
  static constexpr int STAGE_K = PLANES * BKB;  // K bytes per stage
  static constexpr int Q = STAGE / 8192;        // 1 KiB DMA instructions per wave and stage
  static constexpr int WM = TM / 2, WN = TN / 2;
  static constexpr int FM = WM / 16, FN = WN / 16;
  using G = Grid<4, 2, TN, TM>;  // geometry after the exchange
  static constexpr int EXCHANGE = TM * TN * 4;
  static constexpr int LDS_AT_LEAST = EXCHANGE > EpiLayout<G>::BYTES ? EXCHANGE : EpiLayout<G>::BYTES;
  static constexpr int LDS = NST * STAGE > LDS_AT_LEAST ? NST * STAGE : LDS_AT_LEAST;
  static_assert(Traits<MODE>::MD == 16, "16 x 16 blocks");
  static_assert(STAGE % 8192 == 0 && TM % 16 == 0 && FM % 2 == 0, "whole DMA instructions, halves of block rows");
  static_assert(LDS <= 160 * 1024 && NST >= 2, "LDS per CU");
};

template <class C>
struct Frags {
  Frag<C::MODE> a[C::FM];
  Frag<C::MODE> b[C::FN];
};

template <class C>
using Acc = typename Traits<C::MODE>::acc_t[C::FM][C::FN];

template <class C>
using HalfAcc = typename Traits<C::MODE>::acc_t[C::FM / 2][C::FN];

// Wave w: column strip w & 1, K group (w >> 1) & 1, row strip w >> 2.
struct WaveId {
  int wn, kg, wm;
  __device__ __forceinline__ explicit WaveId(int wave) : wn(wave & 1), kg((wave >> 1) & 1), wm(wave >> 2) {}
};

// Lane addresses of the wave's fragments: byte offsets inside a stage of block row 0, chunk term
// included (chunk 4 kg + fq of the 128-byte row; FP8: plane kg, chunks fq and 4 + fq).
template <class C>
struct FragAddr {
  uint32_t a0, a1, b0, b1;
  __device__ __forceinline__ FragAddr(const WaveId& w, int lane) {
    const int frow = lane & 15, fq = lane >> 4, fsw = swz(frow);
    const uint32_t ra = static_cast<uint32_t>((w.wm * C::WM + frow) * BKB);
    const uint32_t rb = static_cast<uint32_t>((C::TM + w.wn * C::WN + frow) * BKB);
    if constexpr (C::MODE == F8) {
      const uint32_t plane = static_cast<uint32_t>(w.kg * C::PLANE_BYTES);
      const uint32_t c0 = static_cast<uint32_t>((fq ^ fsw) << 4), c1 = static_cast<uint32_t>(((4 + fq) ^ fsw) << 4);
      a0 = plane + ra + c0; a1 = plane + ra + c1;
      b0 = plane + rb + c0; b1 = plane + rb + c1;
    } else {
      // The same half of every 128-byte line, so that each group's K order, and with it every bit of a
      // float sum, does not depend on the tile.
      const uint32_t c = static_cast<uint32_t>(((4 * w.kg + fq) ^ fsw) << 4);
      a0 = ra + c; a1 = a0 + C::PLANE_BYTES;
      b0 = rb + c; b1 = b0 + C::PLANE_BYTES;
    }
  }
};

template <class C>
__device__ __forceinline__ void read_block(const uint8_t* st, uint32_t o0, uint32_t o1, int blk, Frag<C::MODE>& f) {
  f.lo = *reinterpret_cast<const v4i*>(st + o0 + blk * 16 * BKB);
  if constexpr (C::PLANES == 2) f.hi = *reinterpret_cast<const v4i*>(st + o1 + blk * 16 * BKB);
}

template <class C>
__device__ __forceinline__ void read_stage(const uint8_t* st, const FragAddr<C>& ad, Frags<C>& f) {
#pragma unroll
  for (int j = 0; j < C::FN; ++j) read_block<C>(st, ad.b0, ad.b1, j, f.b[j]);
#pragma unroll
  for (int i = 0; i < C::FM; ++i) read_block<C>(st, ad.a0, ad.a1, i, f.a[i]);
}

// MFMAs of `cur`, the reads of the next stage's fragments spread before its block rows (B
// fragments first); fences keep each read ahead of the row it is placed before.
template <class C>
__device__ __forceinline__ void mfma_reading(Acc<C>& acc, const Frags<C>& cur, Frags<C>& nxt, const uint8_t* st,
                                             const FragAddr<C>& ad) {
  constexpr int NR = C::FM + C::FN;
#pragma unroll
  for (int i = 0; i < C::FM; ++i) {
#pragma unroll
    for (int r = i * NR / C::FM; r < (i + 1) * NR / C::FM; ++r) {
      if (r < C::FN) read_block<C>(st, ad.b0, ad.b1, r, nxt.b[r]);
      else read_block<C>(st, ad.a0, ad.a1, r - C::FN, nxt.a[r - C::FN]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < C::FN; ++j) mfma<C::MODE>(acc[i][j], cur.a[i], cur.b[j]);
    if constexpr (C::PLANES == 2 && C::MODE != F8) {
#pragma unroll
      for (int j = 0; j < C::FN; ++j)
        mfma<C::MODE>(acc[i][j], Frag<C::MODE>{cur.a[i].hi, {}}, Frag<C::MODE>{cur.b[j].hi, {}});
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The K groups' sums: each wave gives its partner (same sub-tile, other group) one half of its
// block rows and adds the partner's to the half it keeps.  Starts after a barrier that freed the
// LDS and ends with one.
template <class C>
__device__ __forceinline__ void exchange(const Acc<C>& acc, HalfAcc<C>& out, uint8_t* lds, int wave, int lane) {
  constexpr int H = C::FM / 2;
  using acc_t = typename Traits<C::MODE>::acc_t;
  acc_t* slots = reinterpret_cast<acc_t*>(lds);
  const bool high = ((wave >> 1) & 1) != 0;
#pragma unroll
  for (int i = 0; i < H; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
      slots[((wave * H + i) * C::FN + j) * 64 + lane] = high ? acc[i][j] : acc[H + i][j];
  __syncthreads();
  const int partner = wave ^ 2;
#pragma unroll
  for (int i = 0; i < H; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
      out[i][j] = (high ? acc[H + i][j] : acc[i][j]) + slots[((partner * H + i) * C::FN + j) * 64 + lane];
  __syncthreads();
}

// Ring stages of a row of Kb bytes.
template <class C>
__host__ __device__ constexpr int64_t stages(int64_t kb) {
  return (kb + C::STAGE_K - 1) / C::STAGE_K;
}

// Stages [kt_begin, kt_begin + kt_count) of the tile at (m0, n0), by direct-to-LDS loads (rows
// 16-byte multiples of at most 2^23 bytes, bases 16-byte aligned).  Every wave moves Q groups of
// eight rows per stage, A rows first; rows past M or N and chunks past K read as zero through
// out-of-range buffer offsets, stages past the range through an empty window.
//
// Per stage kt: wait for own loads of stage kt + 1 (and the reads of stage kt, issued one stage
// earlier); barrier; load stage kt + NST into the buffer just read; read the fragments of stage
// kt + 1 among the MFMAs of stage kt.
template <class C>
__device__ __forceinline__ void mainloop(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, int M, int N,
                                         int64_t Kb, int m0, int n0, Acc<C>& acc, int64_t kt_begin, int64_t kt_count,
                                         uint8_t* lds) {
  constexpr uint32_t kOob = 0x80000000u;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const WaveId id(wave);
  const int rows_a = min(M - m0, C::TM), rows_b = min(N - n0, C::TN);
  const uint8_t* a_win = A + static_cast<int64_t>(m0) * Kb;
  const uint8_t* b_win = B + static_cast<int64_t>(n0) * Kb;
  const uint32_t rec_a = static_cast<uint32_t>(rows_a * Kb), rec_b = static_cast<uint32_t>(rows_b * Kb);
  uint32_t voff[C::Q], lchunk[C::Q];
#pragma unroll
  for (int i = 0; i < C::Q; ++i) {
    const int rg = (wave * C::Q + i) % (C::ROWS / 8);
    const bool is_b = rg * 8 >= C::TM;
    const int r = rg * 8 - (is_b ? C::TM : 0) + (lane >> 3);
    lchunk[i] = static_cast<uint32_t>(((lane & 7) ^ swz(r)) << 4);
    voff[i] = r < (is_b ? rows_b : rows_a) ? static_cast<uint32_t>(r * Kb) + lchunk[i] : kOob;
  }
  auto dma = [&](uint32_t buf, int64_t kr) {
#pragma unroll
    for (int i = 0; i < C::Q; ++i) {
      const int g = wave * C::Q + i, plane = g / (C::ROWS / 8), rg = g % (C::ROWS / 8);
      const bool is_b = rg * 8 >= C::TM;
      const int64_t kofs = ((kt_begin + kr) * C::PLANES + plane) * BKB;
      const bool live = kr < kt_count && kofs < Kb;
      const uint32_t kill = kofs + static_cast<int64_t>(lchunk[i]) < Kb ? 0u : kOob;
      const uint32_t rec = live ? (is_b ? rec_b : rec_a) : 0u;
      const v4i rsrc = window_rsrc(is_b ? b_win : a_win, rec, live ? static_cast<uint32_t>(kofs) : 0u);
      dma16<true>(lds_addr(lds) + buf + static_cast<uint32_t>(plane * C::PLANE_BYTES + rg * 1024), voff[i] | kill, rsrc);
    }
  };
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) acc[i][j] = typename Traits<C::MODE>::acc_t{};
  const FragAddr<C> ad(id, lane);
  Frags<C> f0, f1;
#pragma unroll
  for (int st = 0; st < C::NST; ++st) dma(st * C::STAGE, st);
  wait_stage<C::Q * (C::NST - 1)>();
  stage_barrier();
  read_stage<C>(lds, ad, f0);
  uint32_t cur = 0;
  auto stage = [&](const Frags<C>& fc, Frags<C>& fn, int64_t kt) {
    const uint32_t nxt = cur + C::STAGE == C::NST * C::STAGE ? 0u : cur + C::STAGE;
    wait_stage<C::Q * (C::NST - 2)>();
    // The loads below overwrite the buffer of stage kt: every wave's reads of it have returned.
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    stage_barrier();
    dma(cur, kt + C::NST);
    mfma_reading<C>(acc, fc, fn, lds + nxt, ad);
    cur = nxt;
  };
  for (int64_t kt = 0; kt < kt_count; kt += 2) {
    stage(f0, f1, kt);
    if (kt + 1 < kt_count) stage(f1, f0, kt + 1);
  }
  // Drain the trailing loads (zeros) before the LDS is reused.
  wait_stage<0>();
  __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  stage_barrier();
}

// The 16 bytes at any byte address p of a row of which `left` bytes remain there; bytes past the row's
// end read as zero, and none of them is touched: a partial chunk is loaded so that it ends with the
// row, and shifted down (rows of under 16 bytes: byte by byte).
__device__ __forceinline__ v4i load_tail_chunk(const uint8_t* p, int64_t left, int64_t kb) {
  v4i v = {0, 0, 0, 0};
  if (left <= 0) return v;
  if (kb < 16) {
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 15; ++e)
      if (e < left) w[e >> 2] |= static_cast<uint32_t>(p[e]) << (8 * (e & 3));
    return v4i{static_cast<int>(w[0]), static_cast<int>(w[1]), static_cast<int>(w[2]), static_cast<int>(w[3])};
  }
  const int drop = left >= 16 ? 0 : static_cast<int>(16 - left);  // bytes of the load before p
  uint64_t q[2];
  __builtin_memcpy(q, p - drop, 16);
  const int s = 8 * (drop & 7);
  const uint64_t lo = drop >= 8 ? q[1] : q[0], hi = drop >= 8 ? 0 : q[1];
  q[0] = (lo >> s) | (s ? hi << (64 - s) : 0);
  q[1] = hi >> s;
  __builtin_memcpy(&v, q, 16);
  return v;
}

// The same tile for rows or bases that are not 16-byte aligned (odd K): a wave loads its share of a
// stage into registers with unaligned 16-byte loads, AHEAD stages before they are written to the LDS,
// in the layout that mainloop's loads give.  Two stage buffers.  300 x 520 x 1000 INT8: 127 us byte by
// byte through one buffer with a full wait per stage, 9.2 us one stage ahead with a byte-by-byte tail,
// 8.3 us this way (aligned operands of that size: 5.5 us).
template <class C>
__device__ __forceinline__ void mainloop_unaligned(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, int M,
                                                   int N, int64_t Kb, int m0, int n0, Acc<C>& acc, uint8_t* lds) {
  static_assert(C::NST >= 2 && C::PLANES == 1, "two buffers of one 128-byte plane");
  constexpr int AHEAD = 3;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const WaveId id(wave);
  const uint8_t* src[C::Q];
  int lchunk[C::Q];
  bool in[C::Q];
#pragma unroll
  for (int i = 0; i < C::Q; ++i) {
    const int rg = wave * C::Q + i;
    const bool is_b = rg * 8 >= C::TM;
    const int r = rg * 8 - (is_b ? C::TM : 0) + (lane >> 3);
    const int64_t row = (is_b ? n0 : m0) + static_cast<int64_t>(r);
    in[i] = row < (is_b ? N : M);
    lchunk[i] = ((lane & 7) ^ swz(r)) << 4;
    src[i] = (is_b ? B : A) + (in[i] ? row : 0) * Kb + lchunk[i];
  }
  const int64_t count = stages<C>(Kb), whole = Kb / BKB;
  v4i regs[AHEAD][C::Q];
  auto load = [&](v4i (&r)[C::Q], int64_t kt) {
#pragma unroll
    for (int i = 0; i < C::Q; ++i) {
      r[i] = v4i{0, 0, 0, 0};
      if (kt < whole) {  // uniform
        if (in[i]) __builtin_memcpy(&r[i], src[i] + kt * BKB, 16);
      } else if (kt < count) {
        r[i] = load_tail_chunk(src[i] + kt * BKB, in[i] ? Kb - kt * BKB - lchunk[i] : 0, Kb);
      }
    }
  };
  auto store = [&](const v4i (&r)[C::Q], int buf) {
#pragma unroll
    for (int i = 0; i < C::Q; ++i)
      *reinterpret_cast<v4i*>(lds + buf * C::STAGE + (wave * C::Q + i) * 1024 + lane * 16) = r[i];
  };
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) acc[i][j] = typename Traits<C::MODE>::acc_t{};
  const FragAddr<C> ad(id, lane);
#pragma unroll
  for (int d = 0; d < AHEAD; ++d) load(regs[d], d);
  store(regs[0], 0);
  load(regs[0], AHEAD);
  __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  stage_barrier();
  // Stage kt + 1 waits in register set (kt + 1) % AHEAD; kt advances AHEAD stages per pass (the
  // trailing ones hold zeros), so the sets are compile-time.
  auto step = [&](auto set_tag, int64_t kt) {
    constexpr int SET = (decltype(set_tag)::value + 1) % AHEAD;
    const int buf = static_cast<int>(kt & 1);
    Frags<C> f;
    read_stage<C>(lds + buf * C::STAGE, ad, f);
    store(regs[SET], buf ^ 1);  // the buffer's last reads ended before the barrier
    load(regs[SET], kt + 1 + AHEAD);
#pragma unroll
    for (int i = 0; i < C::FM; ++i)
#pragma unroll
      for (int j = 0; j < C::FN; ++j) mfma<C::MODE>(acc[i][j], f.a[i], f.b[j]);
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    stage_barrier();
  };
  for (int64_t kt = 0; kt < count; kt += AHEAD) {
    step(std::integral_constant<int, 0>{}, kt);
    if (kt + 1 < count) step(std::integral_constant<int, 1>{}, kt + 1);
    if (kt + 2 < count) step(std::integral_constant<int, 2>{}, kt + 2);
  }
}

// One TM x TN tile per workgroup over all of K.
template <class C, bool ALIGNED, int OUT_DT, int BIAS, int GATE>
__global__ __launch_bounds__(512, 1) void gemm_ring_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                           int M, int N, int64_t Kb, EpiParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[C::LDS];
  using G = typename C::G;
  const int tiles_m = (M + C::TM - 1) / C::TM, tiles_n = (N + C::TN - 1) / C::TN;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * C::TM, n0 = tn * C::TN;
  const TileScalePrefetch<G> pre = detail::prefetch_scales<C::MODE, false, G>(p, M, N, m0, n0);
  Acc<C> acc;
  if constexpr (ALIGNED) mainloop<C>(A, B, M, N, Kb, m0, n0, acc, 0, stages<C>(Kb), lds);
  else mainloop_unaligned<C>(A, B, M, N, Kb, m0, n0, acc, lds);
  HalfAcc<C> half;
  exchange<C>(acc, half, lds, threadIdx.x >> 6, threadIdx.x & 63);
  detail::epilogue<C::MODE, OUT_DT, BIAS, GATE, false, G>(half, M, N, m0, n0, p, pre, lds);
}

// Split-K form: workgroup (tile, s) leaves the raw sums of K range s in partial[s][M][N] for
// splitk_epilogue_kernel.
template <class C, class P>
__global__ __launch_bounds__(512, 1) void gemm_ring_splitk_kernel(const uint8_t* __restrict__ A,
                                                                  const uint8_t* __restrict__ B, int M, int N,
                                                                  int64_t Kb, int splits, int64_t stages_per_split,
                                                                  P* __restrict__ partial) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[C::LDS];
  const int tiles_m = (M + C::TM - 1) / C::TM, tiles_n = (N + C::TN - 1) / C::TN;
  const int tile = static_cast<int>(blockIdx.x) / splits, s = static_cast<int>(blockIdx.x) % splits;
  int tm, tn;
  tile_coords(tile, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * C::TM, n0 = tn * C::TN;
  const int64_t total = stages<C>(Kb);
  const int64_t kt0 = s * stages_per_split;
  const int64_t kt1 = kt0 + stages_per_split < total ? kt0 + stages_per_split : total;
  Acc<C> acc;
  mainloop<C>(A, B, M, N, Kb, m0, n0, acc, kt0, kt1 - kt0, lds);
  HalfAcc<C> half;
  exchange<C>(acc, half, lds, threadIdx.x >> 6, threadIdx.x & 63);
  P* out = partial + static_cast<int64_t>(s) * M * N;
  for_each_acc<typename C::G>(half, m0, n0, [&](int m, int n, auto v) {
    if (m < M && n < N) out[static_cast<int64_t>(m) * N + n] = v;
  });
}

}  // namespace ring
}  // namespace gemm
}  // namespace m5k
