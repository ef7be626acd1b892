// Epilogues of the W8A8 / FP8 / BF16 / FP16 linear layers: a tile of MFMA sums, or one sum, to the
// output.
//
// Contract: src/m5kernels/metal.py:158-269 (gemm) with the epilogue strings of
// metal.py:88-128:
//   quantized  C = O(float(acc) * AS[row] * BS[col])            (left to right, FP32)
//   + bias     C = O(float(acc) * AS[row] * BS[col] + Bias[..])  (before the output cast)
//   gated      branch = bf16(value); C = bf16(float(Residual) + float(branch) * float(Gate[..]))
//   float      C = O(float(acc))
// The library is compiled with -ffp-contract=off so none of these products and sums is
// fused into an FMA: the FP32 rounding sequence is exactly the one written above.  For FP16 outputs the
// compiler joins the last FP32 operation and the cast into one v_fma_mixlo_f16, which rounds once: such
// an output can lie one FP16 step from the rounded FP32 one (the same in every kernel of this library).
#pragma once
#include "gemm_core.h"

namespace m5k {
namespace gemm {
namespace detail {

enum { EPI_NONE = 0, EPI_VECTOR = 1, EPI_TABLE = 2 };

struct EpiParams {
  const float* sa;
  const float* sb;
  void* c;
  const float* bias;
  const int32_t* bias_map;
  const uint16_t* residual;
  const uint16_t* gate;
  const int32_t* gate_map;
  int coalesced;  // 16-bit output with N % 8 == 0 and 16-byte aligned c / residual / gate
};

// RAW: write INT32 accumulators (I8 only).
// Wave grid used by every GEMM kernel of the library.
using KernelGrid = Grid8;

// The tile's scales ahead of the main loop (quantized modes with a scale epilogue; nothing for the
// others).
template <int MODE, bool RAW, class G>
__device__ __forceinline__ TileScalePrefetch<G> prefetch_scales(const EpiParams& p, int M, int N, int m0, int n0) {
  if constexpr ((MODE == I8 || MODE == F8) && !RAW) return TileScalePrefetch<G>(p.sa, p.sb, M, N, m0, n0);
  else return TileScalePrefetch<G>(nullptr, nullptr, 0, 0, 0, 0);
}

// Scale epilogue of one 256 x G::TN tile (every thread of the workgroup calls it; the LDS is
// free).  RAW writes the INT32 accumulators.  The per-row and per-column operands of the
// lane's elements (scales, bias vector) are loaded in one batch before the arithmetic, and a
// bias table's offsets and values one block row at a time, so the epilogue waits for memory a
// few times instead of once per element.
template <int MODE, int OUT_DT, int BIAS, int GATE, bool RAW, class G = KernelGrid>
__device__ __forceinline__ void epilogue(const AccTile<MODE, G>& acc, int M, int N, int m0, int n0,
                                         const EpiParams& p, const TileScalePrefetch<G>& pre, uint8_t* lds = g_lds) {
  using Geo = AccGeom<MODE, G>;
  constexpr bool QUANT = MODE == I8 || MODE == F8;
  const int tid = tid_after_mainloop();
  const Geo geo(tid);
  if constexpr (RAW) {
#pragma unroll
    for (int i = 0; i < Geo::FM; ++i)
#pragma unroll
      for (int j = 0; j < Geo::FN; ++j)
#pragma unroll
        for (int e = 0; e < Geo::PER; ++e) {
          const int m = m0 + geo.row(i, e), n = n0 + geo.col(j);
          if (m < M && n < N) static_cast<int32_t*>(p.c)[(int64_t)m * N + n] = acc[i][j][e];
        }
    return;
  } else {
    float cs[QUANT ? Geo::FN : 1];
    const float* sc = nullptr;
    if constexpr (QUANT) {
      const TileScales<G> ts(pre, tid, lds);
      sc = ts.s;
#pragma unroll
      for (int j = 0; j < Geo::FN; ++j) cs[j] = ts.col(geo.col(j));
    }
    float bvec[BIAS == EPI_VECTOR ? Geo::FN : 1];
    if constexpr (BIAS == EPI_VECTOR) {
#pragma unroll
      for (int j = 0; j < Geo::FN; ++j) {
        const int n = n0 + geo.col(j);
        bvec[j] = n < N ? p.bias[n] : 0.0f;
      }
    }
    // FP32 value of block row i's elements: the scale epilogue, then the bias (a bias table's
    // row offsets and values are loaded per block row, two batches).
    auto row_values = [&](int i, float (&val)[Geo::FN][Geo::PER]) {
      float rs[QUANT ? Geo::PER : 1];
      if constexpr (QUANT) {
#pragma unroll
        for (int e = 0; e < Geo::PER; ++e) rs[e] = sc[geo.row(i, e)];
      }
      float tb[BIAS == EPI_TABLE ? Geo::FN : 1][BIAS == EPI_TABLE ? Geo::PER : 1];
      if constexpr (BIAS == EPI_TABLE) {
        int64_t brow[Geo::PER];
#pragma unroll
        for (int e = 0; e < Geo::PER; ++e) {
          const int m = m0 + geo.row(i, e);
          brow[e] = m < M ? (int64_t)p.bias_map[m] * N : 0;
        }
#pragma unroll
        for (int j = 0; j < Geo::FN; ++j)
#pragma unroll
          for (int e = 0; e < Geo::PER; ++e) {
            const int m = m0 + geo.row(i, e), n = n0 + geo.col(j);
            tb[j][e] = (m < M && n < N) ? p.bias[brow[e] + n] : 0.0f;
          }
      }
#pragma unroll
      for (int j = 0; j < Geo::FN; ++j)
#pragma unroll
        for (int e = 0; e < Geo::PER; ++e) {
          float value;
          if constexpr (QUANT) value = (static_cast<float>(acc[i][j][e]) * rs[e]) * cs[j];
          else value = acc[i][j][e];
          if constexpr (BIAS == EPI_VECTOR) value = value + bvec[j];
          if constexpr (BIAS == EPI_TABLE) value = value + tb[j][e];
          val[j][e] = value;
        }
    };

    // 16-bit outputs: stage the rounded tile (the BF16 branch for the gated form) in the LDS the
    // main loop has released, then write whole 512-byte tile rows with 16-byte streaming stores.
    if constexpr (OUT_DT == M5K_BF16 || OUT_DT == M5K_F16) {
      if (p.coalesced) {
        uint16_t* tile = reinterpret_cast<uint16_t*>(lds);
#pragma unroll
        for (int i = 0; i < Geo::FM; ++i) {
          float val[Geo::FN][Geo::PER];
          row_values(i, val);
#pragma unroll
          for (int j = 0; j < Geo::FN; ++j)
#pragma unroll
            for (int e = 0; e < Geo::PER; ++e) {
              // Entries past M or N are staged unmasked: the write-out below skips them.
              const int r = geo.row(i, e), c = geo.col(j);
              const float value = val[j][e];
              tile[r * EpiLayout<G>::STRIDE + c] = static_cast<uint16_t>(
                  GATE != EPI_NONE || OUT_DT == M5K_BF16 ? f32_to_bf16_bits(value) : f32_to_f16_bits(value));
            }
        }
        __syncthreads();
        constexpr int CPR = G::TN / 8;  // 16-byte chunks per tile row
        for (int c = threadIdx.x; c < G::TM * CPR; c += G::THREADS) {
          const int r = c / CPR, cc = c % CPR;
          const int m = m0 + r, n = n0 + 8 * cc;
          if (m >= M || n >= N) continue;  // N % 8 == 0: a chunk is wholly in or out
          uint4 w = *reinterpret_cast<const uint4*>(tile + r * EpiLayout<G>::STRIDE + 8 * cc);
          const int64_t idx = (int64_t)m * N + n;
          if constexpr (GATE != EPI_NONE) {
            const int64_t goff = GATE == EPI_TABLE ? (int64_t)p.gate_map[m] * N : 0;
            const uint4 rw = *reinterpret_cast<const uint4*>(p.residual + idx);
            const uint4 gw = *reinterpret_cast<const uint4*>(p.gate + goff + n);
            const uint32_t bs[4] = {w.x, w.y, w.z, w.w}, rs[4] = {rw.x, rw.y, rw.z, rw.w},
                           gs[4] = {gw.x, gw.y, gw.z, gw.w};
            uint32_t out[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const float lo = bf16_bits_to_f32(rs[t] & 0xFFFFu) +
                               bf16_bits_to_f32(bs[t] & 0xFFFFu) * bf16_bits_to_f32(gs[t] & 0xFFFFu);
              const float hi =
                  bf16_bits_to_f32(rs[t] >> 16) + bf16_bits_to_f32(bs[t] >> 16) * bf16_bits_to_f32(gs[t] >> 16);
              out[t] = f32x2_to_bf16x2(lo, hi);
            }
            w = make_uint4(out[0], out[1], out[2], out[3]);
          }
          store_stream16(static_cast<uint16_t*>(p.c) + idx, w);
        }
        return;
      }
    }

#pragma unroll
    for (int i = 0; i < Geo::FM; ++i) {
      float val[Geo::FN][Geo::PER];
      row_values(i, val);
      // The gated form's residual and gate values of this block row, loaded in one batch.
      float res[GATE != EPI_NONE ? Geo::FN : 1][GATE != EPI_NONE ? Geo::PER : 1];
      float gte[GATE != EPI_NONE ? Geo::FN : 1][GATE != EPI_NONE ? Geo::PER : 1];
      if constexpr (GATE != EPI_NONE) {
#pragma unroll
        for (int j = 0; j < Geo::FN; ++j)
#pragma unroll
          for (int e = 0; e < Geo::PER; ++e) {
            const int m = m0 + geo.row(i, e), n = n0 + geo.col(j);
            const bool in = m < M && n < N;
            const int64_t goff = GATE == EPI_TABLE && in ? (int64_t)p.gate_map[m] * N : 0;
            res[j][e] = in ? bf16_bits_to_f32(p.residual[(int64_t)m * N + n]) : 0.0f;
            gte[j][e] = in ? bf16_bits_to_f32(p.gate[goff + n]) : 0.0f;
          }
      }
#pragma unroll
      for (int j = 0; j < Geo::FN; ++j)
#pragma unroll
        for (int e = 0; e < Geo::PER; ++e) {
          const int m = m0 + geo.row(i, e), n = n0 + geo.col(j);
          if (m >= M || n >= N) continue;
          const int64_t idx = (int64_t)m * N + n;
          if constexpr (GATE != EPI_NONE) {
            const float branch = round_through<M5K_BF16>(val[j][e]);
            store_elem<M5K_BF16>(p.c, idx, res[j][e] + branch * gte[j][e]);
          } else {
            store_elem<OUT_DT>(p.c, idx, val[j][e]);
          }
        }
    }
  }
}

// The epilogue of one output element: the FP32 sequence of epilogue() above for the sum v, before
// the output cast.
template <int MODE, int BIAS, int GATE, class P>
__device__ __forceinline__ float result_value(const EpiParams& p, P v, int m, int n, int N) {
  float value = static_cast<float>(v);
  if constexpr (MODE == I8 || MODE == F8) value = (value * p.sa[m]) * p.sb[n];
  if constexpr (BIAS != EPI_NONE) {
    const int64_t boff = BIAS == EPI_TABLE ? (int64_t)p.bias_map[m] * N : 0;
    value = value + p.bias[boff + n];
  }
  if constexpr (GATE != EPI_NONE) {
    const int64_t goff = GATE == EPI_TABLE ? (int64_t)p.gate_map[m] * N : 0;
    const float branch = round_through<M5K_BF16>(value);
    const float res = bf16_bits_to_f32(p.residual[static_cast<int64_t>(m) * N + n]);
    value = res + branch * bf16_bits_to_f32(p.gate[goff + n]);
  }
  return value;
}

}  // namespace detail
}  // namespace gemm
}  // namespace m5k
