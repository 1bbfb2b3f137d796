// The lanes' fp32 row contractions: router logits and the shared expert below the matrix-core widths; weights streamed
// once from HBM in their file layout (210-byte Q6_K superblocks / 34-byte Q8_0 blocks), dequantised in registers.  (The
// routed experts and longer rows go through the digit contraction, digits.h.)  Replaces the reference's shared-expert
// gemv / tiled fp32 families (crates/xabe-cuda/src/kernels/moe.rs:3425-3725, :4082-4227).
//
// One wavefront "step" covers 2048 contraction elements of a row: 8 Q6_K superblocks
// (1680 B) or 64 Q8_0 blocks (2176 B), 32 elements per lane.  Rows shorter than 2048
// pack RPS = 2048/K rows into a step; longer rows take KS steps, the last one masked.
// Activations for the lane's fixed element positions live in registers, so a row costs
// its own bytes and nothing else.
//
// Numerics contract: the value of (row, token) is computed by one fixed sequence of
// fp32 operations that does not depend on which other tokens are present, so a token
// decodes to the same bits alone or in a batch (tests/test_gpu_batch_invariance.py).
#pragma once

#include <type_traits>

#include "device_common.h"

namespace xabe {

constexpr int kWavesPerWg = 4;

template <int QUANT>
struct Fmt;
template <>
struct Fmt<kQ6K> {
  using Raw = Q6Raw;
  static constexpr uint32_t kChunkBytes = 8 * kQ6KBytes;
  static constexpr int kBlockElems = 256;
  static constexpr int kBlockBytes = kQ6KBytes;
};
template <>
struct Fmt<kQ8_0> {
  using Raw = Q8Raw;
  static constexpr uint32_t kChunkBytes = 64 * kQ8Bytes;
  static constexpr int kBlockElems = 32;
  static constexpr int kBlockBytes = kQ8Bytes;
};

template <>
struct Fmt<kF32> {
  using Raw = F32Raw;
  static constexpr uint32_t kChunkBytes = 2048 * 4;
  static constexpr int kBlockElems = 1;
  static constexpr int kBlockBytes = 4;
};

struct LaneGeom {
  int lane, slot, half, l8;
  uint32_t lane_off;  // byte offset of the lane's block inside a step's chunk
};

template <int QUANT>
__device__ __forceinline__ LaneGeom lane_geom(int lane = (int)__lane_id()) {
  LaneGeom g;
  g.lane = lane;
  g.slot = g.lane >> 3;
  g.half = (g.lane >> 2) & 1;
  g.l8 = g.lane & 3;
  g.lane_off = QUANT == kQ6K ? (uint32_t)g.slot * kQ6KBytes
             : QUANT == kQ8_0 ? (uint32_t)g.lane * kQ8Bytes
                              : (uint32_t)g.lane * 128u;
  return g;
}

// Offset, within a row, of the first of the 32 elements this lane covers in step `k`.
// For Q6_K that is the start of the lane's superblock (positions inside it: q6_pos).
template <int QUANT, int RPS>
__device__ __forceinline__ int lane_koff(const LaneGeom& g, int k) {
  if (QUANT == kQ6K) return ((g.slot % (8 / RPS)) + k * 8) * 256;
  return ((g.lane % (64 / RPS)) + k * 64) * 32;
}

// Eight consecutive activations starting at xrow + off (off a multiple of 4).
__device__ __forceinline__ void load8(const float* __restrict__ xrow, int off, float (&v)[8]) {
  const float4 a = reinterpret_cast<const float4*>(xrow + off)[0];
  const float4 b = reinterpret_cast<const float4*>(xrow + off)[1];
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

template <int QUANT>
__device__ __forceinline__ void load_x(const float* __restrict__ xrow, int koff, bool active, const LaneGeom& g,
                                       float (&x)[32], float (&xs)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // Q6_K: run j of the lane's superblock unit; Q8_0 / fp32: the j-th eight of 32 consecutive elements
    const int off = QUANT == kQ6K ? koff + g.half * 128 + j * 32 + g.l8 * 8 : koff + j * 8;
    if (active) load8(xrow, off, v);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[j * 8 + i] = v[i];
    if (QUANT == kQ6K) {
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) s += v[i];
      xs[j] = -32.0f * s;
    } else {
      xs[j] = 0.0f;
    }
  }
}

template <int QUANT>
__device__ __forceinline__ void raw_zero(typename Fmt<QUANT>::Raw& r);
template <>
__device__ __forceinline__ void raw_zero<kQ6K>(Q6Raw& r) {
  r.qa0 = r.qa1 = r.qb0 = r.qb1 = r.qh0 = r.qh1 = r.sc0 = r.sc1 = r.dh = 0;
}
template <>
__device__ __forceinline__ void raw_zero<kQ8_0>(Q8Raw& r) {
#pragma unroll
  for (int i = 0; i < 8; ++i) r.q[i] = 0;
  r.dh = 0;
}
template <>
__device__ __forceinline__ void raw_zero<kF32>(F32Raw& r) {
#pragma unroll
  for (int i = 0; i < 32; ++i) r.v[i] = 0.0f;
}

// Loads this lane's block of the step that starts at `chunk` (any 2-byte alignment).
// DIRECT: Q6_K fields read at their own alignment (q6_load_direct); the Raw is the same.
template <int QUANT, bool DIRECT = false>
__device__ __forceinline__ void load_raw(const uint8_t* chunk, bool active, const LaneGeom& g,
                                         typename Fmt<QUANT>::Raw& r) {
  if (!active) {
    raw_zero<QUANT>(r);
    return;
  }
  const uint32_t mis = (uint32_t)(reinterpret_cast<uintptr_t>(chunk) & 3u);
  const uint8_t* chunk4 = chunk - mis;
  if constexpr (QUANT == kQ6K && DIRECT) q6_load_direct(chunk4, g.lane_off + mis, g.half, g.l8, r);
  else if constexpr (QUANT == kQ6K) q6_load(chunk4, g.lane_off + mis, g.half, g.l8, r);
  else if constexpr (QUANT == kQ8_0) q8_load(chunk4, g.lane_off + mis, r);
  else f32_load(chunk, g.lane_off, r);
}

template <int QUANT, int TC>
__device__ __forceinline__ void accum(const typename Fmt<QUANT>::Raw& r, const LaneGeom& g, const float (&x)[TC][32],
                                      const float (&xs)[TC][4], float (&tot)[TC]) {
  if constexpr (QUANT == kQ6K) q6_accum<TC>(r, g.l8, x, xs, tot);
  else if constexpr (QUANT == kQ8_0) q8_accum<TC>(r, x, tot);
  else f32_accum<TC>(r, x, tot);
}

// ---------------------------------------------------------------------------------
// matvec_rows: the body every decode kernel shares.
//   NM = 2: out[t][row] = silu(gate_row . x_t) * (up_row . x_t)      (gate/up + SwiGLU)
//   NM = 1: out[t][row] = scale[t] * (w_row . x_t)                    (down / plain GEMV)
// `w0`/`w1` point at row 0 of the matrix (one expert).  Rows [tile0, tile0+tile_rows)
// are split over the workgroup's four wavefronts.  KS > 0: steps per row, activations
// in registers.  KS == 0: steps from K at run time, activations re-read per step.
// ---------------------------------------------------------------------------------
template <int QUANT, int KS, int RPS, int TC, int NM>
__device__ __forceinline__ void matvec_rows(const uint8_t* __restrict__ w0, const uint8_t* __restrict__ w1, int K,
                                            int n_rows, int tile0, int tile_rows,
                                            const float* const (&xrow)[TC], float* const (&out)[TC],
                                            const float (&scale)[TC]) {
  using F = Fmt<QUANT>;
  using Raw = typename F::Raw;
  constexpr int G = 64 / RPS;
  static_assert(RPS == 1 || KS == 1, "short rows take exactly one step");
  const LaneGeom g = lane_geom<QUANT>();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) % kWavesPerWg;  // (four take a tile, however many there are)
  const size_t row_bytes = (size_t)(K / F::kBlockElems) * F::kBlockBytes;
  const int tile_end = min(tile0 + tile_rows, n_rows);

  if constexpr (KS > 0) {
    float x[KS][TC][32];
    float xs[KS][TC][4];
    bool active[KS];
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const int koff = lane_koff<QUANT, RPS>(g, k);
      active[k] = koff < K;
#pragma unroll
      for (int t = 0; t < TC; ++t)
        load_x<QUANT>(xrow[t], koff, active[k], g, x[k][t], xs[k][t]);
    }
    auto load_item = [&](int row0, Raw (&r)[NM][KS]) {
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        const size_t off = (size_t)row0 * row_bytes + (size_t)k * F::kChunkBytes;
        load_raw<QUANT>(w0 + off, active[k], g, r[0][k]);
        if constexpr (NM == 2) load_raw<QUANT>(w1 + off, active[k], g, r[NM - 1][k]);
      }
    };
    auto finish_item = [&](int row0, const Raw (&r)[NM][KS]) {
      float tot[NM][TC];
#pragma unroll
      for (int m = 0; m < NM; ++m) {
#pragma unroll
        for (int t = 0; t < TC; ++t) tot[m][t] = 0.0f;
#pragma unroll
        for (int k = 0; k < KS; ++k) accum<QUANT, TC>(r[m][k], g, x[k], xs[k], tot[m]);
#pragma unroll
        for (int t = 0; t < TC; ++t) tot[m][t] = group_sum<G>(tot[m][t]);
      }
      const int row = row0 + g.lane / G;
      if ((g.lane % G) == 0 && row < n_rows) {
#pragma unroll
        for (int t = 0; t < TC; ++t) {
          const float v = NM == 2 ? silu_f(tot[0][t]) * tot[NM - 1][t] : scale[t] * tot[0][t];
          out[t][row] = v;
        }
      }
    };
    int row0 = tile0 + wave * RPS;
    if constexpr (KS == 1) {
      // software pipeline: the next item's bytes are in flight while this one is reduced
      Raw cur[NM][KS], nxt[NM][KS];
      if (row0 < tile_end) load_item(row0, cur);
      for (; row0 < tile_end; row0 += kWavesPerWg * RPS) {
        const int nrow = row0 + kWavesPerWg * RPS;
        if (nrow < tile_end) load_item(nrow, nxt);
        finish_item(row0, cur);
#pragma unroll
        for (int m = 0; m < NM; ++m) cur[m][0] = nxt[m][0];
      }
    } else {
      for (; row0 < tile_end; row0 += kWavesPerWg * RPS) {
        Raw cur[NM][KS];
        load_item(row0, cur);
        finish_item(row0, cur);
      }
    }
  } else {
    // long rows: K / 2048 steps (last one masked), activations re-read each step
    const int steps = (K + kStepElems - 1) / kStepElems;
    for (int row0 = tile0 + wave; row0 < tile_end; row0 += kWavesPerWg) {
      float tot[NM][TC];
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int t = 0; t < TC; ++t) tot[m][t] = 0.0f;
      for (int k = 0; k < steps; ++k) {
        const int koff = lane_koff<QUANT, 1>(g, k);
        const bool act = koff < K;
        float x[TC][32];
        float xs[TC][4];
#pragma unroll
        for (int t = 0; t < TC; ++t)
          load_x<QUANT>(xrow[t], koff, act, g, x[t], xs[t]);
        const size_t off = (size_t)row0 * row_bytes + (size_t)k * F::kChunkBytes;
        Raw r0;
        load_raw<QUANT>(w0 + off, act, g, r0);
        accum<QUANT, TC>(r0, g, x, xs, tot[0]);
        if constexpr (NM == 2) {
          Raw r1;
          load_raw<QUANT>(w1 + off, act, g, r1);
          accum<QUANT, TC>(r1, g, x, xs, tot[NM - 1]);
        }
      }
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int t = 0; t < TC; ++t) tot[m][t] = group_sum<64>(tot[m][t]);
      if (g.lane == 0) {
#pragma unroll
        for (int t = 0; t < TC; ++t) {
          const float v = NM == 2 ? silu_f(tot[0][t]) * tot[NM - 1][t] : scale[t] * tot[0][t];
          out[t][row0] = v;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------
// Kernels.  grid.x tiles the output rows, grid.y enumerates work units; every grid is
// a function of the geometry, the live token count is read from `valid_tokens`.
// ---------------------------------------------------------------------------------
struct ExpertArgs {
  const uint8_t* w0;       // gate (NM = 2) or the one matrix
  const uint8_t* w1;       // up (NM = 2)
  const float* x;          // activations: [token][K]
  float* out;              // [token][n_rows]
  const int* valid_tokens; // device scalar
  int K;                   // contraction length
  int n_rows;
  int tile_rows;           // rows per workgroup
};

// Shared expert / dense MLP: every live token, no indirection, no routing weight
// (crates/xabe-cuda/src/kernels/moe.rs:3425-3725, :4082-4227).  One work unit per chunk of two tokens.
template <int QUANT, int KS, int RPS, int NM>
__device__ __forceinline__ void shared_body(const ExpertArgs& a, int chunk, int tile) {
  const int t0 = chunk * 2;
  const int valid = *a.valid_tokens;
  if (t0 >= valid) return;
  if (t0 + 1 < valid) {
    const float* const xr[2] = {a.x + (size_t)t0 * a.K, a.x + (size_t)(t0 + 1) * a.K};
    float* const o[2] = {a.out + (size_t)t0 * a.n_rows, a.out + (size_t)(t0 + 1) * a.n_rows};
    const float sc[2] = {1.0f, 1.0f};
    matvec_rows<QUANT, KS, RPS, 2, NM>(a.w0, a.w1, a.K, a.n_rows, tile * a.tile_rows, a.tile_rows, xr, o, sc);
  } else {
    const float* const xr[1] = {a.x + (size_t)t0 * a.K};
    float* const o[1] = {a.out + (size_t)t0 * a.n_rows};
    const float sc[1] = {1.0f};
    matvec_rows<QUANT, KS, RPS, 1, NM>(a.w0, a.w1, a.K, a.n_rows, tile * a.tile_rows, a.tile_rows, xr, o, sc);
  }
}

// The lane's 32 activations of one step from a row in global memory or LDS, raw (no arithmetic, so a
// caller can request them and other data together and do the arithmetic when they arrive).
template <int QUANT>
__device__ __forceinline__ void lane_x_load(const float* row, int koff, const LaneGeom& g, float (&v)[32]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int off = QUANT == kQ6K ? koff + g.half * 128 + j * 32 + g.l8 * 8 : koff + j * 8;
    const float4 a = reinterpret_cast<const float4*>(row + off)[0];
    const float4 b = reinterpret_cast<const float4*>(row + off)[1];
    v[j * 8 + 0] = a.x; v[j * 8 + 1] = a.y; v[j * 8 + 2] = a.z; v[j * 8 + 3] = a.w;
    v[j * 8 + 4] = b.x; v[j * 8 + 5] = b.y; v[j * 8 + 6] = b.z; v[j * 8 + 7] = b.w;
  }
}

// xs[j] = -32 * (sum of the j-th eight), the Q6_K code offset folded out of the inner loop (as load_x).
template <int QUANT>
__device__ __forceinline__ void lane_x_offsets(const float (&x)[32], float (&xs)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) s += x[j * 8 + i];
    xs[j] = QUANT == kQ6K ? -32.0f * s : 0.0f;
  }
}

// Everything above this point in program order has been issued before anything below it is: keeps the
// compiler from sinking a batch of loads down to their first uses, which would serialise them.
__device__ __forceinline__ void issue_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

template <int QUANT, int KS, int RPS, int NM>
__global__ void __launch_bounds__(256) k_expert_shared(ExpertArgs a) {
  shared_body<QUANT, KS, RPS, NM>(a, blockIdx.y, blockIdx.x);
}

}  // namespace xabe
