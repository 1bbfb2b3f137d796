// The MoE block below the matrix-core widths (max_tokens < 64) as three launches with no intermediate passes.
//
// At a few tokens the block moves ~20 MB per token and every dependent memory access costs 1-2 us, so what
// decides the time is the number of dependent round trips and launch boundaries on the critical path; at a few
// dozen it is vector instructions per weight and token, and bytes.  The eight steps of the block (norm, router, bias,
// route, gate/up, down, shared expert, combine) are regrouped so that each launch issues everything it needs in one or
// two rounds of loads:
//
//   A  k_decode_logits:  router logits (+ bias) and the shared expert's gate/up, both normalising the
//                        residual rows on load; a workgroup per superblock of a token writes the normalised row with
//                        its digits (digits.h), one more per token the sigmoid gate scalar.
//   B  k_decode_up:      one (token, k) pair x share of its row tiles per workgroup.  One wavefront routes the token
//                        from its logits (every workgroup of a token repeats this: a few microseconds of one
//                        wavefront is cheaper than one more launch or a device-wide handshake), then the wavefronts
//                        stream the selected expert's gate/up rows through the digit contraction and write the
//                        intermediate row as digits.
//      (From eight tokens on the routing is a launch of its own between A and B, and the shared gate/up runs beside it
//      instead of in A: k_decode_router, k_decode_route.)
//   C  k_decode_down:    one token x share of its row tiles per workgroup, a wavefront per selection: the routed down
//                        projections (and, at few tokens, the shared one), summed in k order, gated, combined with
//                        the residual.  No partial buffer, no reduction pass.
//
// The routed contractions are pair_dot's (digits.h), as are k_digit_pairs', and sb_dot's in k_digit_rows bit for bit; routing, norm, router
// and shared expert are the per-row device functions of the multi-launch path.  So the outputs are bit-identical to that
// path: the batch-invariance contract.  One multiply-add and one conversion per weight on the vector ALU, which the digit form
// replaced, made B 95 and C 52 us at 32 tokens; six digits instead of four (71 and 39 then) hold the bits beside outliers.
// From 28 tokens B goes by expert, two pairs to a unit (k_decode_up_shared), which leaves C alone in going pair by pair.  At 32
// tokens router and routing take 7 and 8 us, B 69, C 33: B fetches the distinct experts 1.09 times, C 1.15 times (at 45 tokens 1.15
// and 1.43), vector instructions are 49 and 62 % of the cycles (45: 52 and 66).
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "decode_kernels.h"
#include "device_once.h"
#include "digit_rows.h"
#include "host_common.h"
#include "route_device.h"

namespace xabe {

constexpr size_t kDecodeBlockMaxTokens = kMfmaMinTokens - 1;  // every width below the matrix-core regime
// From this width on the routing is a launch of its own between the first two (one wavefront per token) and the second
// launch reads the selections: inside the second launch every workgroup of a token repeats the token's routing, and
// past a few tokens its grid runs in several rounds per CU, each paying for it again.  Measured before the routed
// contractions took their present form, us per block, routing inside / routing launch: 4 tokens 38.6 / 40.5, 6: 49.8 / 51.2, 8: 61.5 / 61.1, 12: 83.3 / 79.4, 16: 101.7 / 94.9,
// 32: 181.3 / 161.5.  With the shared gate/up beside the routing launch, 4: 47.8 / 54.3, 6: 64.1 / 67.0, 7: 71.0 / 71.6,
// 8: 79.4 / 79.3 (one layer by itself, cold).
constexpr int kPreRouteMinTokens = 8;
// From this width on the second and third launches deal their workgroups so that the ones that read the same row
// tile (of whichever experts their pairs or tokens selected) run next to each other on one XCD: workgroup ids go
// round-robin to the eight XCDs, each with its own L2, and at these widths several pairs select the same expert
// (32 tokens: 256 pairs over ~163 experts), whose rows then come out of HBM once per XCD instead of once per pair.
// At 16 tokens and below, where fewer pairs coincide, the plain order measured 0.1-0.5 us faster and is kept.
constexpr int kXcdGroupMinTokens = 24;
// From this width on the second launch of Q6_K gate/up goes by expert, two pairs at a time (k_decode_up_shared): enough pairs
// coincide to pay for making the units.  us per block of four in one graph, by pair / by expert: uniform routing 20 tokens
// 365 / 381, 26: 445 / 445, 32: 507 / 497, 40: 601 / 574, 50: 715 / 659, 63: 860 / 753; skewed 20: 285 / 288, 26: 346 / 339,
// 32: 397 / 377, 63: 687 / 632.  (Q8_0's codes are the matrix operand as they lie: there is no unpacking to share.)
constexpr int kPairUnitsMinTokens = 28;
// the seam's arrival counters: per token one counter and one per group of kSeamGroup workgroups, 128 bytes apart
constexpr int kSeamGroup = 16, kSeamMaxGroups = 64, kSeamCountersPerToken = 1 + kSeamMaxGroups, kSeamCounterStride = 32;
constexpr int kMaxShare = 4;      // consecutive tiles a workgroup of the second or third launch takes at most
constexpr int kMaxTopK = 8;       // contributions held in registers by k_decode_down
// Steps per wavefront of the first launch: a wavefront reads 24 KB of activation rows and norm weights for the 2-4 KB
// of weights of one step, so more steps against the same registers cut what the launch pulls out of L2, at the
// price of fewer workgroups.  Measured per width (launch A, us, depth 1 / 2 / 4): one token 5.2 / 5.3 / 6.6, three
// 7.7 / 6.5 / 8.4, eight 14.2 / 9.4 / 8.4 (which k_decode_router takes now).
static int logits_depth(int max_tokens) { return max_tokens <= 1 ? 1 : max_tokens <= 6 ? 2 : 4; }


struct DecodeArgs {
  const float* residual;
  const float* post_norm;
  const uint8_t* router;
  const uint8_t *gate, *up, *down;
  const uint8_t *sgate, *sup, *sdown;
  const float* shared_gate_inp;
  const float* logit_bias;
  const int* valid_tokens;
  float* normed;
  float* logits;
  int* topk_ids;
  float* topk_weights;
  uint8_t *x_d, *inter_d;  // digits of the normalised rows and of the routed intermediate rows (digits.h)
  float *x_e, *inter_e;    // their scales: of whole superblocks, of groups of 16
  float* inter;            // the routed intermediate rows themselves
  float* shared_inter;
  float* shexp;
  float* gate_out;
  float* routed;
  float* ffn_out;
  float* l_out;
  // the seam to the next layer (all null / zero when the pass ends at l_out): the last workgroup of the third launch to
  // finish a token's row applies the next layer's RMSNorm to it (arrival counters: one int per token, zero between passes)
  const float* next_w;
  float* next_normed;
  _Float16* next_normed_h;
  int* arrivals;
  float next_eps;
  size_t expert_bytes;  // bytes of one expert's gate (= up) matrix
  size_t down_bytes;    // bytes of one expert's down matrix (its format may differ)
  size_t up_len;        // bytes of a whole gate (= up) stack
  float eps;
  int H, I, E, top_k, max_tokens;
  int tiles_r, tiles_s, tiles_g, tiles_d;  // row tiles: router, shared gate/up (launch A), gate/up (B), down (C)
  int shared_units;                        // of the shared down projection in B (k_decode_up_shared)
  int shared_from;                         // first workgroup of the shared down projection in B (wider batches)
  int share_g, share_d;                    // consecutive tiles of a workgroup (B, C): divide tiles_g and tiles_d
};

// Row tiles of the first launch: D steps (RPS rows of K = 2048 / RPS elements each) per wavefront of a matrix, or of
// a gate/up pair, against the TC tokens of the workgroup's chunk, whose rows are normalised on the way in.
//   NM = 2: out[t][row] = silu(gate . x_t) * (up . x_t);   NM = 1: out[t][row] = (w . x_t) (+ bias[row]).
// The workgroup's four wavefronts need the same TC rows and the norm weight.  They are fetched once per workgroup, as
// consecutive 16-byte pieces, and handed to the wavefronts through LDS; each wavefront then derives the RMS scales in
// the canonical order and normalises its own elements, (x * inv) * w: the stand-alone RMSNorm kernel's values.
// (Each wavefront fetching its own copy from global memory cost 1.9 us of the launch at three tokens: a lane's 32
// elements are one cache line, so every one of its eight loads touched 64 lines, and all workgroups of the launch aim
// at the same few rows.)
// LDS rows are padded by four floats per 32, so that lanes reading 16-byte pieces 128 bytes apart take different banks.
constexpr int kXnPad = kStepElems + kStepElems / 8;  // floats per staged row
__device__ __forceinline__ int xn_at(int e) { return e + 4 * (e >> 5); }

// PRE: the rows handed over are normalised already (the previous block's tail wrote them into this block's `normed`):
// they are staged and used as they are, no norm weight, no scale.
template <int QUANT, int RPS, int TC, int NM, int D, bool PRE>
__device__ __forceinline__ void tile_normed(const uint8_t* __restrict__ w0, const uint8_t* __restrict__ w1, int K,
                                            int n_rows, int row0, const float* const (&xrow)[TC],
                                            const float* __restrict__ norm_w, float eps, float* const (&out)[TC],
                                            const float* __restrict__ bias, const int* __restrict__ valid_tokens,
                                            int token0, float* s_xn) {
  using F = Fmt<QUANT>;
  using Raw = typename F::Raw;
  constexpr int G = 64 / RPS;
  const LaneGeom g = lane_geom<QUANT>();
  const int koff = lane_koff<QUANT, RPS>(g, 0);
  const size_t row_bytes = (size_t)(K / F::kBlockElems) * F::kBlockBytes;
  // the rows' weights first: D steps against the same activation registers, all requested here
  // (a step past the matrix re-reads its last one and is never stored)
  Raw r[D][NM];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const int rd = min(row0 + d * RPS, n_rows - RPS);
    load_raw<QUANT, true>(w0 + (size_t)rd * row_bytes, true, g, r[d][0]);
    if constexpr (NM == 2) load_raw<QUANT, true>(w1 + (size_t)rd * row_bytes, true, g, r[d][NM - 1]);
  }
  // the chunk's rows and the norm weight, 16 bytes per thread and piece (K <= 2048: two pieces per thread), as they are
  const int n4 = K / 4;
  float* s_nw = s_xn + TC * kXnPad;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int i = (int)threadIdx.x + 256 * j, ic = min(i, n4 - 1);
    float4 nq = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (!PRE) nq = reinterpret_cast<const float4*>(norm_w)[ic];
    float4 xq[TC];
#pragma unroll
    for (int t = 0; t < TC; ++t) xq[t] = reinterpret_cast<const float4*>(xrow[t])[ic];
    if (i < n4) {
      if constexpr (!PRE) *reinterpret_cast<float4*>(s_nw + xn_at(4 * i)) = nq;
#pragma unroll
      for (int t = 0; t < TC; ++t) *reinterpret_cast<float4*>(s_xn + t * kXnPad + xn_at(4 * i)) = xq[t];
    }
  }
  __syncthreads();
  if (row0 >= n_rows) return;
  // from here on every wavefront works for itself, out of LDS: the RMS scale of each token in the canonical order
  // (lane L folds elements 32L .. 32L+31, then the wavefront tree), its own 32 elements normalised as (x * inv) * w
  auto lds8 = [&](const float* row, int e, float (&v)[32], int at) __attribute__((always_inline)) {
    const float4* p = reinterpret_cast<const float4*>(row + xn_at(e));
    const float4 lo = p[0], hi = p[1];
    v[at + 0] = lo.x; v[at + 1] = lo.y; v[at + 2] = lo.z; v[at + 3] = lo.w;
    v[at + 4] = hi.x; v[at + 5] = hi.y; v[at + 6] = hi.z; v[at + 7] = hi.w;
  };
  float x[TC][32], xs[TC][4], nw[32];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int off = QUANT == kQ6K ? koff + g.half * 128 + j * 32 + g.l8 * 8 : koff + j * 8;
    if constexpr (!PRE) lds8(s_nw, off, nw, j * 8);
#pragma unroll
    for (int t = 0; t < TC; ++t) lds8(s_xn + t * kXnPad, off, x[t], j * 8);
  }
#pragma unroll
  for (int t = 0; t < TC; ++t) {
    if constexpr (PRE) {
      lane_x_offsets<QUANT>(x[t], xs[t]);
      continue;
    }
    float f[32];
    const int base = g.lane * 32;  // (lanes past the row's end fold zeros: fma(0, 0, s) == s)
#pragma unroll
    for (int j = 0; j < 4; ++j) lds8(s_xn + t * kXnPad, min(base, K - 32) + j * 8, f, j * 8);
    float sq = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) sq = __builtin_fmaf(f[i], f[i], sq);
    if (base >= K) sq = 0.0f;
    const float inv = rms_finish(sq, K, eps);
#pragma unroll
    for (int i = 0; i < 32; ++i) x[t][i] = x[t][i] * inv * nw[i];
    lane_x_offsets<QUANT>(x[t], xs[t]);
  }
  // rows past the live-token count were computed from whatever the buffer held (in bounds, sized for max_tokens)
  // and are dropped
  const int valid = *valid_tokens;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    float tot[NM][TC];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
#pragma unroll
      for (int t = 0; t < TC; ++t) tot[m][t] = 0.0f;
      accum<QUANT, TC>(r[d][m], g, x, xs, tot[m]);
#pragma unroll
      for (int t = 0; t < TC; ++t) tot[m][t] = group_sum<G>(tot[m][t]);
    }
    const int row = row0 + d * RPS + g.lane / G;
    if ((g.lane % G) == 0 && row < n_rows) {
#pragma unroll
      for (int t = 0; t < TC; ++t) {
        float v = NM == 2 ? silu_f(tot[0][t]) * tot[NM - 1][t] : 1.0f * tot[0][t];
        if (NM == 1 && bias) v += bias[row];
        if (token0 + t < valid) out[t][row] = v;
      }
    }
  }
}

// group_sum of four values at once, value t in the lanes t and t + 8 of every sixteen: the lanes of a quad add up one value
// each from the second addition on.  The additions pair the same partial sums in the same order as group_sum's, so the
// sums are the same bits.
template <int G>
__device__ __forceinline__ float group_sum_of_four(const float (&v)[4]) {
  static_assert(G == 16 || G == 64, "group width");
  const int lane = __lane_id();
  const bool b0 = lane & 1, b1 = lane & 2;
  const float p = (b0 ? v[1] : v[0]) + dpp_f<0xB1>(b0 ? v[0] : v[1]);  // quad_perm [1,0,3,2]
  const float q = (b0 ? v[3] : v[2]) + dpp_f<0xB1>(b0 ? v[2] : v[3]);
  float s = (b1 ? q : p) + dpp_f<0x4E>(b1 ? p : q);                    // quad_perm [2,3,0,1]
  s += dpp_f<0x12C>(s);  // row_ror:12: the next quad's
  s += dpp_f<0x128>(s);  // row_ror:8: the other eight lanes'
  if constexpr (G == 64) {
    const uint32_t a = __builtin_bit_cast(uint32_t, s);
    const auto r = __builtin_amdgcn_permlane16_swap(a, a, false, false);  // {rows 0 0 2 2, rows 1 1 3 3}
    const uint32_t r0 = r[0], r1 = r[1];
    s = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
    const uint32_t c = __builtin_bit_cast(uint32_t, s);
    const auto h = __builtin_amdgcn_permlane32_swap(c, c, false, false);
    const uint32_t h0 = h[0], h1 = h[1];
    s = __builtin_bit_cast(float, h0) + __builtin_bit_cast(float, h1);
  }
  return s;
}

// The same rows for wider batches: four tokens per pass over the rows' weights (tile_normed: two), a token's row normalised
// once per workgroup instead of once per wavefront, four tokens' sums across the lanes taken together, and one SwiGLU for
// the four.  What bounds it is the chain (a round trip for the rows, a barrier each for staging and norm) and about 300
// vector instructions per wavefront; more steps per wavefront save fetched rows and cost workgroups in flight.  Measured,
// us at 13 / 32 / 45 tokens, steps 1 / 2 / 4 of a wavefront: router 7.0 8.6 11.0 / 6.9 7.6 9.7 / 9.9 8.9 11.2, shared
// gate/up (with the routing beside it, 6.1 alone) 6.1 8.4 10.4 / 6.1 10.2 11.2 / 10.6 11.6 15.1.  With router, shared
// gate/up and norm in one launch of two-token chunks and the routing behind it: 20.5 / 22.8 / 26.2 for what now takes
// 13.0 / 16.0 / 20.1.
constexpr int kGroupTokens = 4;  // (a wavefront of the workgroup each)
template <int QUANT, int RPS, int NM, int D, bool PRE>
__device__ __forceinline__ void tile_group(const uint8_t* __restrict__ w0, const uint8_t* __restrict__ w1, int K, int n_rows,
                                           int row0, const float* __restrict__ rows, int token0, int max_tokens,
                                           const float* __restrict__ norm_w, float eps, float* __restrict__ out,
                                           const float* __restrict__ bias, const int* __restrict__ valid_tokens, float* s_xn) {
  using F = Fmt<QUANT>;
  using Raw = typename F::Raw;
  constexpr int G = 64 / RPS, TC = kGroupTokens;
  const LaneGeom g = lane_geom<QUANT>();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int koff = lane_koff<QUANT, RPS>(g, 0);
  const size_t row_bytes = (size_t)(K / F::kBlockElems) * F::kBlockBytes;
  // (a token past the batch re-reads its last one, a step past the matrix its last one: neither is stored)
  Raw r[D][NM];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const int rd = min(row0 + d * RPS, n_rows - RPS);
    load_raw<QUANT, true>(w0 + (size_t)rd * row_bytes, true, g, r[d][0]);
    if constexpr (NM == 2) load_raw<QUANT, true>(w1 + (size_t)rd * row_bytes, true, g, r[d][NM - 1]);
  }
  const int n4 = K / 4;
  {
    float4 xq[2][TC];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < TC; ++t)
        xq[j][t] = reinterpret_cast<const float4*>(rows + (size_t)min(token0 + t, max_tokens - 1) * K)[min((int)threadIdx.x + 256 * j, n4 - 1)];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = (int)threadIdx.x + 256 * j;
      if (i < n4) {
#pragma unroll
        for (int t = 0; t < TC; ++t) *reinterpret_cast<float4*>(s_xn + t * kXnPad + xn_at(4 * i)) = xq[j][t];
      }
    }
  }
  const int valid = *valid_tokens;
  __syncthreads();
  if constexpr (!PRE) {
    // wavefront t: token t's RMS scale in the canonical order (lane L folds elements 32 L .. 32 L + 31, then the wavefront
    // tree), and the lane's elements put back as (x * inv) * w
    float* row = s_xn + wave * kXnPad + xn_at(min(g.lane * 32, K - 32));  // (lanes past the row's end fold zeros)
    float4 f[8], nw[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) nw[j] = reinterpret_cast<const float4*>(norm_w + min(g.lane * 32, K - 32))[j];
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = reinterpret_cast<const float4*>(row)[j];
    float sq = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      sq = __builtin_fmaf(f[j].x, f[j].x, sq);
      sq = __builtin_fmaf(f[j].y, f[j].y, sq);
      sq = __builtin_fmaf(f[j].z, f[j].z, sq);
      sq = __builtin_fmaf(f[j].w, f[j].w, sq);
    }
    if (g.lane * 32 >= K) sq = 0.0f;
    const float inv = rms_finish(sq, K, eps);
    if (g.lane * 32 < K) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        reinterpret_cast<float4*>(row)[j] = make_float4(f[j].x * inv * nw[j].x, f[j].y * inv * nw[j].y, f[j].z * inv * nw[j].z, f[j].w * inv * nw[j].w);
    }
    __syncthreads();
  }
  if (row0 >= n_rows) return;
  float x[TC][32], xs[TC][4];
#pragma unroll
  for (int t = 0; t < TC; ++t) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int off = QUANT == kQ6K ? koff + g.half * 128 + j * 32 + g.l8 * 8 : koff + j * 8;
      const float4* p = reinterpret_cast<const float4*>(s_xn + t * kXnPad + xn_at(off));
      const float4 lo = p[0], hi = p[1];
      x[t][j * 8 + 0] = lo.x; x[t][j * 8 + 1] = lo.y; x[t][j * 8 + 2] = lo.z; x[t][j * 8 + 3] = lo.w;
      x[t][j * 8 + 4] = hi.x; x[t][j * 8 + 5] = hi.y; x[t][j * 8 + 6] = hi.z; x[t][j * 8 + 7] = hi.w;
    }
    lane_x_offsets<QUANT>(x[t], xs[t]);
  }
  const int t = token0 + (g.lane & 3);
  const bool stores = (g.lane % G) < TC && t < valid;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    float sum[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      float tot[TC] = {0.0f, 0.0f, 0.0f, 0.0f};
      accum<QUANT, TC>(r[d][m], g, x, xs, tot);
      sum[m] = group_sum_of_four<G>(tot);
    }
    const int row = row0 + d * RPS + g.lane / G;
    float v = NM == 2 ? silu_f(sum[0]) * sum[NM - 1] : 1.0f * sum[0];
    if (stores && row < n_rows) {
      if (NM == 1 && bias) v += bias[row];
      out[(size_t)t * n_rows + row] = v;
    }
  }
}

// What the first workgroups of A do: a superblock of a token's normalised row with its digits each, then a token's gate each.
template <bool PRE>
__device__ __forceinline__ void token_rows(const DecodeArgs& a, float* s_red, uint32_t* s_mag) {
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int nsb = a.H / kSbElems;  // (the served widths are multiples of 256)
  const int valid = *a.valid_tokens;
  if ((int)blockIdx.x < a.max_tokens * nsb) {
    // a superblock of the normalised row (callers read it back) and its digits, an element per thread: the order of
    // operations of the stand-alone RMSNorm kernel
    const int t = (int)blockIdx.x / nsb, sb = (int)blockIdx.x % nsb, j = sb * kSbElems + (int)threadIdx.x;
    const float* xr = (PRE ? a.normed : a.residual) + (size_t)t * a.H;
    float v = xr[j];  // (PRE: the row is there already, written by the previous block's tail)
    if constexpr (!PRE) {
      const float nw = a.post_norm[j], inv = row_inv_rms(xr, a.H, a.eps);
      v = v * inv * nw;
    }
    if (t >= valid) return;
    if constexpr (!PRE) a.normed[(size_t)t * a.H + j] = v;
    uint32_t mag = (uint32_t)wave_max_i((int)(__builtin_bit_cast(uint32_t, v) & 0x7fffffffu));
    if ((threadIdx.x & 63) == 0) s_mag[wave] = mag;
    __syncthreads();
    mag = max(max(s_mag[0], s_mag[1]), max(s_mag[2], s_mag[3]));
    const int e = digit_exponent(mag);
    const bool inexact = store_digit_lane(v, digit_shift(e), j, a.x_d + (size_t)t * nsb * kSbDigitBytes, true);
    const float scale = digit_scale(mag, e, __syncthreads_or(inexact));
    if (threadIdx.x == 0) a.x_e[(size_t)t * nsb + sb] = scale;
    return;
  }
  // g = sigmoid(shared_gate_inp . normed): the order of operations of the stand-alone gate kernel
  const int t = (int)blockIdx.x - a.max_tokens * nsb;
  const float* xr = (PRE ? a.normed : a.residual) + (size_t)t * a.H;
  // hidden <= 2048: eight columns per thread, every load issued before the first use
  float xv[8], nv[8], gv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int j = threadIdx.x + 256 * i;
    const bool in = j < a.H;
    xv[i] = in ? xr[j] : 0.0f;
    nv[i] = in && !PRE ? a.post_norm[j] : 0.0f;
    gv[i] = in ? a.shared_gate_inp[j] : 0.0f;
  }
  float inv = 1.0f;
  if constexpr (!PRE) inv = row_inv_rms(xr, a.H, a.eps);
  if (t >= valid) return;
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (256 * i < a.H) s = __builtin_fmaf(gv[i], PRE ? xv[i] : xv[i] * inv * nv[i], s);
  s = group_sum<64>(s);
  if ((threadIdx.x & 63) == 0) s_red[wave] = s;
  __syncthreads();
  const float total = ((s_red[0] + s_red[1]) + s_red[2]) + s_red[3];
  if (threadIdx.x == 0) a.gate_out[t] = 1.0f / (1.0f + expf(-total));
}

// ------------------------------------------------------------------------------------------------
// A: grid = max_tokens * superblocks (norm and digits) + max_tokens (gate scalar) + chunks * tiles_r (router) + chunks * tiles_s (shared gate/up).
// A chunk is two tokens sharing one pass over the weights.
// ------------------------------------------------------------------------------------------------
template <int SQ, int RF, int RPS, int kLogitsDepth, bool PRE = false>
__global__ void __launch_bounds__(256) k_decode_logits(DecodeArgs a) {
  __shared__ float s_red[4];
  __shared__ uint32_t s_mag[4];  // the row writers': a wavefront's largest magnitude
  __shared__ __attribute__((aligned(16))) float s_xn[3 * kXnPad];  // the chunk's rows and the norm weight
  const int chunks = (a.max_tokens + 1) / 2;
  const int n_r = chunks * a.tiles_r;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int first_item = a.max_tokens * (a.H / kSbElems + 1);
  if ((int)blockIdx.x >= first_item) {
    int item = (int)blockIdx.x - first_item;
    const bool router = item < n_r;
    if (!router) item -= n_r;
    const int tiles = router ? a.tiles_r : a.tiles_s;
    const int c = item / tiles, tile = item % tiles, t0 = 2 * c;
    const int row0 = (tile * kWavesPerWg + wave) * RPS * kLogitsDepth;
    const float* x0 = (PRE ? a.normed : a.residual) + (size_t)t0 * a.H;
    if (t0 + 1 < a.max_tokens) {
      const float* const xr[2] = {x0, x0 + a.H};
      if (router) {
        float* const o[2] = {a.logits + (size_t)t0 * a.E, a.logits + (size_t)(t0 + 1) * a.E};
        tile_normed<RF, RPS, 2, 1, kLogitsDepth, PRE>(a.router, nullptr, a.H, a.E, row0, xr, a.post_norm, a.eps, o, a.logit_bias, a.valid_tokens, t0, s_xn);
      } else {
        float* const o[2] = {a.shared_inter + (size_t)t0 * a.I, a.shared_inter + (size_t)(t0 + 1) * a.I};
        tile_normed<SQ, RPS, 2, 2, kLogitsDepth, PRE>(a.sgate, a.sup, a.H, a.I, row0, xr, a.post_norm, a.eps, o, nullptr, a.valid_tokens, t0, s_xn);
      }
    } else {
      const float* const xr[1] = {x0};
      if (router) {
        float* const o[1] = {a.logits + (size_t)t0 * a.E};
        tile_normed<RF, RPS, 1, 1, kLogitsDepth, PRE>(a.router, nullptr, a.H, a.E, row0, xr, a.post_norm, a.eps, o, a.logit_bias, a.valid_tokens, t0, s_xn);
      } else {
        float* const o[1] = {a.shared_inter + (size_t)t0 * a.I};
        tile_normed<SQ, RPS, 1, 2, kLogitsDepth, PRE>(a.sgate, a.sup, a.H, a.I, row0, xr, a.post_norm, a.eps, o, nullptr, a.valid_tokens, t0, s_xn);
      }
    }
    return;
  }
  token_rows<PRE>(a, s_red, s_mag);
}

// ------------------------------------------------------------------------------------------------
// B: grid = max_tokens * top_k * shares of the row tiles (in wide batches padded to whole rounds of the XCDs, and the
// shared expert's down projection behind them).
// ------------------------------------------------------------------------------------------------
// From kPreRouteMinTokens tokens on: A with the router's rows alone ...
constexpr int kRouterSteps = 2, kSharedSteps = 1;  // steps per wavefront (tile_group's D)
template <int RF, int RPS, bool PRE>
__global__ void __launch_bounds__(256, 2) k_decode_router(DecodeArgs a) {
  __shared__ float s_red[4];
  __shared__ uint32_t s_mag[4];
  __shared__ __attribute__((aligned(16))) float s_xn[kGroupTokens * kXnPad];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int item = (int)blockIdx.x - a.max_tokens * (a.H / kSbElems + 1);
  if (item < 0) {
    token_rows<PRE>(a, s_red, s_mag);
    return;
  }
  const int group = item / a.tiles_r, tile = item % a.tiles_r;
  tile_group<RF, RPS, 1, kRouterSteps, PRE>(a.router, nullptr, a.H, a.E, (tile * kWavesPerWg + wave) * RPS * kRouterSteps,
                                            PRE ? a.normed : a.residual, group * kGroupTokens, a.max_tokens, a.post_norm, a.eps,
                                            a.logits, a.logit_bias, a.valid_tokens, s_xn);
}
// ... and, once the logits and the normalised rows are there, the routing (one wavefront per token, one token per workgroup
// so that they spread over the chip: route_one_token, the stand-alone routing kernel's body) beside the shared expert's
// gate/up, which does not wait for it.
template <int SQ, int RPS>
__global__ void __launch_bounds__(256, 2) k_decode_route(DecodeArgs a) {
  __shared__ __attribute__((aligned(16))) float s_xn[kGroupTokens * kXnPad];
  static_assert(kGroupTokens * kXnPad >= (int)kRouteMaxExperts, "a token's logits fit");
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int item = (int)blockIdx.x - a.max_tokens;
  if (item >= 0) {
    const int group = item / a.tiles_s, tile = item % a.tiles_s;
    tile_group<SQ, RPS, 2, kSharedSteps, true>(a.sgate, a.sup, a.H, a.I, (tile * kWavesPerWg + wave) * RPS * kSharedSteps, a.normed,
                                               group * kGroupTokens, a.max_tokens, nullptr, a.eps, a.shared_inter, nullptr,
                                               a.valid_tokens, s_xn);
    return;
  }
  const int t = blockIdx.x;
  if (wave != 0 || t >= *a.valid_tokens) return;
  int sel_i;
  float sel_w;
  route_one_token(a.logits + (size_t)t * a.E, a.E, a.top_k, s_xn, sel_i, sel_w);
  if ((int)threadIdx.x < a.top_k) {
    a.topk_ids[(size_t)t * a.top_k + threadIdx.x] = sel_i;
    a.topk_weights[(size_t)t * a.top_k + threadIdx.x] = sel_w;
  }
}

// Shared expert's down projection, a wavefront's unit: (chunk of two tokens, four steps of RPS rows).
template <int SQ, int RPS>
__device__ __forceinline__ void shared_down_rows(const DecodeArgs& a, int unit) {
  using RawS = typename Fmt<SQ>::Raw;
  constexpr int G = 64 / RPS;
  const int lane = fresh_lane();
  const int units_per_chunk = a.H / (4 * RPS);
  const int t0 = 2 * (unit / units_per_chunk), row0 = (unit % units_per_chunk) * 4 * RPS;
  const int t1 = min(t0 + 1, a.max_tokens - 1);
  const int valid = *a.valid_tokens;
  const LaneGeom g = lane_geom<SQ>(lane);
  const int koff = lane_koff<SQ, RPS>(g, 0);
  const size_t row_bytes = (size_t)(a.I / Fmt<SQ>::kBlockElems) * Fmt<SQ>::kBlockBytes;
  float x[2][32], xs[2][4];
  lane_x_load<SQ>(a.shared_inter + (size_t)t0 * a.I, koff, g, x[0]);
  lane_x_load<SQ>(a.shared_inter + (size_t)t1 * a.I, koff, g, x[1]);
  lane_x_offsets<SQ>(x[0], xs[0]);
  lane_x_offsets<SQ>(x[1], xs[1]);
  // steps in flight: more do not fit the registers of two workgroups per CU (Q6_K with two spilled ten to fifteen: four
  // blocks of 13 / 32 / 45 / 63 tokens 283 / 523 / 642 / 766 us, with one 267 / 470 / 591 / 713)
  constexpr int kFlight = SQ == kQ6K ? 1 : 2;
#pragma unroll 1
  for (int d0 = 0; d0 < 4; d0 += kFlight) {
    RawS raw[kFlight];
#pragma unroll
    for (int d = 0; d < kFlight; ++d) load_raw<SQ, true>(a.sdown + (size_t)(row0 + (d0 + d) * RPS) * row_bytes, true, g, raw[d]);
#pragma unroll
    for (int d = 0; d < kFlight; ++d) {
      float tot[2] = {0.0f, 0.0f};
      accum<SQ, 2>(raw[d], g, x, xs, tot);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const float sh = 1.0f * group_sum<G>(tot[t]);
        if ((lane % G) == 0 && t0 + t < valid) a.shexp[(size_t)(t0 + t) * a.H + row0 + (d0 + d) * RPS + lane / G] = sh;
      }
    }
  }
}

// ROUTED: the token's selection was made by a routing launch between A and this one (wider batches: there a token's
// routing would otherwise be repeated by every one of its workgroups, several rounds of them per CU); the pair's
// expert then comes out of topk_ids through the scalar cache and nothing else of the routing runs here.
// A tile is sixteen gate rows and the sixteen matching up rows; wavefront w takes pair w >> 1 of the rows' superblocks
// (NP pairs: hidden / 512) of matrix w & 1.  A workgroup runs `share_g` consecutive tiles of its pair against one copy of
// the activation digits in registers: a wavefront's slot is free once the tile's bytes are in registers, so the next
// tile's rows are on their way while this one is multiplied.  The tiles' sums wait in LDS for one barrier at the end, so
// that no wavefront of the loop waits for another (with a barrier and one wavefront's SwiGLU per tile a tile took 9 us).
// ROUTED: the workgroups past the pairs' are the shared expert's down projection (its intermediate is launch A's), 8 NP
// steps of RPSI rows each, two tokens per pass, on the lanes' fp32 sums of the separate kernels.  (At fewer tokens a
// wavefront of the third launch does it: here, on a few CUs only, its uncoalesced loads were the launch's last to end,
// 13.5 against 9.3 us for one token.)
// DIRECT (one tile per workgroup, one workgroup per CU): the rows go straight into registers; there is no next tile whose
// bytes the slot would receive meanwhile, and the way through LDS is a trip that everything after it waits for.
template <int RQ, int SQ, int NP, int RPSI, bool ROUTED, bool DIRECT>
__global__ void __launch_bounds__(128 * NP, DIRECT ? 2 : 4) k_decode_up(DecodeArgs a) {
  using Dma = PairDma<RQ>;
  constexpr int kWaves = 2 * NP;
  extern __shared__ __attribute__((aligned(16))) uint8_t s_up[];  // a weight slot per wavefront, then the routing's num_experts floats
  __shared__ int s_expert, s_final;      // the candidate expert of this pair; the one routing settles on
  __shared__ float s_red[kMaxShare][2 * NP][64];  // [tile][superblock][half, matrix, row]
  float* const s_route = reinterpret_cast<float*>(s_up + kWaves * PairDma<RQ>::kSlotBytes);
  if constexpr (ROUTED) {
    if ((int)blockIdx.x >= a.shared_from) {
      shared_down_rows<SQ, RPSI>(a, __builtin_amdgcn_readfirstlane(2 * NP * ((int)blockIdx.x - a.shared_from) + (int)(threadIdx.x >> 6)));
      return;
    }
  }
  const int block = (int)blockIdx.x;
  const int shares = a.tiles_g / a.share_g;
  int p = block / shares, share = block % shares;
  if (ROUTED && a.max_tokens >= kXcdGroupMinTokens) {
    // wide batches (see kXcdGroupMinTokens): all pairs of one share next to each other on one XCD (the grid is padded
    // to whole rounds of eight shares)
    const int n_pairs = a.max_tokens * a.top_k, xcd = block & 7, j = block >> 3;
    share = xcd + 8 * (j / n_pairs);
    p = j % n_pairs;
    if (share >= shares) return;
  }
  const int t = p / a.top_k, k = p % a.top_k;
  [[maybe_unused]] int pre_e = 0;
  if constexpr (ROUTED) pre_e = a.topk_ids[p];
  // everything read before the live-token count is known is sized for max_tokens rows
  const int valid = *a.valid_tokens;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = (int)__lane_id(), quarter = lane >> 4;
  const int mat = wave & 1, sb0 = 2 * (wave >> 1), sb = sb0 + (quarter >> 1);
  // one wavefront routes the token (a different one in neighbouring workgroups, which share a CU); its
  // logits and every wavefront's activation digits are requested together
  const bool routes = !ROUTED && wave == (int)((block >> 8) % kWaves);
  const bool few = a.E <= 256;
  float lg[kRouteMaxPerLane];
  if (routes) {
    if (few) route_load<4>(a.logits + (size_t)t * a.E, a.E, nullptr, nullptr, *reinterpret_cast<float(*)[4]>(lg));
    else route_load<kRouteMaxPerLane>(a.logits + (size_t)t * a.E, a.E, nullptr, nullptr, lg);
  }
  const uint32_t row_bytes = (uint32_t)(2 * NP * SbRaw<RQ>::kBytes);
  const size_t x_sb = (size_t)t * (2 * NP) + sb;
  PairDigits<kWhole> x;
  x.load(a.x_d + x_sb * kSbDigitBytes, a.x_e + x_sb);
  Dma dma;  // (its lane offsets are ready before the expert is known)
  if constexpr (!DIRECT) dma.init(row_bytes, sb0);
  if (t >= valid) return;
  // Routing in two halves (route_device.h).  The first orders the experts by logit: its k-th candidate is
  // the pair's expert unless probabilities tie, and it is known ~2 us before the softmax is, so the
  // wavefronts request the candidate's rows right away.  The routing wavefront then finishes the softmax
  // under its own loads' latency; in the rare pass where the probabilities reorder the candidates, the rows
  // are streamed again for the expert the reference's rule selects.
  // The pair's candidate is known after k + 1 selection rounds; the remaining rounds (the rest of the token's
  // selection and the k + 1-th candidate the verification needs) run after the rows have been requested.
  const int n_cand = min(a.top_k + 1, a.E);
  int cand_i = 0;
  int key[kRouteMaxPerLane];
  if (routes) {
    if (few) {
      route_keys<4>(*reinterpret_cast<float(*)[4]>(lg), a.E, *reinterpret_cast<int(*)[4]>(key));
      route_rounds<4>(*reinterpret_cast<int(*)[4]>(key), 0, k + 1, cand_i);
    } else {
      route_keys<kRouteMaxPerLane>(lg, a.E, key);
      route_rounds<kRouteMaxPerLane>(key, 0, k + 1, cand_i);
    }
    if (lane == k) s_expert = cand_i;
  }
  if constexpr (!ROUTED) __syncthreads();
  uint8_t* const slot = s_up + wave * PairDma<RQ>::kSlotBytes;
  const uint32_t slot_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)slot);
  // the pair's rows of expert e: the request, (the routing wavefront: the rest of the routing,) the contraction
  auto stream_rows = [&](int e, auto finish_c) __attribute__((always_inline)) {
    const size_t e_off = (size_t)e * a.expert_bytes;
    auto run_off = [&](int i) __attribute__((always_inline)) { return e_off + (size_t)(16 * (share * a.share_g + i)) * row_bytes; };
    SbRaw<RQ> raw;
    if constexpr (DIRECT)
      sb_read((mat ? a.up : a.gate) + run_off(0) + (size_t)(lane & 15) * row_bytes + sb * SbRaw<RQ>::kBytes, quarter & 1, raw);
    else
      dma.request(mat ? a.up : a.gate, a.up_len, run_off(0), slot_lds);
    if constexpr (decltype(finish_c)::value) {
      if (routes) {  // (raised priority keeps it ahead of its neighbours' arithmetic)
        __builtin_amdgcn_s_setprio(3);
        int sel_i;
        float sel_w;
        bool exact;
        if (few) route_rounds<4>(*reinterpret_cast<int(*)[4]>(key), k + 1, n_cand, cand_i);
        else route_rounds<kRouteMaxPerLane>(key, k + 1, n_cand, cand_i);
        if (few) route_finish<4>(*reinterpret_cast<float(*)[4]>(lg), a.E, a.top_k, n_cand, cand_i, s_route, sel_i, sel_w, exact);
        else route_finish<kRouteMaxPerLane>(lg, a.E, a.top_k, n_cand, cand_i, s_route, sel_i, sel_w, exact);
        if (lane == k) s_final = sel_i;
        if (k == 0 && share == 0 && lane < a.top_k) {
          a.topk_ids[(size_t)t * a.top_k + lane] = sel_i;
          a.topk_weights[(size_t)t * a.top_k + lane] = sel_w;
        }
        __builtin_amdgcn_s_setprio(0);
      }
    }
#pragma unroll 1
    for (int i = 0; i < (DIRECT ? 1 : a.share_g); ++i) {
      if constexpr (!DIRECT) {
        wait_loads();
        if (RQ == kQ6K && sb0 + 2 == 2 * NP && run_off(i) + (size_t)16 * row_bytes == a.up_len) Dma::patch_tail(mat ? a.up : a.gate, a.up_len, slot);
        sb_read_slot(Dma::row_at(slot, row_bytes, lane & 15, sb0) + (quarter >> 1) * SbRaw<RQ>::kBytes, quarter & 1, raw);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (i + 1 < a.share_g) dma.request(mat ? a.up : a.gate, a.up_len, run_off(i + 1), slot_lds);
      }
      s_red[i][sb][(quarter & 1) * 32 + mat * 16 + (lane & 15)] = pair_dot<RQ>(
          raw, x, [&](int q) __attribute__((always_inline)) { return a.normed + (size_t)t * a.H + (sb0 + (q >> 1)) * kSbElems; });
    }
    __syncthreads();  // (s_final is there, too)
  };
  if constexpr (ROUTED) {
    stream_rows(__builtin_amdgcn_readfirstlane(min(max(pre_e, 0), a.E - 1)), std::false_type{});
  } else {
    const int e = __builtin_amdgcn_readfirstlane(s_expert);
    stream_rows(e, std::true_type{});
    const int e_final = __builtin_amdgcn_readfirstlane(s_final);
    if (e_final != e) stream_rows(e_final, std::false_type{});  // (the sums, written again)
  }
  for (int i = wave; i < a.share_g; i += kWaves) {
    // superblocks in order, then half 0 + half 1; lanes 0..15 hold the gate sums, 16..31 the up sums
    const float (&red)[2 * NP][64] = s_red[i];
    float h0 = red[0][lane & 31], h1 = red[0][32 + (lane & 31)];
#pragma unroll
    for (int c = 1; c < 2 * NP; ++c) {
      h0 += red[c][lane & 31];
      h1 += red[c][32 + (lane & 31)];
    }
    const float total = h0 + h1, up = __shfl_xor(total, 16);
    const int nsb_i = a.I / kSbElems;
    const float v = silu_f(total) * up;
    const int row = 16 * (share * a.share_g + i) + (lane & 15);
    if (lane < 16) a.inter[(size_t)p * a.I + row] = v;
    store_digit_group(v, row, a.inter_d + (size_t)p * nsb_i * kSbDigitBytes, a.inter_e + (size_t)p * nsb_i * 16, lane < 16);
  }
}

// B for kPairUnitsMinTokens tokens and more, routed gate/up in Q6_K: by expert.  A unit is two (token, k) pairs that selected
// one expert, or the one left over; their tiles (k_decode_up's, a wavefront's part the same) unpack a weight once for both
// tokens and fetch it once.  Every workgroup makes the list of units out of topk_ids by itself, alike in all of them (counts by
// ballots, a scan over the experts): it is resident throughout, two workgroups to a CU, and takes whole units in rounds,
// then an even share of the tiles of the last, partial round.  An XCD has an eighth of the row tiles, and the units of one
// expert follow each other, so what more pairs of an expert read again comes out of the L2.  The tokens' digits lie in LDS
// (24.6 KB: with 16 weight slots of 6.9 KB per CU that leaves room for two workgroups; in registers they would not leave any).
// Bound by memory: at 45 tokens (360 pairs, 193 experts) 86 us, 382 MB fetched of 332 MB that are distinct; pair by pair
// 96 us and 590 MB.  Vector instructions 52 % of the cycles.  Measured and not kept: a workgroup per unit, found by a search
// of its own (88 us; 63 tokens 4 % behind); three pairs with the third's digits in registers (113: spills); the shared
// expert's rows under the first request instead of at the end (72 against 70 at 32 tokens).
constexpr int kPairChunks = ((int)kDecodeBlockMaxTokens * kMaxTopK + 63) / 64;
constexpr int kMaxUnits = 16;  // of a workgroup
template <int SQ, int NP, int RPSI>
__global__ void __launch_bounds__(128 * NP, 4) k_decode_up_shared(DecodeArgs a) {
  using Dma = PairDma<kQ6K, 27, true>;
  constexpr int kWaves = 2 * NP, kThreads = 64 * kWaves, kDigits = 2 * NP * kSbDigitBytes;  // bytes of a token's row
  extern __shared__ __attribute__((aligned(16))) uint8_t s_up[];  // two tokens' digits, zeros, a weight slot per wavefront
  __shared__ int s_first[kMaxUnits], s_second[kMaxUnits];
  uint8_t* const s_zeros = s_up + 2 * kDigits;
  uint8_t* const s_slots = s_zeros + kZeroBytes;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = (int)__lane_id(), quarter = lane >> 4;
  const int valid = *a.valid_tokens, n_live = min(valid, a.max_tokens) * a.top_k;

  // ---- the units: the live pairs by expert, two by two; the same in every workgroup
  constexpr int kE = (int)kRouteMaxExperts, kPerLane = kE / 64;
  int* const s_cnt = reinterpret_cast<int*>(s_slots);  // [chunk of 64 pairs][expert]
  int* const s_pos = s_cnt + kPairChunks * kE;         // [wavefront][expert]: twice the first unit, and the pairs before a chunk's
  constexpr int kOwn = (kPairChunks + kWaves - 1) / kWaves;  // chunks of a wavefront
  int id[kOwn], before[kOwn];
#pragma unroll
  for (int j = 0; j < kOwn; ++j) {
    const int q = 64 * (wave + kWaves * j) + lane;
    id[j] = a.topk_ids[min(q, a.max_tokens * a.top_k - 1)];
    id[j] = q < n_live ? min(max(id[j], 0), a.E - 1) : -1;
  }
  typedef int v4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int j = 0; j < kOwn; ++j)
#pragma unroll
    for (int i = 0; i < kPerLane / 4; ++i) reinterpret_cast<v4*>(s_cnt + (wave + kWaves * j) * kE)[64 * i + lane] = v4{0, 0, 0, 0};
  for (int i = (int)threadIdx.x; i < kZeroBytes / 4; i += kThreads) reinterpret_cast<uint32_t*>(s_zeros)[i] = 0;
  if (threadIdx.x < kMaxUnits) s_second[threadIdx.x] = -1;
  // (a wavefront's own LDS operations keep their order)
#pragma unroll
  for (int j = 0; j < kOwn; ++j) {
    const uint64_t same = lanes_alike(id[j], id[j] >= 0);
    before[j] = __builtin_popcountll(same & ((1ull << lane) - 1));
    if (id[j] >= 0 && before[j] == 0) s_cnt[(wave + kWaves * j) * kE + id[j]] = __builtin_popcountll(same);
  }
  __syncthreads();
  // every wavefront scans all experts, eight to a lane
  int n_units;
#pragma unroll
  for (int j = 0; j < kOwn; ++j) {
    int count[kPerLane], ahead[kPerLane];
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) count[i] = ahead[i] = 0;
#pragma unroll
    for (int c = 0; c < kPairChunks; ++c)
#pragma unroll
      for (int q = 0; q < kPerLane / 4; ++q) {
        const v4 n = reinterpret_cast<const v4*>(s_cnt + c * kE + kPerLane * lane)[q];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (c < wave + kWaves * j) ahead[4 * q + i] += n[i];
          count[4 * q + i] += n[i];
        }
      }
    int units = 0;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) units += (count[i] + 1) / 2;
    int scan = units;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(scan, d);
      if (lane >= d) scan += up;
    }
    n_units = __builtin_amdgcn_readlane(scan, 63);
    int first = scan - units;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      s_pos[wave * kE + kPerLane * lane + i] = 2 * first + ahead[i];
      first += (count[i] + 1) / 2;
    }
    if (id[j] >= 0) before[j] += s_pos[wave * kE + id[j]];  // twice the pair's unit, and which of the two it is
  }
  // ---- this workgroup's share: an eighth of the row tiles per XCD, the units' tiles dealt evenly and in order
  const int tiles = a.tiles_g / 8, xcd = (int)blockIdx.x & 7, per_xcd = (int)gridDim.x >> 3, rank = (int)blockIdx.x >> 3;
  // whole units in rounds (neighbours take units of one expert at the same time: its rows come into the L2 once), the tiles
  // of the last, partial round dealt evenly
  const int rounds = n_units / per_xcd, rest = (n_units - rounds * per_xcd) * tiles;
  const int rest_lo = rest * rank / per_xcd, rest_hi = rest * (rank + 1) / per_xcd;
  const int rest_unit = rounds * per_xcd + rest_lo / tiles, hi = rounds * tiles + rest_hi - rest_lo;  // (tiles of this workgroup)
  const uint32_t inverse = ((1u << 20) + per_xcd - 1) / per_xcd;  // (u < 512)
#pragma unroll
  for (int j = 0; j < kOwn; ++j) {
    if (id[j] >= 0) {
      const int u = before[j] >> 1, round = (int)((uint32_t)u * inverse >> 20);
      const int at = round < rounds ? (u - round * per_xcd == rank ? round : -1) : u >= rest_unit ? rounds + u - rest_unit : -1;
      const int p = 64 * (wave + kWaves * j) + lane;
      if (at >= 0 && at < kMaxUnits) {
        if (before[j] & 1) s_second[at] = p;
        else s_first[at] = p | id[j] << 9;
      }
    }
  }
  __syncthreads();
  // the shared expert's down projection (see k_decode_up): its units dealt over the launch's wavefronts, workgroups first
  auto shared_down = [&]() __attribute__((always_inline)) {
    for (int unit = (int)blockIdx.x + wave * (int)gridDim.x; unit < a.shared_units; unit += kWaves * (int)gridDim.x) shared_down_rows<SQ, RPSI>(a, unit);
  };
  if (hi > 0) {
    const int mat = wave & 1, sb0 = 2 * (wave >> 1), sb = sb0 + (quarter >> 1);
    const uint32_t row_bytes = (uint32_t)(2 * NP * SbRaw<kQ6K>::kBytes);
    Dma dma;
    dma.init(row_bytes, sb0);
    uint8_t* const slot = s_slots + wave * Dma::kSlotBytes;
    const uint32_t slot_lds = lds_address(slot);
    const uint8_t* const w = mat ? a.up : a.gate;
    // the at-th tile of this workgroup: its unit, and its place among the unit's
    auto tile_of = [&](int at) __attribute__((always_inline)) { return at < rounds * tiles ? at % tiles : (rest_lo + at - rounds * tiles) % tiles; };
    auto unit_of = [&](int at) __attribute__((always_inline)) {
      const int i = at < rounds * tiles ? at / tiles : rounds + (rest_lo + at - rounds * tiles) / tiles - rest_lo / tiles;
      const int f = __builtin_amdgcn_readfirstlane(s_first[i]), g = __builtin_amdgcn_readfirstlane(s_second[i]);
      return f | (g < 0 ? f & 511 : g) << 18;  // pair, expert, the other pair (or the same)
    };
    auto run_off = [&](int unit, int at) __attribute__((always_inline)) {
      return (size_t)(unit >> 9 & 511) * a.expert_bytes + (size_t)(16 * (xcd * tiles + tile_of(at))) * row_bytes;
    };
    const int at_high = pair_high_at(lane), at_low = pair_low_at(lane);
    const uint8_t *high[2], *low[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint8_t* d = s_up + t * kDigits + sb * kSbDigitBytes;
      high[t] = at_high >= 0 ? d + at_high : s_zeros;
      low[t] = at_low >= 0 ? d + at_low : s_zeros;
    }
    int unit = unit_of(0);
    dma.request(w, a.up_len, run_off(unit, 0), slot_lds);
#pragma unroll 1
    for (int at = 0; at < hi;) {
      const int pairs[2] = {unit & 511, unit >> 18}, tok[2] = {pairs[0] / a.top_k, pairs[1] / a.top_k};
      const bool two = pairs[0] != pairs[1];
      const int end = min(hi, at + tiles - tile_of(at)), n = end - at;
      // the tokens' digits: 3 NP pieces of 1 KB each, three per wavefront
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int piece = wave + kWaves * i, t = piece >= 3 * NP, c = piece - 3 * NP * t;
        lds_dma_16(a.x_d + (size_t)(t ? tok[1] : tok[0]) * kDigits, (uint32_t)(1024 * c + 16 * lane), lds_address(s_up + t * kDigits + 1024 * c));
      }
      float xe[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) xe[t] = a.x_e[(size_t)tok[t] * (2 * NP) + sb];
      wait_loads();
      __syncthreads();
      float sums[2][kMaxShare];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < kMaxShare; ++i) sums[t][i] = 0.0f;
      int next = unit;
      auto run_tiles = [&](auto nt_c) __attribute__((always_inline)) {
        constexpr int NT = decltype(nt_c)::value;
        const uint8_t* hi_at[NT];
        const uint8_t* lo_at[NT];
        float es[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) hi_at[t] = high[t], lo_at[t] = low[t], es[t] = xe[t];
#pragma unroll 1
        for (int i = 0; i < n; ++i) {
          wait_loads();
          if (sb0 + 2 == 2 * NP && run_off(unit, at + i) + (size_t)16 * row_bytes == a.up_len) Dma::patch_tail(w, a.up_len, slot);
          SbRaw<kQ6K> raw;
          sb_read_slot(Dma::row_at(slot, row_bytes, lane & 15, sb0) + (quarter >> 1) * SbRaw<kQ6K>::kBytes, quarter & 1, raw);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          if (at + i + 1 < hi) {
            if (i + 1 == n) next = unit_of(at + i + 1);
            dma.request(w, a.up_len, run_off(next, at + i + 1), slot_lds);
          }
          auto x_of = [&](int t, int q) __attribute__((always_inline)) { return a.normed + (size_t)tok[t] * a.H + (sb0 + (q >> 1)) * kSbElems; };
          float out[NT];
          pair_dot_lds<NT>(raw, hi_at, lo_at, es, x_of, out);
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int j = 0; j < kMaxShare; ++j)
              if (j == i) sums[t][j] = out[t];
        }
      };
      if (two) run_tiles(std::integral_constant<int, 2>{});
      else run_tiles(std::integral_constant<int, 1>{});
      __syncthreads();  // (everyone has read the digits for the last time: the sums go there)
      float (*const s_red)[2][2 * NP][64] = reinterpret_cast<float (*)[2][2 * NP][64]>(s_up);  // [tile][token][superblock][half, matrix, row]
      static_assert(kMaxShare * 2 * 2 * NP * 64 * sizeof(float) <= 2 * kDigits, "the sums fit");
#pragma unroll
      for (int i = 0; i < kMaxShare; ++i)
        if (i < n) {
#pragma unroll
          for (int t = 0; t < 2; ++t)
            if (t == 0 || two) s_red[i][t][sb][(quarter & 1) * 32 + mat * 16 + (lane & 15)] = sums[t][i];
        }
      __syncthreads();
      for (int u = wave; u < (two ? 2 : 1) * n; u += kWaves) {
        const int t = u >= n, i = u - t * n;
        const float (&red)[2 * NP][64] = s_red[i][t];
        float h0 = red[0][lane & 31], h1 = red[0][32 + (lane & 31)];
#pragma unroll
        for (int c = 1; c < 2 * NP; ++c) {
          h0 += red[c][lane & 31];
          h1 += red[c][32 + (lane & 31)];
        }
        const float sum = h0 + h1, up = __shfl_xor(sum, 16);
        const int nsb_i = a.I / kSbElems, pr = t ? pairs[1] : pairs[0];
        const float v = silu_f(sum) * up;
        const int row = 16 * (xcd * tiles + tile_of(at) + i) + (lane & 15);
        if (lane < 16) a.inter[(size_t)pr * a.I + row] = v;
        store_digit_group(v, row, a.inter_d + (size_t)pr * nsb_i * kSbDigitBytes, a.inter_e + (size_t)pr * nsb_i * 16, lane < 16);
      }
      __syncthreads();  // (the sums are read: the next digits go there)
      at = end;
      unit = next;
    }
  }
  shared_down();
}
template <int NP>
constexpr size_t up_shared_lds() {
  return (size_t)2 * 2 * NP * kSbDigitBytes + kZeroBytes +
         std::max((size_t)2 * NP * PairDma<kQ6K, 27, true>::kSlotBytes, (size_t)(kPairChunks + 2 * NP) * kRouteMaxExperts * sizeof(int));
}

// ------------------------------------------------------------------------------------------------
// C: grid = max_tokens * shares of the row tiles.  A tile is sixteen output rows of 512 elements (or 32 of 256: pairs of
// superblocks either way) of one token; a wavefront takes one selection for the `share_d` consecutive tiles of its
// workgroup against one copy of the token's intermediate digits in registers, the next tile's rows on their way while
// this one is multiplied.  The weighted row sums meet in LDS once, at the end, and are added in selection order.
// ------------------------------------------------------------------------------------------------
// SHARED (the widths whose second launch leaves it out): one more wavefront takes the shared expert's rows (four, with a
// step of each tile apiece, were slower: 7.0 against 6.8 us for one token).
template <int RQ, int SQ, int kPairRows, bool SHARED>  // kPairRows: rows a pair of superblocks covers
__global__ void __launch_bounds__(64 * (kMaxTopK + SHARED), SHARED ? 3 : 4) k_decode_down(DecodeArgs a) {
  using Dma = PairRunDma<RQ>;
  constexpr int kRows = 16 * kPairRows;  // rows per tile
  extern __shared__ __attribute__((aligned(16))) uint8_t s_down[];  // a weight slot per selection
  __shared__ float s_part[kMaxShare][kMaxTopK + SHARED][kRows];  // [tile][selection]: the weighted row sums
  const int shares = a.tiles_d / a.share_d;
  int t = blockIdx.x / shares, share = blockIdx.x % shares;
  if (a.max_tokens >= kXcdGroupMinTokens) {
    // wide batches (see kXcdGroupMinTokens): all tokens of one share next to each other on one XCD (the grid is padded
    // to whole rounds of eight shares)
    const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
    share = xcd + 8 * (j / a.max_tokens);
    t = j % a.max_tokens;
    if (share >= shares) return;
  }
  // every buffer read below is sized for max_tokens rows, so round one is issued before the live-token
  // count is known; rows past it hold an earlier pass's values or zeros, and nothing is stored for them
  const int valid = *a.valid_tokens;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = (int)__lane_id(), quarter = lane >> 4;
  const int tile0 = share * a.share_d;  // hidden is a multiple of kRows * share_d
  // what the thread's output row needs besides the sums: requested with round one where the launch is a single round of
  // workgroups, at the end where others are at work meanwhile (held all along they spill; 13 tokens 504 -> 499 us)
  float gate = SHARED ? a.gate_out[t] : 0.0f;
  const int n_out = a.share_d * kRows, n0 = min((int)threadIdx.x, n_out - 1);
  const size_t o0 = (size_t)t * a.H + (size_t)tile0 * kRows;  // (a share's rows are consecutive)
  float sh = 0.0f, res = SHARED ? a.residual[o0 + n0] : 0.0f;
  if (SHARED && wave >= a.top_k) {
    constexpr int RPS = kRows / 4, G = 64 / RPS;
    const LaneGeom gs = lane_geom<SQ>();
    const int koff = lane_koff<SQ, RPS>(gs, 0);
    const size_t rb_s = (size_t)(a.I / Fmt<SQ>::kBlockElems) * Fmt<SQ>::kBlockBytes;
    float x[1][32], xs[1][4];
    lane_x_load<SQ>(a.shared_inter + (size_t)t * a.I, koff, gs, x[0]);
    typename Fmt<SQ>::Raw raw[4];
    auto request = [&](int i) __attribute__((always_inline)) {
#pragma unroll
      for (int d = 0; d < 4; ++d) load_raw<SQ, true>(a.sdown + (size_t)((tile0 + i) * kRows + d * RPS) * rb_s, true, gs, raw[d]);
    };
    request(0);
    if (t >= valid) return;
    lane_x_offsets<SQ>(x[0], xs[0]);
#pragma unroll 1
    for (int i = 0; i < a.share_d; ++i) {
      float tot[4][1];
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        tot[d][0] = 0.0f;
        accum<SQ, 1>(raw[d], gs, x, xs, tot[d]);
      }
      if (i + 1 < a.share_d) request(i + 1);
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const float v = 1.0f * group_sum<G>(tot[d][0]);
        if ((lane % G) == 0) s_part[i][kMaxTopK][d * RPS + lane / G] = v;
      }
    }
  } else {
    const int p = t * a.top_k + wave;
    const int id = a.topk_ids[p];
    const float sel_w = a.topk_weights[p];
    constexpr int nsb = kPairRows == 1 ? 2 : 1;
    const size_t x_sb = (size_t)p * nsb + (kPairRows == 1 ? quarter >> 1 : 0);
    PairDigits<kGroups> x;  // (requested with the expert's index, not after it)
    x.load(a.inter_d + x_sb * kSbDigitBytes, a.inter_e + x_sb * 16);
    const int e = __builtin_amdgcn_readfirstlane(min(max(id, 0), a.E - 1));
    const uint32_t pair_bytes = 2 * SbRaw<RQ>::kBytes;
    uint8_t* const slot = s_down + wave * Dma::kSlotBytes;
    const uint32_t slot_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)slot);
    auto run = [&](int i) __attribute__((always_inline)) { return a.down + (size_t)e * a.down_bytes + (size_t)(tile0 + i) * 16 * pair_bytes; };
    if (t >= valid) return;
    Dma dma;
    dma.init();
    dma.request(run(0), slot_lds);
#pragma unroll 1
    for (int i = 0; i < a.share_d; ++i) {
      wait_loads();
      SbRaw<RQ> raw;
      sb_read_words(slot + (lane & 15) * Dma::kRowStride + (quarter >> 1) * SbRaw<RQ>::kBytes, quarter & 1, raw);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (i + 1 < a.share_d) dma.request(run(i + 1), slot_lds);
      float v = pair_dot<RQ>(
          raw, x, [&](int q) __attribute__((always_inline)) { return a.inter + ((size_t)p * nsb + (kPairRows == 1 ? q >> 1 : 0)) * kSbElems; });
      // superblock 0 + superblock 1 of each half, then half 0 + half 1
      if constexpr (kPairRows == 1) v += __shfl_xor(v, 32);
      v += __shfl_xor(v, 16);
      if constexpr (kPairRows == 1) {
        if (lane < 16) s_part[i][wave][lane] = sel_w * v;
      } else {
        if ((quarter & 1) == 0) s_part[i][wave][2 * (lane & 15) + (quarter >> 1)] = sel_w * v;
      }
    }
  }
  __syncthreads();
  if constexpr (!SHARED) gate = a.gate_out[t];
  // rows kRows * i + r of the share: the routed sum in selection order, shared expert, gate, residual
  for (int n = (int)threadIdx.x; n < n_out; n += (int)blockDim.x) {
    const int i = n / kRows, row = n % kRows;
    const size_t o = o0 + n;
    if (!SHARED || n >= (int)blockDim.x) res = a.residual[o];
    if constexpr (SHARED) sh = s_part[i][kMaxTopK + SHARED - 1][row], a.shexp[o] = sh;
    else sh = a.shexp[o];
    float r = 0.0f;
#pragma unroll
    for (int j = 0; j < kMaxTopK; ++j)
      if (j < a.top_k) r += s_part[i][j][row];
    const float v = r + sh * gate;
    a.routed[o] = r;
    if (a.ffn_out) a.ffn_out[o] = v;
    const float lo = v + res;
    // (with the seam on, another workgroup of this launch reads the row back: the store goes through to memory)
    if (a.next_normed) __hip_atomic_store(a.l_out + o, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else a.l_out[o] = lo;
  }
  if (!a.next_normed) return;
  if (a.share_d * kRows > 64) {  // (several wavefronts have stored: all of them acknowledged before one counts the workgroup in)
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  if (wave != 0) return;
  // The seam (docs/BENCHMARKS.md:1376 of the reference: the next layer's RMSNorm in the combine's tail).  A token's
  // row is finished by several workgroups, and the wavefront that finishes it last applies the norm.  Arrivals are
  // counted in two levels so that no counter sees more than a few dozen of them (atomics on one address are served
  // one after the other, ~70 ns each: 256 arrivals on one counter cost 18 us per pass at 32 tokens): 16 workgroups on
  // a group counter, the groups on the token's counter, every counter on a 128-byte line of its own.  A wavefront
  // counts itself once its own stores are acknowledged (they go through to memory: no fence, whose L2 write-back costs
  // microseconds here), so whoever sees a count complete knows all stores below it have landed.
  __builtin_amdgcn_s_waitcnt(0);
  int prev = 0;
  int* const token_ctr = a.arrivals + (size_t)t * kSeamCountersPerToken * kSeamCounterStride;
  const int groups = (shares + kSeamGroup - 1) / kSeamGroup, grp = share / kSeamGroup;
  const int in_group = min(kSeamGroup, shares - grp * kSeamGroup);
  int* const group_ctr = token_ctr + (1 + grp) * kSeamCounterStride;
  if (lane == 0) prev = __hip_atomic_fetch_add(group_ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (__builtin_amdgcn_readfirstlane(prev) != in_group - 1) return;
  if (lane == 0) {
    __hip_atomic_store(group_ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // (zero again for the next pass)
    prev = __hip_atomic_fetch_add(token_ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (__builtin_amdgcn_readfirstlane(prev) != groups - 1) return;
  if (lane == 0) __hip_atomic_store(token_ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // the row comes in coalesced (element 64 j + lane per load) and changes hands through LDS (the weight slots are free
  // now), padded by four floats per 32 as the first launch pads its rows
  float* s_l = reinterpret_cast<float*>(s_down);  // (kXnPad floats; one wavefront per workgroup gets here)
  const float* lrow = a.l_out + (size_t)t * a.H;
  float in[32];
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    const int e = 64 * j + lane;
    in[j] = e < a.H ? __hip_atomic_load(lrow + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0f;
  }
#pragma unroll
  for (int j = 0; j < 32; ++j) s_l[xn_at(64 * j + lane)] = in[j];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  RmsRaw rowq;
#pragma unroll
  for (int j = 0; j < 8; ++j) rowq.q[j] = *reinterpret_cast<const float4*>(s_l + xn_at(32 * lane + 4 * j));
  const float inv = rms_finish(rms_fold(rowq, 0.0f), a.H, a.next_eps);
  // out the same way: element 64 j + lane, (x * inv) * w
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    const int e = 64 * j + lane;
    if (e < a.H) {
      const float v = in[j] * inv * a.next_w[e];
      a.next_normed[(size_t)t * a.H + e] = v;
      if (a.next_normed_h) a.next_normed_h[(size_t)t * a.H + e] = (_Float16)v;
    }
  }
}

// ------------------------------------------------------------------ host side
// Tiles per workgroup of the second launch: the largest power of two up to kMaxShare that divides the tiles and
// leaves 192 workgroups.  Same box, us per block, tiles of (second, third) launch: one token (1, 1) 24.1, (2, 1) 24.3,
// (1, 2) 25.6; three (1, 1) 37.4, (2, 2) 31.8, (4, 2) 31.4, (4, 4) 34.5; thirteen (1, 1) 91.1, (2, 2) 80.9, (4, 4) 79.9;
// thirty-two (1, 1) 172, (2, 2) 146, (4, 4) 132.
static int decode_share(size_t units, int tiles) {
  int share = 1;
  while (share < kMaxShare && tiles % (2 * share) == 0 && units * tiles >= (size_t)384 * share) share *= 2;
  return share;
}

// Tiles per workgroup of the third launch: the number whose workgroups, dealt in rounds to the CUs, end first, a workgroup's
// time being that of its tiles and half a tile more; the larger of two alike.  Blocks (of four in one graph, us), two / four
// tiles: four tokens 132 / 144, five 181 / 171, seven 202 / 192, eight 212 / 210, nine 233 / 242, twelve 264 / 267, fourteen
// 291 / 286, thirty-two 509 / 498; one / two: two tokens 102 / 108, three 128 / 119.  Past three rounds of the largest the
// workgroups no longer end together and it is the best (twenty-seven tokens 458 / 448).
static int down_share(const xabe_moe_kernels* k, size_t tokens, int tiles) {
  if (tiles % kMaxShare == 0 && tokens * (size_t)(tiles / kMaxShare) > 3 * (size_t)k->num_cus) return kMaxShare;
  int best = 1;
  size_t best_cost = ~(size_t)0;
  for (int share = 1; share <= kMaxShare && tiles % share == 0; share *= 2) {
    const size_t rounds = (tokens * (size_t)(tiles / share) + k->num_cus - 1) / k->num_cus, cost = rounds * (2 * share + 1);
    if (cost <= best_cost) best_cost = cost, best = share;
  }
  return best;
}

struct Launch {
  const DecodeArgs& a;
  hipStream_t s;
  unsigned grid_a, grid_route, grid_b, grid_shared, grid_c;
  bool pre_routed;  // k_decode_router and k_decode_route instead of k_decode_logits and routing inside B
  bool pair_units;  // k_decode_up_shared instead of k_decode_up
  bool pre_normed;  // `normed` holds this pass's rows already (the previous block's tail): A neither normalises nor writes them
  unsigned launches;  // bit i: issue launch i (A, B, C); all three outside measurements
};

// Each launch is chosen by the formats it reads: A by the shared gate/up and router formats, B by the routed
// gate/up format, C by the routed and shared down formats (the shipped layers mix them: gate/up Q6_K with
// down Q8_0).
template <int NP>
static size_t up_lds(int gq, int num_experts) {
  return 2 * NP * (size_t)(gq == XABE_QUANT_Q6K ? PairDma<kQ6K>::kSlotBytes : PairDma<kQ8_0>::kSlotBytes) + num_experts * sizeof(float);
}
static size_t down_lds(int dq, int top_k) {  // (the seam's tail stages a row in it)
  return std::max((size_t)top_k * (dq == XABE_QUANT_Q6K ? PairRunDma<kQ6K>::kSlotBytes : PairRunDma<kQ8_0>::kSlotBytes), (size_t)kXnPad * sizeof(float));
}

template <int RPSH, int NP, int RPSI>
static bool launch_all(const Launch& l, int gq, int dq, int sgq, int sdq, int router_quant) {
  const bool g6 = gq == XABE_QUANT_Q6K, d6 = dq == XABE_QUANT_Q6K, sg6 = sgq == XABE_QUANT_Q6K, sd6 = sdq == XABE_QUANT_Q6K;
  const bool rf32 = router_quant < 0;
  if (!rf32 && router_quant != XABE_QUANT_Q8_0) return false;
  if (l.launches & 1u) {
#define XABE_A1(SQ, RF, PRE)                                                                                        \
  do {                                                                                                            \
    const int da = logits_depth(l.a.max_tokens);                                                                  \
    if (da == 1) hipLaunchKernelGGL((k_decode_logits<SQ, RF, RPSH, 1, PRE>), dim3(l.grid_a), dim3(256), 0, l.s, l.a);  \
    else if (da == 2) hipLaunchKernelGGL((k_decode_logits<SQ, RF, RPSH, 2, PRE>), dim3(l.grid_a), dim3(256), 0, l.s, l.a); \
    else hipLaunchKernelGGL((k_decode_logits<SQ, RF, RPSH, 4, PRE>), dim3(l.grid_a), dim3(256), 0, l.s, l.a);     \
  } while (0)
#define XABE_AR(RF)                                                                                                      \
  do {                                                                                                                   \
    if (l.pre_normed) hipLaunchKernelGGL((k_decode_router<RF, RPSH, true>), dim3(l.grid_a), dim3(256), 0, l.s, l.a);     \
    else hipLaunchKernelGGL((k_decode_router<RF, RPSH, false>), dim3(l.grid_a), dim3(256), 0, l.s, l.a);                 \
  } while (0)
#define XABE_A(SQ, RF)                  \
  do {                                  \
    if (l.pre_normed) XABE_A1(SQ, RF, true); \
    else XABE_A1(SQ, RF, false);        \
  } while (0)
    if (l.pre_routed && rf32) XABE_AR(kF32);
    else if (l.pre_routed) XABE_AR(kQ8_0);
    else if (sg6 && rf32) XABE_A(kQ6K, kF32);
    else if (sg6) XABE_A(kQ6K, kQ8_0);
    else if (rf32) XABE_A(kQ8_0, kF32);
    else XABE_A(kQ8_0, kQ8_0);
#undef XABE_A
#undef XABE_AR
#undef XABE_A1
  }
  if (l.launches & 2u) {
    const size_t lds = up_lds<NP>(gq, l.a.E);
    const dim3 grid(l.grid_b), block(128 * NP);
    if (l.pre_routed) {
      if (sg6) hipLaunchKernelGGL((k_decode_route<kQ6K, RPSH>), dim3(l.grid_route), dim3(256), 0, l.s, l.a);
      else hipLaunchKernelGGL((k_decode_route<kQ8_0, RPSH>), dim3(l.grid_route), dim3(256), 0, l.s, l.a);
    }
    if (l.pair_units) {
      if (sd6) hipLaunchKernelGGL((k_decode_up_shared<kQ6K, NP, RPSI>), dim3(l.grid_shared), block, up_shared_lds<NP>(), l.s, l.a);
      else hipLaunchKernelGGL((k_decode_up_shared<kQ8_0, NP, RPSI>), dim3(l.grid_shared), block, up_shared_lds<NP>(), l.s, l.a);
    } else
#define XABE_B(RQ, SQ)                                                                                            \
  do {                                                                                                            \
    if (l.pre_routed) hipLaunchKernelGGL((k_decode_up<RQ, SQ, NP, RPSI, true, false>), grid, block, lds, l.s, l.a); \
    else if (l.a.share_g == 1) hipLaunchKernelGGL((k_decode_up<RQ, SQ, NP, RPSI, false, true>), grid, block, lds, l.s, l.a); \
    else hipLaunchKernelGGL((k_decode_up<RQ, SQ, NP, RPSI, false, false>), grid, block, lds, l.s, l.a);            \
  } while (0)
    if (g6 && sd6) XABE_B(kQ6K, kQ6K);
    else if (g6) XABE_B(kQ6K, kQ8_0);
    else if (sd6) XABE_B(kQ8_0, kQ6K);
    else XABE_B(kQ8_0, kQ8_0);
#undef XABE_B
  }
  if (l.launches & 4u) {
    const size_t lds = down_lds(dq, l.a.top_k);
    const dim3 grid(l.grid_c), block(64 * (l.a.top_k + (l.pre_routed ? 0 : 1)));
    if (l.pre_routed) {
      if (d6) hipLaunchKernelGGL((k_decode_down<kQ6K, kQ8_0, RPSI / 4, false>), grid, block, lds, l.s, l.a);
      else hipLaunchKernelGGL((k_decode_down<kQ8_0, kQ8_0, RPSI / 4, false>), grid, block, lds, l.s, l.a);
    } else if (d6 && sd6) hipLaunchKernelGGL((k_decode_down<kQ6K, kQ6K, RPSI / 4, true>), grid, block, lds, l.s, l.a);
    else if (d6) hipLaunchKernelGGL((k_decode_down<kQ6K, kQ8_0, RPSI / 4, true>), grid, block, lds, l.s, l.a);
    else if (sd6) hipLaunchKernelGGL((k_decode_down<kQ8_0, kQ6K, RPSI / 4, true>), grid, block, lds, l.s, l.a);
    else hipLaunchKernelGGL((k_decode_down<kQ8_0, kQ8_0, RPSI / 4, true>), grid, block, lds, l.s, l.a);
  }
  return true;
}

// LDS limits of the launches that ask for more than the static 64 KB
static int decode_block_set_limits() {
#define XABE_LDS(kernel, bytes) \
  XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(&kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)(bytes)))
#define XABE_UP(Q, code, SQ, NP, RPSI)                                                              \
  XABE_LDS((k_decode_up<Q, SQ, NP, RPSI, false, false>), up_lds<NP>(code, (int)kRouteMaxExperts)); \
  XABE_LDS((k_decode_up<Q, SQ, NP, RPSI, false, true>), up_lds<NP>(code, (int)kRouteMaxExperts));  \
  XABE_LDS((k_decode_up<Q, SQ, NP, RPSI, true, false>), up_lds<NP>(code, (int)kRouteMaxExperts))
#define XABE_DOWN(Q, code)                                          \
  XABE_LDS((k_decode_down<Q, kQ8_0, 1, false>), down_lds(code, kMaxTopK));  \
  XABE_LDS((k_decode_down<Q, kQ8_0, 2, false>), down_lds(code, kMaxTopK));  \
  XABE_LDS((k_decode_down<Q, kQ6K, 1, true>), down_lds(code, kMaxTopK));    \
  XABE_LDS((k_decode_down<Q, kQ6K, 2, true>), down_lds(code, kMaxTopK));    \
  XABE_LDS((k_decode_down<Q, kQ8_0, 1, true>), down_lds(code, kMaxTopK));   \
  XABE_LDS((k_decode_down<Q, kQ8_0, 2, true>), down_lds(code, kMaxTopK));   \
  XABE_UP(Q, code, kQ6K, 4, 4);                                              \
  XABE_UP(Q, code, kQ8_0, 4, 4);                                             \
  XABE_UP(Q, code, kQ6K, 1, 8);                                              \
  XABE_UP(Q, code, kQ8_0, 1, 8)
  XABE_LDS((k_decode_up_shared<kQ6K, 4, 4>), up_shared_lds<4>());
  XABE_LDS((k_decode_up_shared<kQ8_0, 4, 4>), up_shared_lds<4>());
  XABE_DOWN(kQ6K, XABE_QUANT_Q6K);
  XABE_DOWN(kQ8_0, XABE_QUANT_Q8_0);
#undef XABE_DOWN
#undef XABE_UP
#undef XABE_LDS
  return XABE_OK;
}

// at handle creation (or a first call without one), for the current device
int decode_block_configure() {
  static DeviceOnce once;
  int dev = 0;
  XABE_HIP_TRY(hipGetDevice(&dev));
  return once.run(dev, decode_block_set_limits);
}

static bool launch_shape(const Launch& l, int gq, int dq, int sgq, int sdq, int router_quant) {
  if (l.a.H == 2048 && l.a.I == 512) return launch_all<1, 4, 4>(l, gq, dq, sgq, sdq, router_quant);
  if (l.a.H == 512 && l.a.I == 256) return launch_all<4, 1, 8>(l, gq, dq, sgq, sdq, router_quant);
  return false;
}

size_t seam_counter_ints_per_token() { return (size_t)kSeamCountersPerToken * kSeamCounterStride; }

bool decode_block_supported(const xabe_moe_kernels* k, const xabe_moe_buffers* b, const xabe_moe_layer_weights* w) {
  const xabe_moe_geometry& g = k->g;
  if (g.max_tokens > kDecodeBlockMaxTokens || k->force_community || b->scope != XABE_SCOPE_ROUTED) return false;
  if (!((g.hidden == 2048 && g.intermediate == 512) || (g.hidden == 512 && g.intermediate == 256))) return false;
  if (g.experts_per_token > (size_t)kMaxTopK || g.num_experts > kRouteMaxExperts || g.num_experts % 4 != 0) return false;
  auto ok = [](int q) { return q == XABE_QUANT_Q6K || q == XABE_QUANT_Q8_0; };
  if (!ok(w->gate_exps.quant) || w->gate_exps.quant != w->up_exps.quant || !ok(w->down_exps.quant)) return false;
  if (!ok(w->shared_gate.quant) || w->shared_gate.quant != w->shared_up.quant || !ok(w->shared_down.quant)) return false;
  if (!(w->router_quant < 0 || w->router_quant == XABE_QUANT_Q8_0)) return false;
  return true;
}

int launch_decode_block(const xabe_moe_kernels* k, hipStream_t s, xabe_moe_buffers* b, const xabe_moe_layer_weights* w,
                        const float* residual, const float* logit_bias, float eps, float* normed, float* logits,
                        float* shexp, float* gate_out, float* routed, float* ffn_out, float* l_out, unsigned launches,
                        const DecodeSeam* seam) {
  const xabe_moe_geometry& g = k->g;
  DecodeArgs a;
  memset(&a, 0, sizeof(a));
  if (seam && seam->next_normed) {
    if (!b->seam_arrivals || b->n_seam_arrivals < g.max_tokens * seam_counter_ints_per_token())
      return set_error(XABE_ERR_INVALID_ARGUMENT, "decode block: these buffers carry no arrival counters for the seam");
    a.next_w = seam->next_w;
    a.next_normed = seam->next_normed;
    a.next_normed_h = static_cast<_Float16*>(seam->next_normed_h);
    a.next_eps = seam->next_eps;
    a.arrivals = b->seam_arrivals;
  }
  a.residual = residual;
  a.post_norm = w->post_norm;
  a.router = static_cast<const uint8_t*>(w->router);
  a.gate = static_cast<const uint8_t*>(w->gate_exps.bytes);
  a.up = static_cast<const uint8_t*>(w->up_exps.bytes);
  a.down = static_cast<const uint8_t*>(w->down_exps.bytes);
  a.sgate = static_cast<const uint8_t*>(w->shared_gate.bytes);
  a.sup = static_cast<const uint8_t*>(w->shared_up.bytes);
  a.sdown = static_cast<const uint8_t*>(w->shared_down.bytes);
  a.shared_gate_inp = w->shared_gate_inp;
  a.logit_bias = logit_bias;
  a.valid_tokens = b->valid_tokens;
  a.normed = normed;
  a.logits = logits;
  a.topk_ids = b->topk_ids;
  a.topk_weights = b->topk_weights;
  a.x_d = b->x_d;
  a.x_e = b->x_e;
  a.inter_d = b->inter_d;
  a.inter_e = b->inter_e;
  a.inter = b->inter;
  a.up_len = w->gate_exps.len;
  a.shared_inter = b->shared_inter;
  a.shexp = shexp;
  a.gate_out = gate_out;
  a.routed = routed;
  a.ffn_out = ffn_out;
  a.l_out = l_out;
  const int rq = w->gate_exps.quant, dq = w->down_exps.quant;
  a.expert_bytes = g.intermediate * g.hidden / xabe_expert_quant_block_elements(rq) * xabe_expert_quant_block_bytes(rq);
  a.down_bytes = g.intermediate * g.hidden / xabe_expert_quant_block_elements(dq) * xabe_expert_quant_block_bytes(dq);
  a.eps = eps;
  a.H = (int)g.hidden;
  a.I = (int)g.intermediate;
  a.E = (int)g.num_experts;
  a.top_k = (int)g.experts_per_token;
  a.max_tokens = (int)g.max_tokens;
  const int rps_h = 2048 / a.H, rps_i = 2048 / a.I;
  const int da = logits_depth(a.max_tokens);
  a.tiles_r = (a.E + kWavesPerWg * rps_h * da - 1) / (kWavesPerWg * rps_h * da);
  a.tiles_s = (a.I + kWavesPerWg * rps_h * da - 1) / (kWavesPerWg * rps_h * da);
  a.tiles_g = a.I / 16;
  a.tiles_d = a.H / (4 * rps_i);
  if (a.E % rps_h != 0)
    return set_error(XABE_ERR_UNSUPPORTED_GEOMETRY, "decode block: %d experts do not fill whole steps of %d rows", a.E, rps_h);
  a.share_g = decode_share((size_t)a.max_tokens * a.top_k, a.tiles_g);
  a.share_d = down_share(k, (size_t)a.max_tokens, a.tiles_d);
  const int chunks = (a.max_tokens + 1) / 2;
  const bool pre_routed = a.max_tokens >= kPreRouteMinTokens;
  const bool pair_units = a.max_tokens >= kPairUnitsMinTokens && rq == XABE_QUANT_Q6K;
  Launch l{a, s, 0, 0, 0, 0, 0, pre_routed, pair_units, seam && seam->input_normed, launches};
  const int row_wgs = a.max_tokens * (a.H / kSbElems + 1);
  if (pre_routed) {
    const int groups = (a.max_tokens + kGroupTokens - 1) / kGroupTokens;
    auto tiles_of = [&](int rows, int steps) { return (rows + kWavesPerWg * rps_h * steps - 1) / (kWavesPerWg * rps_h * steps); };
    a.tiles_r = tiles_of(a.E, kRouterSteps);
    a.tiles_s = tiles_of(a.I, kSharedSteps);
    l.grid_a = (unsigned)(row_wgs + groups * a.tiles_r);
    l.grid_route = (unsigned)(a.max_tokens + groups * a.tiles_s);
  } else {
    l.grid_a = (unsigned)(row_wgs + chunks * (a.tiles_r + a.tiles_s));
  }
  // wide batches pad the shares of a pair (token) to whole rounds of eight, one per XCD
  auto grid_of = [&](size_t units, int shares) { return (unsigned)(units * (a.max_tokens >= kXcdGroupMinTokens ? (shares + 7) / 8 * 8 : shares)); };
  a.shared_from = (int)grid_of((size_t)a.max_tokens * a.top_k, a.tiles_g / a.share_g);
  l.grid_b = (unsigned)(a.shared_from + (pre_routed ? chunks * (a.H / (4 * rps_i * (a.H / 512) * 2)) : 0));
  a.shared_units = chunks * (a.H / (4 * rps_i));
  l.grid_shared = 8u * (unsigned)std::max<size_t>(k->num_cus / 4, ((size_t)a.max_tokens * a.top_k + kMaxUnits - 3) / (kMaxUnits - 2));
  l.grid_c = grid_of((size_t)a.max_tokens, a.tiles_d / a.share_d);
  const bool ok = launch_shape(l, w->gate_exps.quant, w->down_exps.quant, w->shared_gate.quant, w->shared_down.quant, w->router_quant);
  if (!ok) return set_error(XABE_ERR_UNSUPPORTED_GEOMETRY, "decode block: no kernels for this shape or format");
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

}  // namespace xabe
