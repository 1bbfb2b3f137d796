// LM head: logits[t][v] = sum_h W[v][h] * x[t][h] for a [vocab][hidden] matrix in Q8_0, Q6_K, bf16 or f16,
// and the device half of greedy sampling.  Takes the place of crates/xabe-cuda/src/kernels/lm_head.rs.
//
// Three forms.  Hidden sizes up to 2048 in Q8_0 and bf16, and from five tokens on in Q6_K, take k_head_tiles_*
// (lm_head_tiles.hip), up to sixteen tokens per pass over the weights; other quantized matrices k_lm_head_quant, on the
// digit contraction (digits.h), up to eight; f16 and longer bf16 rows k_lm_head_half, on the vector ALU, up to four.
// Nothing depends on the batch: a token's logits are the same bits at every batch width and position.
#include <string.h>

#include <algorithm>
#include <utility>

#include "../../include/xabe_gguf.h"
#include "../../include/xabe_lm_head.h"
#include "decode_kernels.h"
#include "digits.h"
#include "host_common.h"
#include "lm_head_tiles.h"

namespace xabe {

// Q8_0 / Q6_K rows, NT tokens.  The launch is one workgroup per CU; every wavefront owns a contiguous range of the
// vocabulary and takes it 32 rows and one superblock at a time through its own LDS slot (SliceDma), against the tokens'
// digits, which the workgroup makes once and keeps in LDS.  A wavefront's ranges are equal to within a row, so the last
// round of tiles is as long for everyone: 7760 tiles of 32 rows do not divide over 2048 wavefronts, rows do.
// Per row and token: superblock sums in order, each half of the wavefront its own, then half 0 + half 1.
// Bound by bytes up to a few tokens (the model's Q6_K matrix: 82 us for one, 93 for three), by the vector ALU beyond.  Eight
// wavefronts per CU: twelve and sixteen measured slower.
// SEG: rows whose digits do not fit in LDS are staged seg_sb superblocks at a time, again for every tile.
constexpr size_t kHeadLdsMax = 160 * 1024;
constexpr size_t kHeadQuantTokens = 8;  // tokens per pass over a quantized matrix

template <int QUANT, int NT, bool SEG>
__global__ void __launch_bounds__(512, 2) k_lm_head_quant(LmHeadArgs a) {
  using Dma = SliceDma<QUANT>;
  extern __shared__ __attribute__((aligned(16))) uint8_t s_head[];
  const int lane = (int)__lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int waves = (int)(blockDim.x >> 6);
  const int nsb = a.K / kSbElems, seg_sb = SEG ? a.seg_sb : nsb;
  uint8_t* const s_zero = s_head;
  uint8_t* const s_x = s_zero + kZeroBytes;                             // [superblock][token][kSbLdsBytes]
  uint8_t* const slot = s_x + (size_t)seg_sb * NT * kSbLdsBytes + (size_t)wave * Dma::kSlotBytes;
  const uint32_t slot_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)slot;
  const uint32_t row_bytes = (uint32_t)nsb * SbRaw<QUANT>::kBytes;
  const int index = (int)blockIdx.x * waves + wave, n_waves = (int)gridDim.x * waves;
  const int row_lo = (int)((long long)a.vocab * index / n_waves), row_hi = (int)((long long)a.vocab * (index + 1) / n_waves);
  const int tiles = SEG ? (int)((a.vocab / n_waves + 1 + 31) / 32) : (row_hi - row_lo + 31) / 32;  // (SEG: barriers inside, so the same for all)

  auto stage = [&](int sb0) __attribute__((always_inline)) {
    const int n = min(seg_sb, nsb - sb0) * 16;  // groups of 16 per token
    for (int i = threadIdx.x; i < NT * n; i += (int)blockDim.x) {
      const int t = i / n, gi = i % n, sb = gi >> 4, pos = gi & 15;
      const float4* src = reinterpret_cast<const float4*>(a.x + (size_t)(a.t0 + min(t, a.nt - 1)) * a.K + (size_t)sb0 * kSbElems + gi * 16);
      float x[16];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4 f = src[j];
        x[4 * j] = f.x, x[4 * j + 1] = f.y, x[4 * j + 2] = f.z, x[4 * j + 3] = f.w;
      }
      uint8_t* base = s_x + (size_t)(sb * NT + t) * kSbLdsBytes;
      const float scale = digitize_superblock(x, pos, base);  // (a superblock's groups: sixteen consecutive threads)
      if (pos == 0) *reinterpret_cast<float*>(base + kSbDigitBytes) = scale;
    }
  };

  Dma dma[2];
  int row0 = 0;
  auto take_tile = [&](int i) __attribute__((always_inline)) {
    row0 = min(row_lo + 32 * i, a.vocab - 1);
    const int live = max(1, row_hi - row0);
    if (i == 0 || live < 32) {
#pragma unroll
      for (int u = 0; u < 2; ++u) dma[u].init(row_bytes, min(max(live - 16 * u, 1), 16));
    }
  };
  auto run_off = [&](int u) __attribute__((always_inline)) { return (size_t)min(row0 + 16 * u, a.vocab - 1) * row_bytes; };
  auto request = [&](int sb) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) dma[u].request(a.w, a.w_bytes, run_off(u), sb, slot_lds + u * Dma::kRunBytes);
  };
  if (tiles > 0) {
    take_tile(0);
    request(0);
  }
  for (int i = threadIdx.x; i < kZeroBytes / 16; i += (int)blockDim.x) reinterpret_cast<v4u_t*>(s_zero)[i] = v4u_t{0, 0, 0, 0};
  if constexpr (!SEG) {
    stage(0);
    __syncthreads();
  }
  const int u = (lane >> 4) & 1, r = lane & 15, h = lane >> 5;
  for (int i = 0; i < tiles; ++i) {
    float acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = 0.0f;
    const int my_row = row0 + (lane & 31);
#pragma unroll 1
    for (int sb = 0; sb < nsb; ++sb) {
      if constexpr (SEG) {
        if (sb % seg_sb == 0) {
          __syncthreads();
          stage(sb);
          __syncthreads();
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (sb == nsb - 1 && dma[0].ends_apart(a.w_bytes)) {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          const int live = a.vocab - (row0 + 16 * v);
          if (live >= 1 && live <= 16 && row_hi == a.vocab) dma[v].patch_tail(a.w, run_off(v), live, sb, slot + v * Dma::kRunBytes);
        }
      }
      SbRaw<QUANT> raw;
      sb_read_slot(dma[0].row_at(slot + u * Dma::kRunBytes, run_off(u), r, sb), h, raw);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (sb + 1 < nsb) {
        request(sb + 1);
      } else if (i + 1 < tiles) {
        take_tile(i + 1);
        request(0);
      }
      LdsDigits<NT, kSbLdsBytes, QUANT == kQ8_0> x;
      const uint8_t* sb_x = s_x + (size_t)(SEG ? sb % seg_sb : sb) * NT * kSbLdsBytes;
      x.point(sb_x, sb_x + kSbDigitBytes, s_zero);
      float v[NT];
      sb_dot<QUANT, kWhole, NT>(
          raw, [&](int s, int l, int tg) { return x.high(s, l, tg); }, [&](int s, int l, int tg) { return x.low(s, l, tg); },
          [&](int t, int) { return *reinterpret_cast<const float*>(sb_x + t * kSbLdsBytes + kSbDigitBytes); },
          [&](int t) { return a.x + (size_t)(a.t0 + min(t, a.nt - 1)) * a.K + sb * kSbElems; }, v,
          __builtin_amdgcn_ballot_w64(my_row < row_hi));
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] += v[t];
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float total = acc[t] + __shfl_xor(acc[t], 32, 64);
      if (h == 0 && my_row < row_hi && t < a.nt) a.out[(size_t)(a.t0 + t) * a.vocab + my_row] = total;
    }
  }
}

// bf16 / f16 rows: lane l covers elements j*512 + 8*l .. +8 of every 512-element section j.
typedef uint32_t piece16 __attribute__((ext_vector_type(4)));

template <bool F16>
__device__ __forceinline__ void widen8(const piece16& p, float (&w)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (F16) {
      w[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(p[i] & 0xffffu));
      w[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(p[i] >> 16));
    } else {  // bf16 is a truncated f32: the widening is a shift
      w[2 * i] = __builtin_bit_cast(float, p[i] << 16);
      w[2 * i + 1] = __builtin_bit_cast(float, p[i] & 0xffff0000u);
    }
  }
}

// SEC > 0: K = 512 * SEC, activations in registers; SEC == 0: sections from K at run time, activations re-read.
template <bool F16, int R, int TOK, int SEC>
__global__ void __launch_bounds__(256) k_lm_head_half(LmHeadArgs a) {
  const int lane = (int)__lane_id();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int groups = (a.vocab + R - 1) / R;
  const int stride = (int)gridDim.x * kWavesPerWg;
  const int sections = a.K / 512;
  constexpr int kHeld = SEC > 0 ? SEC : 1;
  float x[TOK][kHeld][8];
  auto load_x = [&](int j, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TOK; ++t) {
      const float4* p = reinterpret_cast<const float4*>(a.x + (size_t)(a.t0 + min(t, a.nt - 1)) * a.K + j * 512 + lane * 8);
      const float4 u = p[0], v = p[1];
      x[t][slot][0] = u.x, x[t][slot][1] = u.y, x[t][slot][2] = u.z, x[t][slot][3] = u.w;
      x[t][slot][4] = v.x, x[t][slot][5] = v.y, x[t][slot][6] = v.z, x[t][slot][7] = v.w;
    }
  };
  if constexpr (SEC > 0) {
#pragma unroll
    for (int j = 0; j < SEC; ++j) load_x(j, j);
  }
  auto row_ptr = [&](int rg, int r) __attribute__((always_inline)) {
    const int row = min(rg * R + r, a.vocab - 1);
    return reinterpret_cast<const piece16*>(a.w + (size_t)row * a.K * 2) + lane;
  };
  int rg = (int)blockIdx.x * kWavesPerWg + wave;
  if (rg >= groups) return;
  piece16 pend[R][kHeld];
  auto issue_w = [&](int g2, int j0) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int j = 0; j < kHeld; ++j) pend[r][j] = row_ptr(g2, r)[(j0 + j) * 64];
    issue_fence();
  };
  issue_w(rg, 0);
#pragma unroll 1
  for (; rg < groups; rg += stride) {
    float acc[R][TOK];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int t = 0; t < TOK; ++t) acc[r][t] = 0.0f;
    const int n_sec = SEC > 0 ? 1 : sections;
#pragma unroll 1
    for (int j = 0; j < n_sec; ++j) {
      piece16 cur[R][kHeld];
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int h = 0; h < kHeld; ++h) cur[r][h] = pend[r][h];
      if (SEC == 0) load_x(j, 0);
      // next pieces: the next section of this group, or the first of the next group
      if (j + 1 < n_sec) issue_w(rg, j + 1);
      else if (rg + stride < groups) issue_w(rg + stride, 0);
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int h = 0; h < kHeld; ++h) {
          float w[8];
          widen8<F16>(cur[r][h], w);
#pragma unroll
          for (int t = 0; t < TOK; ++t)
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[r][t] += w[i] * x[t][h][i];
        }
    }
#pragma unroll
    for (int t = 0; t < TOK; ++t) {
      if (t >= a.nt) break;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float tot = group_sum<64>(acc[r][t]);
        const int row = rg * R + r;
        if (lane == 0 && row < a.vocab) a.out[(size_t)(a.t0 + t) * a.vocab + row] = tot;
      }
    }
  }
}

// ---------------------------------------------------------------------------------
// argmax with the scalar reference's semantics (crates/xabe-kernels/src/gemv.rs:103-112: `best` moves only on
// a strictly greater value, so the first maximum wins, a NaN never wins, and a NaN at index 0 is never
// displaced).  A candidate is (value, index); NaN candidates are dropped, equal values keep the lower index.
// ---------------------------------------------------------------------------------
struct Cand {
  float v;
  int i;
};
__device__ __forceinline__ Cand better(Cand a, Cand b) {
  const bool take_b = b.i >= 0 && (a.i < 0 || b.v > a.v || (b.v == a.v && b.i < a.i));
  return take_b ? b : a;
}
template <int CTRL>
__device__ __forceinline__ Cand dpp_best(Cand c) {
  const Cand o{dpp_f<CTRL>(c.v), dpp_i<CTRL>(c.i)};
  return better(c, o);
}
__device__ __forceinline__ Cand lane_cand(Cand c, int lane) {
  return Cand{lane_bcast(c.v, lane), __builtin_amdgcn_readlane(c.i, lane)};
}
// The order of the comparisons does not matter (equal values keep the lower index), so the wavefront goes by data
// parallel moves inside its 16-lane rows and scalar reads across them, without a trip through LDS.
__device__ __forceinline__ Cand block_best(Cand c, Cand* s) {
  c = dpp_best<0xB1>(c);
  c = dpp_best<0x4E>(c);
  c = dpp_best<0x141>(c);
  c = dpp_best<0x140>(c);
  c = better(better(lane_cand(c, 0), lane_cand(c, 16)), better(lane_cand(c, 32), lane_cand(c, 48)));
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) s[wave] = c;
  __syncthreads();
  Cand r = s[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = better(r, s[w]);
  return r;
}

// Bound by latency (a megabyte of logits over the whole chip): one 16-byte load per thread covers the vocabulary of
// the shipped model in one round, where a strided scalar loop made two.
__global__ void __launch_bounds__(256) k_argmax_partial(const float* __restrict__ v, int n, float* __restrict__ pv,
                                                         int* __restrict__ pi) {
  __shared__ Cand s[4];
  Cand c{0.0f, -1};
  auto take = [&](float x, int i) __attribute__((always_inline)) {
    if (x == x) c = better(c, Cand{x, i});
  };
  const int head = min(n, (int)((16 - (reinterpret_cast<uintptr_t>(v) & 15)) & 15) / 4);  // values before the first 16-byte boundary
  const int quads = (n - head) / 4;
  for (int q = blockIdx.x * 256 + threadIdx.x; q < quads; q += gridDim.x * 256) {
    const float4 x = reinterpret_cast<const float4*>(v + head)[q];
    const int i = head + 4 * q;
    take(x.x, i);
    take(x.y, i + 1);
    take(x.z, i + 2);
    take(x.w, i + 3);
  }
  if (blockIdx.x == gridDim.x - 1) {
    if ((int)threadIdx.x < head) take(v[threadIdx.x], threadIdx.x);
    const int rest = head + 4 * quads + (int)threadIdx.x;
    if (rest < n) take(v[rest], rest);
  }
  c = block_best(c, s);
  if (threadIdx.x == 0) {
    pv[blockIdx.x] = c.v;
    pi[blockIdx.x] = c.i;
  }
}

__global__ void __launch_bounds__(256) k_argmax_final(const float* __restrict__ pv, const int* __restrict__ pi, int blocks,
                                                       const float* __restrict__ v, int* __restrict__ out) {
  __shared__ Cand s[4];
  const float first = v[0];
  const int b0 = min((int)threadIdx.x, blocks - 1), b1 = min((int)threadIdx.x + 256, blocks - 1);  // (at most 512)
  Cand c = better(Cand{pv[b0], pi[b0]}, Cand{pv[b1], pi[b1]});
  c = block_best(c, s);
  if (threadIdx.x == 0) out[0] = (first != first || c.i < 0) ? 0 : c.i;
}

// 1 / sum(exp(x - max)): one workgroup, a maximum pass and a sum pass, both in a fixed order.
__global__ void __launch_bounds__(256) k_argmax_prob(const float* __restrict__ v, int n, float* __restrict__ out) {
  __shared__ float s[4];
  float m = -INFINITY;
  for (int i = threadIdx.x; i < n; i += 256) m = fmaxf(m, v[i]);
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
  __syncthreads();
  float sum = 0.0f;
  for (int i = threadIdx.x; i < n; i += 256) sum += expf(v[i] - m);
  sum = group_sum<64>(sum);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) out[0] = 1.0f / ((s[0] + s[1]) + (s[2] + s[3]));
}

static size_t format_elements(int format, size_t bytes, size_t* block_bytes) {
  switch (format) {
    case XABE_HEAD_Q8_0: *block_bytes = kQ8Bytes; return bytes / kQ8Bytes * 32;
    case XABE_HEAD_Q6K: *block_bytes = kQ6KBytes; return bytes / kQ6KBytes * 256;
    default: *block_bytes = 2; return bytes / 2;
  }
}

template <int QUANT, int NT, bool SEG>
static int head_raise_lds() {
  XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_lm_head_quant<QUANT, NT, SEG>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kHeadLdsMax));
  return XABE_OK;
}
template <int QUANT, int... NT>
static int head_raise_all(std::integer_sequence<int, NT...>) {
  int st = head_raise_lds<QUANT, 1, true>();
  ((st = st == XABE_OK ? head_raise_lds<QUANT, NT + 1, false>() : st), ...);
  return st;
}
// at handle creation, not on the launch path (launches are captured into graphs)
static int head_configure() {
  XABE_TRY(head_tiles_configure());
  XABE_TRY((head_raise_all<kQ8_0>(std::make_integer_sequence<int, (int)kHeadQuantTokens>())));
  return head_raise_all<kQ6K>(std::make_integer_sequence<int, (int)kHeadQuantTokens>());
}

}  // namespace xabe

using xabe::set_error;

struct xabe_lm_head {
  xabe_lm_head_geometry g;
  int num_cus;
};

static int bad_head(const xabe_lm_head_geometry& g, const char* reason) {
  return set_error(XABE_ERR_UNSUPPORTED_GEOMETRY, "unsupported LM head geometry LmHeadGeometry { hidden: %zu, vocab: %zu, max_tokens: %zu }: %s",
                   g.hidden, g.vocab, g.max_tokens, reason);
}

static int check_len(const char* what, size_t expected, size_t got) {
  if (got == expected) return XABE_OK;
  return set_error(XABE_ERR_SHAPE_MISMATCH, "%s: expected %zu elements, got %zu", what, expected, got);
}

extern "C" {

int xabe_head_format_from_ggml(int t) {
  switch (t) {
    case XABE_GGML_Q8_0: return XABE_HEAD_Q8_0;
    case XABE_GGML_BF16: return XABE_HEAD_BF16;
    case XABE_GGML_Q6_K: return XABE_HEAD_Q6K;
    case XABE_GGML_F16: return XABE_HEAD_F16;
    case XABE_GGML_Q4_0: return XABE_HEAD_Q4_0;
    case XABE_GGML_Q4_K: return XABE_HEAD_Q4K;
    case XABE_GGML_Q5_K: return XABE_HEAD_Q5K;
  }
  return -1;
}

xabe_lm_head_geometry xabe_lm_head_geometry_qwen3_6(size_t max_tokens) {
  xabe_lm_head_geometry g = {2048, 248320, max_tokens};
  return g;
}

size_t xabe_lm_head_row_bytes_for(const xabe_lm_head_geometry* g, int format) {
  if (!g) return 0;
  switch (format) {
    case XABE_HEAD_Q8_0: return g->hidden / 32 * 34;
    case XABE_HEAD_Q6K: return g->hidden / 256 * 210;
    case XABE_HEAD_BF16: case XABE_HEAD_F16: return g->hidden * 2;
    case XABE_HEAD_Q4_0: return g->hidden / 32 * 18;
    case XABE_HEAD_Q4K: return g->hidden / 256 * 144;
    case XABE_HEAD_Q5K: return g->hidden / 256 * 176;
  }
  return 0;
}

size_t xabe_lm_head_weight_bytes_for(const xabe_lm_head_geometry* g, int format) {
  return g ? g->vocab * xabe_lm_head_row_bytes_for(g, format) : 0;
}
size_t xabe_lm_head_elements(const xabe_lm_head_geometry* g) { return g ? g->vocab * g->hidden : 0; }
size_t xabe_lm_head_weight_passes(const xabe_lm_head_geometry*, size_t tokens) {
  return (tokens + XABE_LM_HEAD_MAX_BATCH_TILE - 1) / XABE_LM_HEAD_MAX_BATCH_TILE;
}
size_t xabe_lm_head_weight_bytes_read(const xabe_lm_head_geometry* g, int format, size_t tokens) {
  return xabe_lm_head_weight_bytes_for(g, format) * xabe_lm_head_weight_passes(g, tokens);
}

int xabe_lm_head_new(const xabe_lm_head_geometry* geometry, xabe_lm_head** out) {
  if (!geometry || !out) return set_error(XABE_ERR_INVALID_ARGUMENT, "null geometry or output pointer");
  const xabe_lm_head_geometry& g = *geometry;
  if (g.hidden == 0 || g.vocab == 0) return bad_head(g, "hidden and vocab must be non-zero");
  if (g.hidden % 512 != 0) return bad_head(g, "hidden must be a whole number of 16-block staging segments (a multiple of 512)");
  if (g.max_tokens == 0) return bad_head(g, "max_tokens must be non-zero");
  if (g.vocab > 0x7fffffffu || g.hidden > 0x7fffffffu) return bad_head(g, "vocabulary exceeds the grid.x limit");
  int dev = 0, cus = 256;
  XABE_HIP_TRY(hipGetDevice(&dev));
  XABE_HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  XABE_TRY(xabe::head_configure());
  xabe_lm_head* h = new xabe_lm_head();
  h->g = g;
  h->num_cus = cus;
  *out = h;
  return XABE_OK;
}

void xabe_lm_head_free(xabe_lm_head* h) { delete h; }

int xabe_lm_head_geometry_of(const xabe_lm_head* h, xabe_lm_head_geometry* out) {
  if (!h || !out) return set_error(XABE_ERR_INVALID_ARGUMENT, "null handle or output pointer");
  *out = h->g;
  return XABE_OK;
}

}  // extern "C"

namespace xabe {

template <int QUANT, int NT, bool SEG>
static int launch_quant(unsigned grid, unsigned waves, size_t smem, hipStream_t s, const LmHeadArgs& a) {
  hipLaunchKernelGGL((k_lm_head_quant<QUANT, NT, SEG>), dim3(grid), dim3(64 * waves), smem, s, a);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

// Wavefronts of a workgroup in a pass of nt tokens: as many, up to eight, as the digits leave LDS for (0: not even one).
template <int QUANT>
static size_t head_waves(size_t K, size_t nt) {
  const size_t room = kHeadLdsMax - kZeroBytes, digits = K / kSbElems * nt * kSbLdsBytes;
  return digits > room ? 0 : std::min<size_t>(8, (room - digits) / SliceDma<QUANT>::kSlotBytes);
}
// Tokens of one pass over the matrix: as many as leave room for four wavefronts, or one.
template <int QUANT>
static size_t head_tokens(size_t K) {
  size_t nt = kHeadQuantTokens;
  while (nt > 1 && head_waves<QUANT>(K, nt) < 4) --nt;
  return nt;
}

template <int QUANT>
static int launch_quant_pass(const xabe_lm_head* h, hipStream_t s, LmHeadArgs a) {
  constexpr size_t kSlot = SliceDma<QUANT>::kSlotBytes;
  const size_t fit = head_waves<QUANT>(a.K, a.nt), waves = std::max<size_t>(1, fit);
  // one workgroup per CU, and no more than there are tiles for
  const unsigned w = (unsigned)waves, grid = (unsigned)std::max<size_t>(1, std::min<size_t>(h->num_cus, ((size_t)a.vocab + 32 * waves - 1) / (32 * waves)));
  a.seg_sb = fit ? a.K / kSbElems : (int)((kHeadLdsMax - kZeroBytes - kSlot) / kSbLdsBytes);
  const size_t smem = kZeroBytes + (size_t)a.seg_sb * a.nt * kSbLdsBytes + waves * kSlot;
  if (!fit) return launch_quant<QUANT, 1, true>(grid, 1, smem, s, a);  // (rows of more than 24 000 elements, one token)
  switch (a.nt) {
    case 1: return launch_quant<QUANT, 1, false>(grid, w, smem, s, a);
    case 2: return launch_quant<QUANT, 2, false>(grid, w, smem, s, a);
    case 3: return launch_quant<QUANT, 3, false>(grid, w, smem, s, a);
    case 4: return launch_quant<QUANT, 4, false>(grid, w, smem, s, a);
    case 5: return launch_quant<QUANT, 5, false>(grid, w, smem, s, a);
    case 6: return launch_quant<QUANT, 6, false>(grid, w, smem, s, a);
    case 7: return launch_quant<QUANT, 7, false>(grid, w, smem, s, a);
    default: return launch_quant<QUANT, 8, false>(grid, w, smem, s, a);
  }
}

template <int TOK>
static void launch_half_pass(const xabe_lm_head* h, hipStream_t s, bool f16, const LmHeadArgs& a) {
  // rows per wavefront iteration: four for one token, two once the tile's activations take the registers
  constexpr int R = TOK == 1 ? 4 : 2;
  const int groups = (a.vocab + R - 1) / R;
  const unsigned grid = (unsigned)std::max(1, std::min((groups + kWavesPerWg - 1) / kWavesPerWg, h->num_cus * 4));
  if (!f16) hipLaunchKernelGGL((k_lm_head_half<false, R, TOK, 0>), dim3(grid), dim3(256), 0, s, a);  // (of more than 2048 elements)
  else if (a.K == 2048) hipLaunchKernelGGL((k_lm_head_half<true, R, TOK, 4>), dim3(grid), dim3(256), 0, s, a);
  else hipLaunchKernelGGL((k_lm_head_half<true, R, TOK, 0>), dim3(grid), dim3(256), 0, s, a);
}

}  // namespace xabe

extern "C" {

int xabe_lm_head_forward(const xabe_lm_head* h, void* stream, int format, const void* weight, size_t weight_len,
                         const float* hidden_states, size_t hidden_states_len, size_t tokens, float* logits,
                         size_t logits_len) {
  if (!h || !weight || !hidden_states || !logits) return set_error(XABE_ERR_INVALID_ARGUMENT, "null handle or buffer");
  const xabe_lm_head_geometry& g = h->g;
  switch (format) {
    case XABE_HEAD_Q8_0: case XABE_HEAD_Q6K: case XABE_HEAD_BF16: case XABE_HEAD_F16: break;
    case XABE_HEAD_Q4_0: case XABE_HEAD_Q4K: case XABE_HEAD_Q5K:
      return set_error(XABE_ERR_UNSUPPORTED_QUANT, "LM head: format %d is recognised, but this library has kernels for Q8_0, Q6_K, bf16 and f16 only", format);
    default: return set_error(XABE_ERR_INVALID_ARGUMENT, "LM head: unknown format %d", format);
  }
  if (format == XABE_HEAD_Q6K && g.hidden % 256 != 0)
    return set_error(XABE_ERR_UNSUPPORTED_GEOMETRY, "the Q6_K GEMV covers 256 elements per warp step, so `hidden` must be a multiple of 256, not %zu", g.hidden);
  size_t block_bytes = 0;
  const size_t found = xabe::format_elements(format, weight_len, &block_bytes);
  if (weight_len % block_bytes != 0)
    return set_error(XABE_ERR_RAGGED_WEIGHTS, "LM head: %zu bytes is not a whole number of %zu B blocks", weight_len, block_bytes);
  if (found != g.vocab * g.hidden)
    return set_error(XABE_ERR_WRONG_ELEMENT_COUNT, "LM head: expected %zu elements for this geometry, tensor holds %zu", g.vocab * g.hidden, found);
  if (tokens == 0 || tokens > g.max_tokens)
    return set_error(XABE_ERR_TOO_MANY_TOKENS, "%zu tokens is outside 1..=%zu, the range the buffers were sized for", tokens, g.max_tokens);
  XABE_TRY(check_len("hidden states", g.max_tokens * g.hidden, hidden_states_len));
  XABE_TRY(check_len("logits", g.max_tokens * g.vocab, logits_len));
  if ((reinterpret_cast<uintptr_t>(weight) & 15u) != 0 || (reinterpret_cast<uintptr_t>(hidden_states) & 15u) != 0)
    return set_error(XABE_ERR_INVALID_ARGUMENT, "LM head: the weight tensor and the hidden states must start on 16-byte boundaries");
  hipStream_t s = xabe::as_stream(stream);
  xabe::LmHeadArgs a;
  a.w = static_cast<const uint8_t*>(weight);
  a.x = hidden_states;
  a.out = logits;
  a.K = (int)g.hidden;
  a.vocab = (int)g.vocab;
  a.w_bytes = weight_len;
  a.seg_sb = 0;
  const bool quant = format == XABE_HEAD_Q8_0 || format == XABE_HEAD_Q6K;
  // (Q6_K: forward pass over the model's vocabulary, us, k_lm_head_quant / tiles: one token 82 / 112, two 84 / 107, three 90 / 104, four
  // 94 / 104, five 119 / 108, eight 160 / 106, sixteen 311 / 152; the same bits)
  const bool tiles = xabe::head_tiles_width(g.hidden) &&
                     (format == XABE_HEAD_Q8_0 || format == XABE_HEAD_BF16 || (format == XABE_HEAD_Q6K && tokens > 4));
  // passes of equal width: nine tokens as five and four, not as eight and one
  const size_t most = tiles ? xabe::kHeadTileTokens
                    : !quant ? XABE_LM_HEAD_MAX_BATCH_TILE
                    : format == XABE_HEAD_Q8_0 ? xabe::head_tokens<xabe::kQ8_0>(g.hidden) : xabe::head_tokens<xabe::kQ6K>(g.hidden);
  const size_t passes = (tokens + most - 1) / most, width = (tokens + passes - 1) / passes;
  for (size_t base = 0; base < tokens; base += width) {
    const int tile = (int)std::min<size_t>(width, tokens - base);
    a.t0 = (int)base;
    a.nt = tile;
    if (tiles) {
      XABE_TRY(format == XABE_HEAD_BF16 ? xabe::launch_head_tiles_bf16(s, h->num_cus, a)
               : format == XABE_HEAD_Q8_0 ? xabe::launch_head_tiles_q8(s, h->num_cus, a)
                                          : xabe::launch_head_tiles_q6k(s, h->num_cus, a));
      continue;
    }
    if (format == XABE_HEAD_Q8_0) {
      XABE_TRY(xabe::launch_quant_pass<xabe::kQ8_0>(h, s, a));
      continue;
    }
    if (format == XABE_HEAD_Q6K) {
      XABE_TRY(xabe::launch_quant_pass<xabe::kQ6K>(h, s, a));
      continue;
    }
    const bool f16 = format == XABE_HEAD_F16;
    switch (tile) {
      case 1: xabe::launch_half_pass<1>(h, s, f16, a); break;
      case 2: xabe::launch_half_pass<2>(h, s, f16, a); break;
      case 3: xabe::launch_half_pass<3>(h, s, f16, a); break;
      default: xabe::launch_half_pass<4>(h, s, f16, a); break;
    }
    XABE_HIP_TRY(hipGetLastError());
  }
  return XABE_OK;
}

int xabe_lm_head_argmax(const xabe_lm_head* h, void* stream, const float* values, size_t values_len, size_t n,
                        float* partial_values, size_t partial_values_len, int32_t* partial_indices,
                        size_t partial_indices_len, int32_t* out, size_t out_len) {
  if (!h || !values || !partial_values || !partial_indices || !out) return set_error(XABE_ERR_INVALID_ARGUMENT, "null handle or buffer");
  if (n == 0 || n > values_len || n > 0x7fffffffu)
    return set_error(XABE_ERR_SHAPE_MISMATCH, "argmax length: expected %zu elements, got %zu", values_len, n);
  XABE_TRY(check_len("argmax partial values", XABE_LM_HEAD_ARGMAX_BLOCKS, partial_values_len));
  XABE_TRY(check_len("argmax partial indices", XABE_LM_HEAD_ARGMAX_BLOCKS, partial_indices_len));
  XABE_TRY(check_len("argmax output", 1, out_len));
  const unsigned blocks = (unsigned)std::min<size_t>((n + 1023) / 1024, XABE_LM_HEAD_ARGMAX_BLOCKS);
  hipStream_t s = xabe::as_stream(stream);
  hipLaunchKernelGGL(xabe::k_argmax_partial, dim3(blocks), dim3(256), 0, s, values, (int)n, partial_values, partial_indices);
  XABE_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(xabe::k_argmax_final, dim3(1), dim3(256), 0, s, partial_values, partial_indices, (int)blocks, values, out);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

int xabe_lm_head_argmax_prob(const xabe_lm_head* h, void* stream, const float* values, size_t values_len, size_t n,
                             float* out, size_t out_len) {
  if (!h || !values || !out) return set_error(XABE_ERR_INVALID_ARGUMENT, "null handle or buffer");
  if (n == 0 || n > values_len || n > 0x7fffffffu)
    return set_error(XABE_ERR_SHAPE_MISMATCH, "argmax_prob length: expected %zu elements, got %zu", values_len, n);
  XABE_TRY(check_len("argmax_prob output", 1, out_len));
  hipLaunchKernelGGL(xabe::k_argmax_prob, dim3(1), dim3(256), 0, xabe::as_stream(stream), values, (int)n, out);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

}  // extern "C"
