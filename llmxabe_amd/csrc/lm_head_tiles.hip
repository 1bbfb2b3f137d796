// LM head rows of up to 2048 elements against up to sixteen tokens in one pass over the matrix.
//
// A workgroup has one wavefront per 256 elements of the contraction and a contiguous share of the vocabulary, which it
// takes 32 rows at a time: every wavefront multiplies its 256 columns of the tile, the sums meet in LDS and are added in a
// fixed order.  A wavefront's activations never change, so its operands of the matrix instruction stay in registers for the
// whole launch (up to sixteen tokens: 96 or 128 registers), and LDS carries nothing but weight bytes (a slot per wavefront,
// filled by DMA) and the sums.  Wavefronts that own rows instead (k_lm_head_quant) read the digits of every superblock out
// of LDS for every tile and find room for those of eight tokens at most; lanes that hold activations, for four tokens.
//
// A tile is two sets of sixteen rows, each with its half of the slot: once a set's bytes are in registers the same rows of
// the next tile are requested, so that between one and two halves are on their way at any time.  Waits are by count.  The
// tile before is added up and stored between the second set's wait and its request: stores count with the loads, and
// there half a tile's time passes before one is waited for.  Shares are whole tiles, so that a token's 32 logits are one
// line of memory.
//
// Bound by bytes, but for Q6_K's vector instructions at more than eight tokens.  248 320 x 2048, us for a pass over the
// matrix, before / with these (1 / 3 / 8 / 16 tokens): Q8_0 99 / 107 / 153 / 294, now 97 / 102 / 111 / 128 (5.6 to
// 4.2 TB/s); bf16 178 / 189 / 389 / 756, now 173 / 180 / 186 / 197 (5.9 to 5.2 TB/s); Q6_K at 5 / 8 / 16 tokens 119 / 160
// / 311, now 108 / 106 / 152.  (One request per tile, and shares that do not start on a line: Q8_0 106 / 108 / 119 / 150.)
//
// Per (row, token) the order of operations is fixed: a token's logits are the same bits at every batch width.
#include <algorithm>

#include "digits.h"
#include "host_common.h"
#include "lm_head_tiles.h"
#include "planes.h"

namespace xabe {

typedef _Float16 v8h_t __attribute__((ext_vector_type(8)));
typedef __bf16 v8b_t __attribute__((ext_vector_type(8)));
typedef float v4f_t __attribute__((ext_vector_type(4)));
typedef _Float16 v2h_t __attribute__((ext_vector_type(2)));

constexpr int kTileRows = 32;

// What every form has in common: the workgroup's rows, the sums' places, the reduction.
struct HeadShare {
  int lane, wave, waves, r, g;   // r, g: the lane's weight row of a set of sixteen and its quarter
  int row_lo, row_hi, tiles;
  __device__ __forceinline__ HeadShare(int vocab) {
    lane = (int)__lane_id();
    wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    waves = (int)(blockDim.x >> 6);
    r = lane & 15;
    g = lane >> 4;
    // whole tiles, so that a token's 32 logits of a tile are a line of memory (shares equal to within a row are as long)
    const int all = (vocab + kTileRows - 1) / kTileRows, lo = (int)((long long)all * blockIdx.x / gridDim.x);
    tiles = (int)((long long)all * (blockIdx.x + 1) / gridDim.x) - lo;
    row_lo = lo * kTileRows;
    row_hi = min(row_lo + tiles * kTileRows, vocab);
  }
};

// All but the last N of this wavefront's requests are there (stores count, too); the last tile waits for everything.
template <int N>
__device__ __forceinline__ void wait_tile(bool last) {
  if (last) wait_but<0>();
  else wait_but<N>();
}

// The sums the wavefronts left at red[wave][half][token][32], added and stored.  HALVES 2: one after the other, each half of
// the superblocks by itself, then the two (k_lm_head_quant's order); otherwise in pairs.
template <int HALVES, int TOKENS>
__device__ __forceinline__ void head_reduce(const float* red, const HeadShare& sh, const LmHeadArgs& a, int row0) {
  constexpr int kStride = HALVES * TOKENS * kTileRows;
#pragma unroll 1
  for (int i = threadIdx.x; i < a.nt * kTileRows; i += (int)blockDim.x) {
    const int t = i / kTileRows, row = row0 + i % kTileRows;
    float part[HALVES][8], total[HALVES];
#pragma unroll
    for (int h = 0; h < HALVES; ++h)
#pragma unroll
      for (int w = 0; w < 8; ++w) part[h][w] = red[min(w, sh.waves - 1) * kStride + h * TOKENS * kTileRows + i];
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
      float (&p)[8] = part[h];
#pragma unroll
      for (int w = 0; w < 8; ++w) p[w] = w < sh.waves ? p[w] : 0.0f;
      if constexpr (HALVES == 2) {
        total[h] = 0.0f;
#pragma unroll
        for (int w = 0; w < 8; ++w) total[h] += p[w];
      } else {
        total[h] = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
      }
    }
    if (row < sh.row_hi) a.out[(size_t)(a.t0 + t) * a.vocab + row] = HALVES == 2 ? total[0] + total[HALVES - 1] : total[0];
  }
}

// Activations of the tokens whose superblock is marked, as they came: the LDS behind the sums holds those of the first PLACES
// tokens of every wavefront, 1 KB each, for the whole launch.  Fetched per tile they would be waited for behind the requested rows, and
// every wavefront of the workgroup waits for the one that sums a superblock again, so that it takes its weights, too, from where they
// are: registers, or the slot.  248 320 x 2048, one marked superblock in the pass, us, weights and activations fetched / this: Q8_0 at 1
// / 3 / 8 / 16 tokens 238 / 240 / 220 / 217, now 98 / 101 / 130 / 157; Q6_K at 5 / 8 / 16 174 / 175 / 205, now 137 / 137 / 172.
template <int PLACES>
struct MarkedRows {
  const float* at;  // the wavefront's
  uint32_t marks;
  // (the wavefronts are done with the digits that lay there)
  __device__ __forceinline__ void fill(const LmHeadArgs& a, const HeadShare& sh, float* lds, uint32_t marks_) {
    float* const mine = lds + sh.wave * PLACES * kSbElems;
    at = mine;
    marks = marks_;
    int place = 0;
#pragma unroll 1
    for (uint32_t m = marks; m != 0 && place < PLACES; m &= m - 1, ++place)
      reinterpret_cast<float4*>(mine + place * kSbElems)[sh.lane] =
          reinterpret_cast<const float4*>(a.x + (size_t)(a.t0 + __builtin_ctz(m)) * a.K + sh.wave * kSbElems)[sh.lane];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // which place a token has (PLACES or more: none)
  __device__ __forceinline__ int place(int t) const { return marks >> t & 1 ? __builtin_popcount(marks & ((1u << t) - 1)) : PLACES; }
};

// ------------------------------------------------------------------------------------------------
// bf16.  A fp32 activation is the sum of three bf16 numbers, each the leading eight bits of what is left, so every product
// is exact in the matrix instruction's fp32.  The first pieces' sums of 32 columns are added in pairs, and so are the
// wavefronts'; the second and third pieces, 2^-8 of the first, are one chain.  The sums round less often than the lanes'
// multiplications and additions they replace (against float64, 2048 columns: root mean square of the error over
// that of the outputs 0.76e-7, the lanes 1.24e-7).
// A lane's pieces of an activation reach down to bf16's (fp32's) smallest exponent: columns whose largest is below 2^-30
// are multiplied by 2^90 first, and those with a value that would lose its last piece all the same are marked by a NaN
// scale.  A sum of 256 columns that is not finite, by a mark, an infinity or a NaN, is made again by fp32 multiply-adds, so
// that it is what those make of it (one such token, 1 / 3 / 8 / 16 tokens 195 / 198 / 211 / 226 us; the whole row again by a lane per logit
// 1350 to 1380).
// ------------------------------------------------------------------------------------------------
constexpr int kBf16Slot = kTileRows * 512;

// 256 columns by multiply-adds out of a lane's weights and its token's activations `x` (uniform); the four quarters' sums are added
// in pairs.  Scalar loads: vector ones would be waited for behind the rows that are on their way.
__device__ __forceinline__ float bf16_plain(const float* x, const v8b_t (&w)[8], int g) {
  typedef const __attribute__((address_space(4))) float* scalars_t;
  scalars_t at = (scalars_t)(uintptr_t)x;
  float u[4] = {0, 0, 0, 0};  // by quarter; the lane's own is used
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    v4u_t own = __builtin_bit_cast(v4u_t, w[j]);
    // (step by step: all weights as fp32, and all loads, at once were 140 spilled registers)
    asm volatile("" : "+s"(at), "+v"(own), "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]));
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float f = __builtin_bit_cast(float, i & 1 ? own[i / 2] & 0xffff0000u : own[i / 2] << 16);
#pragma unroll
      for (int q = 0; q < 4; ++q) u[q] = __builtin_fmaf(f, at[32 * j + 8 * q + i], u[q]);
    }
  }
  float v = g & 2 ? (g & 1 ? u[3] : u[2]) : (g & 1 ? u[1] : u[0]);
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

__global__ void __launch_bounds__(512, 2) k_head_tiles_bf16(LmHeadArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t s_tiles[];
  const HeadShare sh(a.vocab);
  const uint32_t row_bytes = (uint32_t)a.K * 2;
  uint8_t* const slot = s_tiles + (size_t)sh.wave * kBf16Slot;
  const uint32_t slot_lds = lds_address(slot);
  float* const red = reinterpret_cast<float*>(s_tiles + (size_t)sh.waves * kBf16Slot);
  constexpr int kRed = 16 * kTileRows;

  // Two rows' 512 bytes per DMA instruction.  The 16-byte pieces of a row lie in LDS permuted by the row (piece p at
  // p ^ (row mod 16)), so that the sixteen rows of a read lie in different banks.
  auto request = [&](int row0, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 8 * s; i < 8 * s + 8; ++i) {
      const int row = 2 * i + (sh.lane >> 5), piece = (sh.lane & 31) ^ (row & 15);
      const int at = min(row0 + 2 * i, a.vocab - 1);  // (uniform; the row after it only where there is one)
      const uint32_t next = row0 + 2 * i + 1 < a.vocab ? row_bytes : 0;
      lds_dma_16(a.w + (size_t)at * row_bytes + sh.wave * 512, (uint32_t)(sh.lane >> 5) * next + piece * 16, slot_lds + i * 1024);
    }
  };

  // ---- the pieces of token r's columns 32 j + 8 g .. + 7
  v8b_t p[3][8];
  float down;
  {
    const bool in = sh.r < a.nt;
    const float4* src = reinterpret_cast<const float4*>(a.x + (size_t)(a.t0 + min(sh.r, a.nt - 1)) * a.K + sh.wave * 256 + 8 * sh.g);
    float4 f[8][2];
    uint32_t mag = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        f[j][i] = src[8 * j + i];
        const float v[4] = {f[j][i].x, f[j][i].y, f[j][i].z, f[j][i].w};
#pragma unroll
        for (int c = 0; c < 4; ++c) mag = max(mag, __builtin_bit_cast(uint32_t, v[c]) & 0x7fffffffu);
      }
    wait_loads();  // (the compiler's loads are done, and the pieces are made while the first tile is on its way)
    request(sh.row_lo, 0);
    request(sh.row_lo, 1);
    mag = max(mag, (uint32_t)__shfl_xor((int)mag, 16, 64));
    mag = max(mag, (uint32_t)__shfl_xor((int)mag, 32, 64));
    const bool small = mag < 0x30800000u;  // (2^-30)
    const float up = small ? 0x1p90f : 1.0f;
    bool lost = false;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      uint32_t q[3][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4 v = f[j][i >> 1];
        uint32_t b[2][3];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const float x = (in ? (i & 1 ? (c ? v.w : v.z) : (c ? v.y : v.x)) : 0.0f) * up;
          lost = lost || (x != 0.0f && __builtin_fabsf(x) < 0x1p-100f);
          b[c][0] = __builtin_bit_cast(uint32_t, x);
          const float rest = x - __builtin_bit_cast(float, b[c][0] & 0xffff0000u);
          b[c][1] = __builtin_bit_cast(uint32_t, rest);
          b[c][2] = __builtin_bit_cast(uint32_t, rest - __builtin_bit_cast(float, b[c][1] & 0xffff0000u));
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) q[k][i] = __builtin_amdgcn_perm(b[1][k], b[0][k], 0x07060302u);
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) p[k][j] = __builtin_bit_cast(v8b_t, v4u_t{q[k][0], q[k][1], q[k][2], q[k][3]});
    }
    lost = (__builtin_amdgcn_ballot_w64(lost) >> sh.r & 0x0001000100010001ull) != 0;
    down = lost ? __builtin_nanf("") : small ? 0x1p-90f : 1.0f;
  }
  float scale[4];  // of tokens 4 g + i, whose sums the lane's result registers are
#pragma unroll
  for (int i = 0; i < 4; ++i) scale[i] = __shfl(down, 4 * sh.g + i, 64);
  auto reduce = [&](int n) __attribute__((always_inline)) {
    head_reduce<1, 16>(red + (size_t)(n & 1) * sh.waves * kRed, sh, a, sh.row_lo + kTileRows * n);
  };

#pragma unroll 1
  for (int n = 0; n < sh.tiles; ++n) {
    const int row0 = sh.row_lo + kTileRows * n;
    float* const buf = red + (size_t)(n & 1) * sh.waves * kRed;
    const bool last = n + 1 == sh.tiles;
    float* const mine = buf + sh.wave * kRed;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      wait_tile<8>(last);
      v8b_t w[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) w[j] = *reinterpret_cast<const v8b_t*>(slot + (16 * s + sh.r) * 512 + (((4 * j + sh.g) ^ sh.r) * 16));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (s == 1 && n > 0) reduce(n - 1);
      if (!last) request(row0 + kTileRows, s);
      const v4f_t zero = {0, 0, 0, 0};
      v4f_t hi[8], lo = zero;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[2][j], w[j], lo, 0, 0, 0);
        hi[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[0][j], w[j], zero, 0, 0, 0);
        lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[1][j], w[j], lo, 0, 0, 0);
      }
      float out[4];
      bool finite = true;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float sum = ((hi[0][i] + hi[1][i]) + (hi[2][i] + hi[3][i])) + ((hi[4][i] + hi[5][i]) + (hi[6][i] + hi[7][i]));
        out[i] = (sum + lo[i]) * scale[i];
        finite = finite && __builtin_isfinite(out[i]);
      }
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(!finite && row0 + 16 * s + sh.r < sh.row_hi) != 0, 0)) {
        uint32_t m = 0;  // tokens with a sum that is not finite
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint64_t lanes = __builtin_amdgcn_ballot_w64(!__builtin_isfinite(out[i]));
#pragma unroll
          for (int g = 0; g < 4; ++g) m |= (uint32_t)((lanes >> (16 * g) & 0xffff) != 0) << (4 * g + i);
        }
#pragma unroll 1
        for (m &= (1u << a.nt) - 1; m != 0; m &= m - 1) {
          const int t = __builtin_ctz(m);
          const float plain = bf16_plain(a.x + (size_t)(a.t0 + t) * a.K + sh.wave * 256, w, sh.g);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (t == 4 * sh.g + i && !__builtin_isfinite(out[i])) out[i] = plain;
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) mine[(4 * sh.g + i) * kTileRows + 16 * s + sh.r] = out[i];
    }
    __syncthreads();
  }
  reduce(sh.tiles - 1);
}

// ------------------------------------------------------------------------------------------------
// Q8_0.  An activation is a 48-bit number relative to the largest of its superblock (digits.h) written as four signed
// base-4096 digits.  Codes and digits are fp16 integers (digits up to 2048, which fp16 holds), a block's digit sums at most
// 32 * 128 * 2048 = 2^23: exact in the matrix instruction's fp32.  What is left per (row, block, token) is four fused
// multiply-adds by the block's scale into sums of their own, joined once per superblock; six base-256 digits on the int8
// instruction leave nine instructions to join and scale.  The operand's rows are four digits of four tokens.  Against
// float64, 2048 columns: root mean square of the error over that of the outputs 0.76e-7, six digits 0.79e-7.
// ------------------------------------------------------------------------------------------------
using Q8Dma = SliceDma<kQ8_0>;
constexpr int kQ8Digits = 8192;  // LDS of four tokens' digits of a superblock, as the instruction takes them: [block][lane][16]

// Places for marked tokens' activations behind the sums of 4 nq tokens, where the digits were.
template <int NQ>
constexpr int kQ8Places = 8 - NQ;
static_assert(2 * 4 * 4 * kTileRows * 4 + kQ8Places<4> * kSbElems * 4 <= kQ8Digits, "the sums and the places lie where the digits did");

// For which of four tokens a lane of quarter g, token g's, holds a NaN.
__device__ __forceinline__ uint32_t marked_tokens(float v) {
  const uint64_t lanes = __builtin_amdgcn_ballot_w64(v != v);
  uint32_t m = 0;
#pragma unroll
  for (int g = 0; g < 4; ++g) m |= (uint32_t)((lanes >> (16 * g) & 0xffff) != 0) << g;
  return m;
}

// A superblock by multiply-adds out of a lane's codes and its token's activations `x` (the superblock's, plus 8 g): eight columns of every
// block; the four quarters' sums are added in pairs.
__device__ __forceinline__ float q8_plain(const float* x, const uint32_t (&code)[8][2], const uint32_t (&d)[4]) {
  float v = 0.0f;
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const float ws = f16_bits_to_f32(d[b / 2] >> (16 * (b & 1)) & 0xffffu);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float4 f = *reinterpret_cast<const float4*>(x + 32 * b + 4 * i);
      v = __builtin_fmaf(f.x, ws * (float)(int8_t)code[b][i], v);
      v = __builtin_fmaf(f.y, ws * (float)(int8_t)(code[b][i] >> 8), v);
      v = __builtin_fmaf(f.z, ws * (float)(int8_t)(code[b][i] >> 16), v);
      v = __builtin_fmaf(f.w, ws * (float)(int8_t)(code[b][i] >> 24), v);
    }
  }
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

// The lane's activations of tokens t0 + half and t0 + 2 + half: eight columns each.
__device__ __forceinline__ void q8_load(const LmHeadArgs& a, const HeadShare& sh, int t0, float4 (&f)[2][2]) {
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int t = t0 + 2 * it + (sh.lane >> 5);
    const float4* src = reinterpret_cast<const float4*>(a.x + (size_t)(a.t0 + min(t, a.nt - 1)) * a.K + sh.wave * kSbElems + 8 * (sh.lane & 31));
    f[it][0] = src[0];
    f[it][1] = src[1];
  }
}
// Digits of the four tokens from t0 on: operands to `op`, the scale of token t0 + g returned.
__device__ __forceinline__ float q8_digits(const LmHeadArgs& a, const HeadShare& sh, int t0, const float4 (&f)[2][2], uint8_t* lds, v8h_t (&op)[8]) {
  const int octet = sh.lane & 31, b = octet >> 2, q = octet & 3;
  float own[2];
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int t = 2 * it + (sh.lane >> 5);
    const bool in = t0 + t < a.nt;
    const float4 f0 = f[it][0], f1 = f[it][1];
    float v[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
    uint32_t mag = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[i] = in ? v[i] : 0.0f;
      mag = max(mag, __builtin_bit_cast(uint32_t, v[i]) & 0x7fffffffu);
    }
    mag = row16_max(mag);
    mag = max(mag, (uint32_t)__shfl_xor((int)mag, 16, 64));
    const int e = digit_exponent(mag), shift = digit_shift(e);
    bool inexact = false;
    v4u_t plane[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float d[2][4];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        float rest = __builtin_ldexpf(v[2 * i + c], shift);
        inexact = inexact || __builtin_rintf(rest) != rest;
        d[c][0] = __builtin_rintf(rest * 0x1p-36f);
        rest = __builtin_fmaf(d[c][0], -0x1p36f, rest);
        d[c][1] = __builtin_rintf(rest * 0x1p-24f);
        rest = __builtin_fmaf(d[c][1], -0x1p24f, rest);
        d[c][2] = __builtin_rintf(rest * 0x1p-12f);
        d[c][3] = __builtin_fmaf(d[c][2], -0x1p12f, rest);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) plane[k][i] = __builtin_bit_cast(uint32_t, v2h_t{(_Float16)d[0][k], (_Float16)d[1][k]});
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) *reinterpret_cast<v4u_t*>(lds + b * 1024 + (q * 16 + 4 * t + k) * 16) = plane[k];
    const uint64_t any = __builtin_amdgcn_ballot_w64(inexact);
    own[it] = digit_scale(mag, e, (uint32_t)(sh.lane >> 5 ? any >> 32 : any) != 0);
  }
  const float s0 = __shfl(own[0], 32 * (sh.g & 1), 64), s1 = __shfl(own[1], 32 * (sh.g & 1), 64);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int j = 0; j < 8; ++j) op[j] = *reinterpret_cast<const v8h_t*>(lds + j * 1024 + sh.lane * 16);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  return sh.g >> 1 ? s1 : s0;
}

template <int NQ>
__global__ void __launch_bounds__(512, 2) k_head_tiles_q8(LmHeadArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t s_tiles[];
  const HeadShare sh(a.vocab);
  const int sb = sh.wave;
  const uint32_t row_bytes = (uint32_t)sh.waves * SbRaw<kQ8_0>::kBytes;
  uint8_t* const slot = s_tiles + (size_t)sh.wave * Q8Dma::kSlotBytes;
  const uint32_t slot_lds = lds_address(slot);
  uint8_t* const rest = s_tiles + (size_t)sh.waves * Q8Dma::kSlotBytes;  // the digits' places at first, then the sums'
  float* const red = reinterpret_cast<float*>(rest);
  constexpr int kRed = 4 * NQ * kTileRows;

  Q8Dma dma;
  dma.init(row_bytes, 16);
  auto request = [&](int row0, int s) __attribute__((always_inline)) {
    dma.request(a.w, a.w_bytes, (size_t)min(row0 + 16 * s, a.vocab - 1) * row_bytes, sb, slot_lds + s * Q8Dma::kRunBytes);
  };
  v8h_t op[NQ][8];
  float e[NQ];
  float4 f[NQ][2][2];
#pragma unroll
  for (int q = 0; q < NQ; ++q) q8_load(a, sh, 4 * q, f[q]);
  wait_loads();  // (the compiler's loads are done, and the digits are made while the first tile is on its way)
  request(sh.row_lo, 0);
  request(sh.row_lo, 1);
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    e[q] = 16.0f * q8_digits(a, sh, 4 * q, f[q], rest + (size_t)sh.wave * kQ8Digits, op[q]);  // (2^36 of the digits, 2^32 of the scale)
  }
  __syncthreads();
  MarkedRows<kQ8Places<NQ>> kept;
  {
    uint32_t m = 0;
#pragma unroll
    for (int q = 0; q < NQ; ++q) m |= marked_tokens(e[q]) << (4 * q);
    kept.fill(a, sh, red + 2 * sh.waves * kRed, m & ((1u << a.nt) - 1));
  }
  auto reduce = [&](int n) __attribute__((always_inline)) {
    head_reduce<1, 4 * NQ>(red + (size_t)(n & 1) * sh.waves * kRed, sh, a, sh.row_lo + kTileRows * n);
  };

#pragma unroll 1
  for (int n = 0; n < sh.tiles; ++n) {
    const int row0 = sh.row_lo + kTileRows * n;
    float* const buf = red + (size_t)(n & 1) * sh.waves * kRed;
    const bool last = n + 1 == sh.tiles;
    float* const mine = buf + sh.wave * kRed;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      wait_tile<Q8Dma::kInstr>(last);
      // The lane's eight codes of every block: on a word in odd blocks, half a word past one in even ones.
      uint32_t code[8][2], d[4];  // (two blocks' scales to a register)
      const uint8_t* p = slot + s * Q8Dma::kRunBytes + sh.r * SbRaw<kQ8_0>::kBytes;
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const uint8_t* at = p + kQ8Bytes * b + 8 * sh.g;
        const uint32_t scale = *reinterpret_cast<const uint16_t*>(p + kQ8Bytes * b);
        d[b / 2] = b & 1 ? d[b / 2] | scale << 16 : scale;
        if (b & 1) {
          code[b][0] = lds_word(at + 2);
          code[b][1] = lds_word(at + 6);
        } else {
          const uint32_t w0 = lds_word(at), w1 = lds_word(at + 4), w2 = lds_word(at + 8);
          code[b][0] = __builtin_amdgcn_alignbit(w1, w0, 16);
          code[b][1] = __builtin_amdgcn_alignbit(w2, w1, 16);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (s == 1 && n > 0) reduce(n - 1);
      if (!last) request(row0 + kTileRows, s);
      v4f_t acc[NQ];
#pragma unroll
      for (int q = 0; q < NQ; ++q) acc[q] = v4f_t{0, 0, 0, 0};
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        // 1024 + 128 + code as halves, less 1152
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint32_t u = code[b][i] ^ 0x80808080u;
          h[2 * i] = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
          h[2 * i + 1] = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
        }
        v8h_t w;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const v2h_t v = __builtin_bit_cast(v2h_t, h[i]) - v2h_t{(_Float16)1152.0f, (_Float16)1152.0f};
          w[2 * i] = v[0];
          w[2 * i + 1] = v[1];
        }
        const float ws = f16_bits_to_f32(d[b / 2] >> (16 * (b & 1)));
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const v4f_t sums = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[q][b], w, v4f_t{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
          for (int k = 0; k < 4; ++k) acc[q][k] = __builtin_fmaf(ws, sums[k], acc[q][k]);
        }
      }
      float out[NQ];
      bool nan = false;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        out[q] = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(acc[q][3], 0x1p-12f, acc[q][2]), 0x1p-12f, acc[q][1]), 0x1p-12f, acc[q][0]) * e[q];
        nan |= out[q] != out[q];
      }
      // (a block's scale that is not finite makes NaNs, too)
      uint32_t m = 0;
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(nan && row0 + 16 * s + sh.r < sh.row_hi) != 0, 0)) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) m |= marked_tokens(out[q]) << (4 * q);
      }
      for (; __builtin_expect(m != 0, 0); m &= m - 1) {
        const int t = __builtin_ctz(m);
        if (t >= a.nt) break;
        const int place = kept.place(t);
        const float plain = place < kQ8Places<NQ> ? q8_plain(kept.at + place * kSbElems + 8 * sh.g, code, d)
                                                  : q8_plain(a.x + (size_t)(a.t0 + t) * a.K + sb * kSbElems + 8 * sh.g, code, d);
#pragma unroll
        for (int q = 0; q < NQ; ++q)
          if (t == 4 * q + sh.g && out[q] != out[q]) out[q] = plain;
      }
#pragma unroll
      for (int q = 0; q < NQ; ++q) mine[(4 * q + sh.g) * kTileRows + 16 * s + sh.r] = out[q];
    }
    __syncthreads();
  }
  reduce(sh.tiles - 1);
}

// ------------------------------------------------------------------------------------------------
// Q6_K, from five tokens on.  The sums of half a superblock are integers (digits.h): codes times their group's scale times
// digits.  Here the scale goes to the code first, once for all tokens: the product has fifteen bits and is two int8 planes,
// high and low, so the matrix instruction carries a digit's sum through the whole half superblock and what is left per
// (row, half, token) is one shift and addition per digit and the join, where a scale per group left six multiply-adds for
// every sixteen elements.  That costs ten instructions per four weights to make both planes and twice the matrix
// instructions, which are full here: the rows of the operand are four digits of four tokens (twice), then the two low
// digits of all eight.  The same integers, joined the same way: the bits of k_lm_head_quant, which up to four tokens is
// the faster one.
// ------------------------------------------------------------------------------------------------
using Q6Dma = SliceDma<kQ6K>;
constexpr int kQ6Digits = 8 * kSbDigitBytes;  // LDS of eight tokens' digits of a superblock
template <int NO>
constexpr int kQ6Places = 12 - 4 * NO;  // (kQ8Places)
static_assert(2 * 2 * 8 * 2 * kTileRows * 4 + kQ6Places<2> * kSbElems * 4 <= kQ6Digits, "the sums and the places lie where the digits did");

template <int NO>
__global__ void __launch_bounds__(512, 2) k_head_tiles_q6(LmHeadArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t s_tiles[];
  const HeadShare sh(a.vocab);
  const int sb = sh.wave, r = sh.r, g = sh.g;
  const uint32_t row_bytes = (uint32_t)sh.waves * kQ6KBytes;
  uint8_t* const slot = s_tiles + (size_t)sh.wave * Q6Dma::kSlotBytes;
  const uint32_t slot_lds = lds_address(slot);
  uint8_t* const rest = s_tiles + (size_t)sh.waves * Q6Dma::kSlotBytes;  // the digits' places at first, then the sums'
  float* const red = reinterpret_cast<float*>(rest);
  constexpr int kRed = 2 * 8 * NO * kTileRows;

  Q6Dma dma;
  dma.init(row_bytes, 16);
  auto run_off = [&](int row0, int u) __attribute__((always_inline)) { return (size_t)min(row0 + 16 * u, a.vocab - 1) * row_bytes; };
  auto request = [&](int row0, int s) __attribute__((always_inline)) {
    dma.request(a.w, a.w_bytes, run_off(row0, s), sb, slot_lds + s * Q6Dma::kRunBytes);
  };
  v4i_t op[NO][4][3];  // [step of 64 elements: half, step][digits 0..3 of tokens 0..3, of tokens 4..7, digits 4 and 5]
  float e[NO][2];      // scales of tokens g and 4 + g
  uint32_t marks = 0;  // tokens whose superblock is marked
  float4 f[8 * NO];
#pragma unroll
  for (int t = 0; t < 8 * NO; ++t)
    f[t] = reinterpret_cast<const float4*>(a.x + (size_t)(a.t0 + min(t, a.nt - 1)) * a.K + sb * kSbElems)[sh.lane];
  wait_loads();  // (the compiler's loads are done, and the digits are made while the first tile is on its way)
  request(sh.row_lo, 0);
  request(sh.row_lo, 1);
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    uint8_t* const lds = rest + (size_t)sh.wave * kQ6Digits;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const bool in = 8 * o + t < a.nt;
      const float v[4] = {in ? f[8 * o + t].x : 0.0f, in ? f[8 * o + t].y : 0.0f, in ? f[8 * o + t].z : 0.0f, in ? f[8 * o + t].w : 0.0f};
      const float scale = digitize_quads(v, lds + t * kSbDigitBytes);
      if ((t & 3) == 0 || g == (t & 3)) e[o][t >> 2] = scale;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    planes_operands(lds, kSbDigitBytes, op[o]);
    marks |= (marked_tokens(e[o][0]) | marked_tokens(e[o][1]) << 4) << (8 * o);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  __syncthreads();
  MarkedRows<kQ6Places<NO>> kept;
  kept.fill(a, sh, red + 2 * sh.waves * kRed, marks);
  auto reduce = [&](int n) __attribute__((always_inline)) {
    head_reduce<2, 8 * NO>(red + (size_t)(n & 1) * sh.waves * kRed, sh, a, sh.row_lo + kTileRows * n);
  };
  const uint32_t shift[2] = {4u - 2u * (uint32_t)(g >> 1), 2u * (uint32_t)(g >> 1)};

#pragma unroll 1
  for (int n = 0; n < sh.tiles; ++n) {
    const int row0 = sh.row_lo + kTileRows * n;
    float* const buf = red + (size_t)(n & 1) * sh.waves * kRed;
    const bool last = n + 1 == sh.tiles;
    float* const mine = buf + sh.wave * kRed;
    SbRaw<kQ6K> raw;  // of a marked superblock, a lane per row and half: lane 32 h + 16 s + r
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      wait_tile<Q6Dma::kInstr>(last);
      if (sb == sh.waves - 1 && row0 + kTileRows >= a.vocab) {  // (the tensor's last bytes, which no whole piece held)
        const int live = a.vocab - (row0 + 16 * s);
        if (live >= 1 && live <= 16) dma.patch_tail(a.w, run_off(row0, s), live, sb, slot + s * Q6Dma::kRunBytes);
      }
      Q6Quarter w;
      w.read(slot + s * Q6Dma::kRunBytes + r * (Q6Dma::kP * 16), (uint32_t)(sb & 1) * 2, g);  // (rows are whole words)
      if (__builtin_expect(marks != 0, 0) && (s == 0 || (sh.lane & 16)))
        sb_read_slot(slot + s * Q6Dma::kRunBytes + r * (Q6Dma::kP * 16) + (sb & 1) * 2, sh.lane >> 5, raw);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (s == 1 && n > 0) reduce(n - 1);
      if (!last) request(row0 + kTileRows, s);
      float out[2][NO][2];
      const float quarter = f16_bits_to_f32(w.d) * 0.25f;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        v4i_t hi[2], lo[2];
        w.planes(h, shift, hi, lo);
#pragma unroll
        for (int o = 0; o < NO; ++o) {
          const float eo[2] = {quarter * e[o][0], quarter * e[o][1]};
          planes_dot(op[o][2 * h], op[o][2 * h + 1], hi, lo, eo, out[h][o]);
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int o = 0; o < NO; ++o)
#pragma unroll
          for (int t = 0; t < 2; ++t) mine[(h * 8 * NO + 8 * o + 4 * t + g) * kTileRows + 16 * s + r] = out[h][o][t];
    }
    for (uint32_t m = marks; __builtin_expect(m != 0, 0); m &= m - 1) {  // both sets' rows in place of the NaNs
      const int t = __builtin_ctz(m), place = kept.place(t);
      float own[8];
      if (place < kQ6Places<NO>) half_own(kept.at + place * kSbElems, sh.lane >> 5, sh.lane, own);
      else half_own(a.x + (size_t)(a.t0 + t) * a.K + sb * kSbElems, sh.lane >> 5, sh.lane, own);
      opaque(raw);
      mine[((sh.lane >> 5) * 8 * NO + t) * kTileRows + (sh.lane & 31)] = half_fp32_all<kQ6K>(raw, own, HalfOrder{});
    }
    __syncthreads();
  }
  reduce(sh.tiles - 1);
}

// ------------------------------------------------------------------ host side
typedef void (*HeadKernel)(LmHeadArgs);

static int head_tiles_limit(HeadKernel kernel, size_t smem) {
  XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
  return XABE_OK;
}
static size_t head_bf16_lds(size_t waves) { return waves * (kBf16Slot + 2 * 16 * kTileRows * sizeof(float)); }
static size_t head_q8_lds(size_t waves, size_t nq) {
  return waves * (Q8Dma::kSlotBytes + std::max<size_t>(kQ8Digits, 2 * 4 * nq * kTileRows * sizeof(float)));
}
static size_t head_q6_lds(size_t waves, size_t no) {
  return waves * (Q6Dma::kSlotBytes + std::max<size_t>(kQ6Digits, 2 * 2 * 8 * no * kTileRows * sizeof(float)));
}
static const HeadKernel kHeadQ8[4] = {k_head_tiles_q8<1>, k_head_tiles_q8<2>, k_head_tiles_q8<3>, k_head_tiles_q8<4>};
static const HeadKernel kHeadQ6[2] = {k_head_tiles_q6<1>, k_head_tiles_q6<2>};

// at handle creation, not on the launch path (launches are captured into graphs)
int head_tiles_configure() {
  XABE_TRY(head_tiles_limit(k_head_tiles_bf16, head_bf16_lds(8)));
  for (size_t i = 0; i < 4; ++i) XABE_TRY(head_tiles_limit(kHeadQ8[i], head_q8_lds(8, i + 1)));
  for (size_t i = 0; i < 2; ++i) XABE_TRY(head_tiles_limit(kHeadQ6[i], head_q6_lds(8, i + 1)));
  return XABE_OK;
}

// As many workgroups as are resident at once (eight wavefronts to a compute unit), and no more than there are tiles.
static int head_tiles_go(HeadKernel kernel, hipStream_t s, int num_cus, size_t smem, const LmHeadArgs& a) {
  const int waves = a.K / kSbElems, tiles = (a.vocab + kTileRows - 1) / kTileRows;
  hipLaunchKernelGGL(kernel, dim3((unsigned)std::min(tiles, num_cus * (8 / waves))), dim3((unsigned)(64 * waves)), smem, s, a);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}
int launch_head_tiles_bf16(hipStream_t s, int num_cus, const LmHeadArgs& a) {
  return head_tiles_go(k_head_tiles_bf16, s, num_cus, head_bf16_lds(a.K / kSbElems), a);
}
int launch_head_tiles_q8(hipStream_t s, int num_cus, const LmHeadArgs& a) {
  const size_t nq = ((size_t)a.nt + 3) / 4;
  return head_tiles_go(kHeadQ8[nq - 1], s, num_cus, head_q8_lds(a.K / kSbElems, nq), a);
}
int launch_head_tiles_q6k(hipStream_t s, int num_cus, const LmHeadArgs& a) {
  const size_t no = ((size_t)a.nt + 7) / 8;
  return head_tiles_go(kHeadQ6[no - 1], s, num_cus, head_q6_lds(a.K / kSbElems, no), a);
}

}  // namespace xabe
