// Q6_K codes times their group's scale as two int8 planes, and the contraction on them (lm_head_tiles.hip,
// digit_columns.hip): half a superblock's digit sums without a scale in between.
//
// On v_mfma_i32_16x16x64_i8 a lane holds sixteen codes of row lane & 15 per step of 64 elements, those of quarter
// g = lane >> 4.  A half superblock is two steps: the groups of quarter g are the low nibbles of ql[64 h + 16 g ..] (step 0) and
// the high ones (step 1), with two bits each of qh[32 h + 16 (g & 1) ..]; their scale is number 8 h + 4 step + g.  The other
// operand's sixteen rows are digits: four of four tokens each (twice), then the two low digits of all eight, so that the
// lane's result registers are those of tokens g and 4 + g.
#pragma once

#include "digits.h"

namespace xabe {

typedef uint16_t v2s_t __attribute__((ext_vector_type(2)));

// One superblock of a set of sixteen rows as a lane holds it.
struct Q6Quarter {
  v4u_t ql[2], qh[2];  // by half
  int sc[4];           // 2 h + step
  uint32_t d;

  // `b`: the row's window in LDS, on a 16-byte boundary, in which the superblock starts `mis` (0 or 2) bytes in
  __device__ __forceinline__ void read(const uint8_t* b, uint32_t mis, int g) {
    b = static_cast<const uint8_t*>(__builtin_assume_aligned(b, 16));
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const v4u_t l = *reinterpret_cast<const v4u_t*>(b + 64 * h + 16 * g), m = *reinterpret_cast<const v4u_t*>(b + 128 + 32 * h + 16 * (g & 1));
      const uint32_t l4 = lds_word(b + 64 * h + 16 * g + 16), m4 = lds_word(b + 128 + 32 * h + 16 * (g & 1) + 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ql[h][i] = __builtin_amdgcn_alignbit(i < 3 ? l[i + 1] : l4, l[i], 8 * mis);
        qh[h][i] = __builtin_amdgcn_alignbit(i < 3 ? m[i + 1] : m4, m[i], 8 * mis);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) sc[2 * h + j] = *reinterpret_cast<const int8_t*>(b + mis + 192 + 8 * h + 4 * j + g);
    }
    d = *reinterpret_cast<const uint16_t*>(b + mis + 208);
  }

  // Both planes of half h, by step.  `shift`: how far the two high bits of the lane's groups are from bits 4 and 5, up in
  // step 0 and down in step 1.  A product is (code - 32) times four times the scale, fifteen bits: 128 more are added, the
  // high byte is the high plane, the low byte with its top bit flipped the low one.
  __device__ __forceinline__ void planes(int h, const uint32_t (&shift)[2], v4i_t (&hi)[2], v4i_t (&lo)[2]) const {
#pragma unroll
    for (int step = 0; step < 2; ++step) {
      const uint16_t four = (uint16_t)(sc[2 * h + step] << 2);
      const v2s_t scale = {four, four}, add = (v2s_t){128, 128} - (v2s_t)(scale << 5);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // (five and six instructions to the codes in halves, spelled out because the compiler makes seven and eight)
        const uint32_t l = step == 0 ? ql[h][i] : ql[h][i] >> 4, m = (step == 0 ? qh[h][i] << shift[0] : qh[h][i] >> shift[1]) & 0x30303030u;
        const uint32_t t = __builtin_amdgcn_bitop3_b32(l, m, 0x0f0f0f0fu, 0xEC);  // (l & k) | m
        const v2s_t even = __builtin_bit_cast(v2s_t, t & 0x00ff00ffu), odd = __builtin_bit_cast(v2s_t, __builtin_amdgcn_perm(0u, t, 0x0c030c01u));
        const uint32_t pe = __builtin_bit_cast(uint32_t, (v2s_t)(even * scale + add)), po = __builtin_bit_cast(uint32_t, (v2s_t)(odd * scale + add));
        hi[step][i] = (int)__builtin_amdgcn_perm(po, pe, 0x07030501u);
        lo[step][i] = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
      }
    }
  }
};

// Half a superblock of the lane's row against tokens g and 4 + g: `a0`, `a1` the operands of its two steps; `e`: a quarter of d
// times the tokens' scales.  The same integers as sb_dot's, joined the same way.
__device__ __forceinline__ void planes_dot(const v4i_t (&a0)[3], const v4i_t (&a1)[3], const v4i_t (&hi)[2], const v4i_t (&lo)[2],
                                           const float (&e)[2], float (&out)[2]) {
  const v4i_t zero = {0, 0, 0, 0};
  v4i_t H[3], L[3];
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    H[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0[f], hi[0], zero, 0, 0, 0);
    L[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0[f], lo[0], zero, 0, 0, 0);
  }
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    H[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1[f], hi[1], H[f], 0, 0, 0);
    L[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1[f], lo[1], L[f], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    int sum[6];
#pragma unroll
    for (int k = 0; k < 4; ++k) sum[k] = (H[t][k] << 8) + L[t][k];
#pragma unroll
    for (int k = 0; k < 2; ++k) sum[4 + k] = (H[2][2 * t + k] << 8) + L[2][2 * t + k];
    out[t] = join_sums(sum) * e[t];
  }
}

// The operands of eight tokens' digits of a superblock, `stride` bytes apart in LDS, as [2 half + step].
__device__ __forceinline__ void planes_operands(const uint8_t* digits, int stride, v4i_t (&op)[4][3]) {
  const int lane = (int)__lane_id(), g = lane >> 4, t = (lane & 15) >> 2, i = lane & 3;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint8_t* group = digits + (4 * (2 * (j & 1) + (g >> 1)) + 2 * (j >> 1) + (g & 1)) * kGroupBytes;
    op[j][0] = *reinterpret_cast<const v4i_t*>(group + t * stride + 16 * i);
    op[j][1] = *reinterpret_cast<const v4i_t*>(group + (4 + t) * stride + 16 * i);
    op[j][2] = *reinterpret_cast<const v4i_t*>(group + (t + 4 * (i >> 1)) * stride + 16 * (4 + (i & 1)));
  }
}

// The same by step out of LDS in which the 16-byte pieces of token t's superblock (96 of them) lie permuted by the token, piece p
// at p ^ 4 (t mod 4): tokens' superblocks are a multiple of the banks' 256 bytes long, and a read of four tokens' digits as they
// lie would take four turns where this takes one.
__device__ __forceinline__ int planes_piece(int lane, int t) { return lane ^ (4 * (t & 3)); }  // which piece to put in place `lane`
struct PlanesOperands {
  uint32_t at[2][3];  // [half][operand]
  __device__ __forceinline__ void init() {
    const int lane = (int)__lane_id(), g = lane >> 4, t = (lane & 15) >> 2, i = lane & 3;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int piece = 6 * (4 * (g >> 1) + 2 * h + (g & 1));
      at[h][0] = (uint32_t)(t * kSbDigitBytes + ((piece + i) ^ (4 * t)) * 16);
      at[h][1] = at[h][0] + 4 * kSbDigitBytes;
      at[h][2] = (uint32_t)((t + 4 * (i >> 1)) * kSbDigitBytes + ((piece + 4 + (i & 1)) ^ (4 * t)) * 16);
    }
  }
  // (a step further is 48 pieces further)
  __device__ __forceinline__ void read(const uint8_t* digits, int half, int step, v4i_t (&op)[3]) const {
#pragma unroll
    for (int f = 0; f < 3; ++f) op[f] = *reinterpret_cast<const v4i_t*>(digits + at[half][f] + step * 768);
  }
};

}  // namespace xabe
