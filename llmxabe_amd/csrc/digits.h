// Quantized rows times fp32 activations on the int8 matrix instruction, at full fp32 precision of the operands: the
// contraction every fp32 regime of this library goes through (decode and dense widths, the LM head).
//
// A Q6_K or Q8_0 weight is an integer code times a scale per 16 or 32 elements.  An activation is written as a 48-bit
// fixed-point number relative to the largest of its superblock of 256 or of its group of 16 (a power-of-two scale that
// puts the largest magnitude between 2^46 and 2^47) and that number as six signed base-256 digits.  Codes and digits are
// int8, so the digit sums of a group of 16 come out of the int8 matrix instruction exact, and what is left for the vector
// ALU depends on how the activations are scaled:
//   whole superblocks (kWhole: rows that exist before the launch).  Q6_K's scales inside a superblock are integers, too:
//     six integer multiply-adds per (row, group, token) carry the sums through the half superblock, eleven instructions
//     join them once at its end.  Q8_0's two groups of a block share a scale: the matrix instruction adds them, and nine
//     instructions per (row, block, token) join the six sums and apply the scale.
//   groups of 16 (kGroups: rows whose groups are written by different workgroups, SwiGLU's).  Ten instructions per (row,
//     group, token): three shift-adds that pair the digit sums, three conversions, two fused multiply-adds that join the
//     pairs, the product of the two scales, the fused multiply-add into the row's sum.
//
// Precision: six digits hold all 24 bits of every value within a factor of 2^22 of its group's (superblock's) largest.
// One they do not hold exactly (a wider range, an infinity or a NaN, magnitudes so near the ends of the exponent range
// that a scale would leave it) is marked by a NaN scale; the NaN reaches the sum of the half superblock, and that half
// superblock is summed again by plain fp32 multiply-adds (half_fp32), lane by lane.  So no operand ever loses a bit,
// infinities keep their signs, and ordinary data (one superblock in ten thousand for normal rows, one half in four
// thousand for SwiGLU's) hardly ever pays for it.  Sums inside a group are exact, where sixteen fp32 multiply-adds
// round sixteen times: measured against float64, 1e-7 of the outputs' peak, the lanes' fp32 sums 1.7e-7.  (Four digits
// held values within 2^6 of the largest only: beside an outlier of 3e4 whose codes are zero the rest of the row was off
// by 7e-6 of its peak.)
// SwiGLU's rows in whole superblocks have such a value in one superblock of four hundred for normal rows, and in one of
// twelve where 0.4 % of them are a thousand times the others.  There up to kRests values are held to whole numbers all the same and
// what is left of them, exactly, is added weight by weight (digit_rests): a multiply-add and a few bytes per row and
// value instead of 256 multiply-adds per row.  More than that, infinities, NaN and magnitudes near the ends are marked as above.
//
// Why this form: one conversion and one multiply-add per weight and token on a 16-lane SIMD (4.9 vector instructions
// per weight in all) bound every batch wider than a few tokens.  Here a weight costs ~1.3 instructions to unpack
// (none for Q8_0, whose codes are the operand as they lie) and at most 10/16 per token.
//
// The matrix instruction's layout: operand A (activations) row m = lane & 31, operand B (weights) column = lane & 31,
// both with the sixteen K positions of half `lane >> 5` in the lane's four registers; the result's column is the
// lane's own, its row 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3) for register i.  Only the half (m >> 2) & 1 of A's row m is
// nonzero: a result register of half h then holds a digit sum over the sixteen elements that half h of the wavefront
// unpacked, so scales and codes meet in one lane, which has sixteen registers per instruction.  One or two tokens take
// eight of them each (register 8 t + d: digit d of token t).  More take two instructions per four tokens: register
// 4 t + d of the first is digit d < 4 of token t; the second multiplies the two low digits, and the groups l = 0 and
// l = 1 share its operand (registers 4 t + 2 l + d - 4): against the codes of either group the registers of that group
// are its sums and the others are not looked at, which saves half of the operand's registers.  (Where the instruction
// adds the two groups up, Q8_0 in whole superblocks, the second group's operand has the two swapped, so that its sums
// land on the first's.)
//
// Order of operations (the numerics contract: a row's value depends on the row and the token only).  A superblock of
// 256 elements is split between the wavefront's halves: half h takes elements 128 h + 32 s + 16 l + [0, 16), s = 0..3,
// l = 0, 1, and sums its eight groups: exactly (Q6_K, whole superblocks), its four blocks in order (Q8_0, whole
// superblocks), or the groups from zero with l outermost.  Superblock sums are added in the order a kernel states.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

#include "device_common.h"

namespace xabe {

typedef int v4i_t __attribute__((ext_vector_type(4)));
typedef int v16i_t __attribute__((ext_vector_type(16)));
typedef uint32_t v4u_t __attribute__((ext_vector_type(4)));

constexpr int kSbElems = 256;
constexpr bool kWhole = true, kGroups = false;  // what an activation scale belongs to

// One superblock of one token: digits as [s][2 h + l][digit, most significant first][16 elements]; scales as floats, one
// (kWhole) or [2 h + l][s] (kGroups).
constexpr int kGroupBytes = 96, kSbDigitBytes = 16 * kGroupBytes, kSbScaleBytes = 64;
constexpr int kZeroBytes = 1280;  // zeros for the lanes without a digit, as far as a group's offset reaches

// The scale of a group (a superblock) whose largest magnitude has the bits `mag`: values times 2^digit_shift(e) are the 48-bit numbers.
// e is the largest's biased exponent, one more where its significand exceeds 0xfefefe, so that the number stays below
// 0x7f7f7f7f7f7f and its top digit below 128.
__device__ __forceinline__ int digit_exponent(uint32_t mag) { return (int)((mag + 0x10101u) >> 23); }
// (outside 48..200 the products of scales could leave fp32's normal range: such groups are marked, with any shift)
__device__ __forceinline__ int digit_shift(int e) { return 173 - min(max(e, 48), 200); }
__device__ __forceinline__ float digit_scale(uint32_t mag, int e, bool inexact) {
  const float scale = __builtin_ldexpf(1.0f, 32 - digit_shift(e));  // (x = the digits' value 2^-32 times this)
  return mag == 0 ? 0.0f : (inexact || e < 48 || e > 200) ? __builtin_nanf("") : scale;
}
// The six digits of x: `high` holds digits 0..3, most significant first, `low` digits 4 and 5 in its lower half.  A
// number plus 0x80 per lower byte, minus it again byte by byte, has signed bytes for digits.
__device__ __forceinline__ void digits_of(float x, int shift, uint32_t& high, uint32_t& low, bool& inexact) {
  const float v = __builtin_ldexpf(x, shift);
  inexact = inexact || __builtin_rintf(v) != v;
  const float top = __builtin_rintf(v * 0x1p-16f);
  const int rest = (int)__builtin_fmaf(top, -65536.0f, v);  // exact, at most 2^15 in magnitude
  const long long y = (((long long)(int)top * 65536 + rest) + 0x8080808080ll) ^ 0x8080808080ll;
  high = (uint32_t)(y >> 16);
  low = (uint32_t)y;
}

__device__ __forceinline__ uint32_t magnitude16(const float (&x)[16]) {
  uint32_t mag = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) mag = max(mag, __builtin_bit_cast(uint32_t, x[i]) & 0x7fffffffu);
  return mag;
}
// The digits of four and of sixteen activations, a word (a 16-byte piece) per digit; `inexact` is set where they do not
// hold one.
__device__ __forceinline__ void digitize4(const float (&x)[4], int shift, uint32_t (&plane)[6], bool& inexact) {
  uint32_t y[4], z[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) digits_of(x[i], shift, y[i], z[i], inexact);
  const uint32_t ab_hi = __builtin_amdgcn_perm(y[1], y[0], 0x07030602u), cd_hi = __builtin_amdgcn_perm(y[3], y[2], 0x07030602u);
  const uint32_t ab_lo = __builtin_amdgcn_perm(y[1], y[0], 0x05010400u), cd_lo = __builtin_amdgcn_perm(y[3], y[2], 0x05010400u);
  const uint32_t ab_z = __builtin_amdgcn_perm(z[1], z[0], 0x05010400u), cd_z = __builtin_amdgcn_perm(z[3], z[2], 0x05010400u);
  plane[0] = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x07060302u);
  plane[1] = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x05040100u);
  plane[2] = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x07060302u);
  plane[3] = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x05040100u);
  plane[4] = __builtin_amdgcn_perm(cd_z, ab_z, 0x07060302u);
  plane[5] = __builtin_amdgcn_perm(cd_z, ab_z, 0x05040100u);
}
__device__ __forceinline__ void digitize16(const float (&x)[16], int shift, v4u_t (&plane)[6], bool& inexact) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float q[4] = {x[4 * w], x[4 * w + 1], x[4 * w + 2], x[4 * w + 3]};
    uint32_t word[6];
    digitize4(q, shift, word, inexact);
#pragma unroll
    for (int p = 0; p < 6; ++p) plane[p][w] = word[p];
  }
}
// The largest of sixteen consecutive lanes' values (a DPP row), and whether any of them says yes.
__device__ __forceinline__ uint32_t row16_max(uint32_t v) {
  int m = (int)v;  // (magnitudes: the sign bit is clear)
  m = max(m, dpp_i<0xB1>(m));
  m = max(m, dpp_i<0x4E>(m));
  m = max(m, dpp_i<0x141>(m));
  return (uint32_t)max(m, dpp_i<0x140>(m));
}
__device__ __forceinline__ bool row16_any(bool b) { return (__builtin_amdgcn_ballot_w64(b) >> (__lane_id() & 48) & 0xffffu) != 0; }

// Group `pos` of a superblock whose sixteen groups sixteen consecutive lanes hold: digits into the superblock's at `base`;
// returns the superblock's scale.
__device__ __forceinline__ int digit_group_offset(int pos);
__device__ __forceinline__ float digitize_superblock(const float (&x)[16], int pos, uint8_t* base) {
  const uint32_t mag = row16_max(magnitude16(x));
  const int e = digit_exponent(mag);
  v4u_t plane[6];
  bool inexact = false;
  digitize16(x, digit_shift(e), plane, inexact);
  uint8_t* d = base + digit_group_offset(pos);
#pragma unroll
  for (int p = 0; p < 6; ++p) reinterpret_cast<v4u_t*>(d)[p] = plane[p];
  return digit_scale(mag, e, row16_any(inexact));
}

// A superblock whose sixty-four quads of elements the wavefront's lanes hold: digits to `base`; returns its scale.  RESTS: where
// at most kRests values are not held exactly, the digits are of whole numbers beside theirs, and the scale is negative (digit_rests).
constexpr int kRests = 8;
template <bool RESTS = false>
__device__ __forceinline__ float digitize_quads(const float (&x)[4], uint8_t* base) {
  const int lane = (int)__lane_id();
  uint32_t mag = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) mag = max(mag, __builtin_bit_cast(uint32_t, x[i]) & 0x7fffffffu);
  mag = (uint32_t)wave_max_i((int)mag);
  const int e = digit_exponent(mag), shift = digit_shift(e);
  uint32_t plane[6];
  bool inexact = false;
  digitize4(x, shift, plane, inexact);
  uint8_t* d = base + digit_group_offset(lane >> 2) + 4 * (lane & 3);
#pragma unroll
  for (int p = 0; p < 6; ++p) *reinterpret_cast<uint32_t*>(d + 16 * p) = plane[p];
  const uint64_t any = __builtin_amdgcn_ballot_w64(inexact);
  if constexpr (RESTS) {
    if (any == 0) return digit_scale(mag, e, false);
    int n = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = __builtin_ldexpf(x[i], shift);
      n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(__builtin_rintf(v) != v));
    }
    return -digit_scale(mag, e, n > kRests);
  }
  return digit_scale(mag, e, any != 0);
}
// What the digits of a superblock with a negative scale leave of its values, the lane's quad: exact, and zero but for a few.
__device__ __forceinline__ void digit_rests(const float (&x)[4], float scale, float (&rest)[4]) {
  const int shift = 159 - (int)(__builtin_bit_cast(uint32_t, scale) >> 23 & 0xffu);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float v = __builtin_ldexpf(x[i], shift), low = __builtin_fmaf(__builtin_rintf(v * 0x1p-16f), -65536.0f, v);  // (digits_of)
    rest[i] = __builtin_ldexpf(low - __builtin_truncf(low), -shift);
  }
}
// Calls add(element, rest) for each, in the order that every kernel adds them in.
template <typename Add>
__device__ __forceinline__ void for_rests(const float (&rest)[4], Add add) {
  float v = rest[0], r1 = rest[1], r2 = rest[2], r3 = rest[3];
#pragma unroll 1
  for (int i = 0; i < 4; ++i, v = r1, r1 = r2, r2 = r3) {
#pragma unroll 1
    for (uint64_t m = __builtin_amdgcn_ballot_w64(v != 0.0f); m; m &= m - 1) {
      const int l = __builtin_ctzll(m);
      add(4 * l + i, lane_bcast(v, l));
    }
  }
}
// Element p's weight out of its superblock's bytes, which lie at sb + off.
__device__ __forceinline__ float q6k_weight(const uint8_t* sb, uint32_t off, int p) {
  const int h = p >> 7, k = p >> 5 & 3, l = p & 31;
  const int low = (sb + (64 * h + 32 * (k & 1) + l))[off] >> (4 * (k >> 1)) & 15, high = (sb + (128 + 32 * h + l))[off] >> (2 * k) & 3;
  const float d = f16_bits_to_f32(*reinterpret_cast<const uint16_t*>(sb + 208 + off));
  return d * (float)(int8_t)(sb + (192 + 8 * h + 2 * k + (l >> 4)))[off] * (float)((low | high << 4) - 32);
}

// The same with the scale of every group, sixteen at `scales`.
__device__ __forceinline__ int scale_group_index(int pos);
__device__ __forceinline__ void digitize_quads_by_group(const float (&x)[4], uint8_t* base, float* scales) {
  const int lane = (int)__lane_id();
  int m = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) m = max(m, (int)(__builtin_bit_cast(uint32_t, x[i]) & 0x7fffffffu));
  m = max(m, dpp_i<0xB1>(m));  // (four lanes hold a group)
  m = max(m, dpp_i<0x4E>(m));
  const int e = digit_exponent((uint32_t)m);
  uint32_t plane[6];
  bool inexact = false;
  digitize4(x, digit_shift(e), plane, inexact);
  uint8_t* d = base + digit_group_offset(lane >> 2) + 4 * (lane & 3);
#pragma unroll
  for (int p = 0; p < 6; ++p) *reinterpret_cast<uint32_t*>(d + 16 * p) = plane[p];
  const bool any = (__builtin_amdgcn_ballot_w64(inexact) >> (lane & 60) & 15) != 0;
  if ((lane & 3) == 0) scales[scale_group_index(lane >> 2)] = digit_scale((uint32_t)m, e, any);
}

// Where group `pos` (elements 16 pos .. 16 pos + 15 of its superblock) lies among the digits and the scales.
__device__ __forceinline__ int digit_group_offset(int pos) {
  const int h = pos >> 3, s = (pos >> 1) & 3, l = pos & 1;
  return (4 * s + 2 * h + l) * kGroupBytes;
}
__device__ __forceinline__ int scale_group_index(int pos) {
  const int h = pos >> 3, s = (pos >> 1) & 3, l = pos & 1;
  return (2 * h + l) * 4 + s;
}

// ---------------------------------------------------------------------------------
// One superblock of 32 rows, as a lane of half h holds it: its row's 128 codes and their scales.
// ---------------------------------------------------------------------------------
template <int QUANT>
struct SbRaw;
template <>
struct SbRaw<kQ6K> {
  v4u_t ql[4], qh[2];  // ql[64 h ..], qh[32 h ..]
  uint2 sc;            // scales 8 h .. 8 h + 7
  uint32_t d;
  static constexpr int kBytes = kQ6KBytes;
  static constexpr int kPieces = 15;  // 16-byte pieces of a row's window: 210 bytes from the word boundary below, and one
                                      // more that spreads the rows of a tile over the LDS banks
  static constexpr uint32_t kStart = 3;  // windows start on words (so that they lie on 16 bytes in LDS, see sb_read_slot)
};
template <>
struct SbRaw<kQ8_0> {
  uint32_t v[34];  // blocks 4 h .. 4 h + 3, 34 bytes each
  static constexpr int kBytes = 8 * kQ8Bytes;
  static constexpr int kPieces = 17;  // 272 bytes, 16-byte aligned where rows are whole superblocks (18 otherwise)
  static constexpr uint32_t kStart = 15;
};

// `p`: the row's superblock (any even address, global or LDS)
__device__ __forceinline__ void sb_read(const uint8_t* p, int h, SbRaw<kQ6K>& r) {
#pragma unroll
  for (int i = 0; i < 4; ++i) __builtin_memcpy(&r.ql[i], __builtin_assume_aligned(p + 64 * h + 16 * i, 2), 16);
#pragma unroll
  for (int i = 0; i < 2; ++i) __builtin_memcpy(&r.qh[i], __builtin_assume_aligned(p + 128 + 32 * h + 16 * i, 2), 16);
  __builtin_memcpy(&r.sc, __builtin_assume_aligned(p + 192 + 8 * h, 2), 8);
  r.d = *reinterpret_cast<const uint16_t*>(p + 208);
}
// The raw words as registers nothing is known about.
__device__ __forceinline__ void opaque(SbRaw<kQ6K>& r) {
#pragma unroll
  for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(r.ql[i]));
#pragma unroll
  for (int i = 0; i < 2; ++i) asm volatile("" : "+v"(r.qh[i]));
  asm volatile("" : "+v"(r.sc.x), "+v"(r.sc.y), "+v"(r.d));
}
// A word of LDS by itself: the compiler would merge neighbours into a read wider than their alignment.
__device__ __forceinline__ uint32_t lds_word(const uint8_t* p) {
  return *reinterpret_cast<const volatile __attribute__((address_space(3))) uint32_t*>(
      (const volatile __attribute__((address_space(3))) uint8_t*)p);
}
// The same out of LDS, where a read that does not start on a multiple of its own width takes 64 cycles of the unit, one lane
// after the other (on such a multiple 4.4 for sixteen bytes per lane): superblocks lie at even offsets, so the words are
// read where words are and shifted by the half word that is left.  `p`: at most two bytes past a 16-byte boundary.
// (Seven reads at any even address held the unit 448 cycles per superblock of a tile, two thirds of the block's second
// launch at 45 tokens; these ten 60, and 26 shifts.)
__device__ __forceinline__ void sb_read_slot(const uint8_t* p, int h, SbRaw<kQ6K>& r) {
  const uint32_t at = (uint32_t)(uintptr_t)p, shift = (at & 2u) << 3;
  const uint8_t* const b = static_cast<const uint8_t*>(__builtin_assume_aligned(p - (at & 2u), 16));
  // (in place, run by run: the shifted words of all three runs beside the unshifted ones are registers the widest passes
  // do not have)
  auto shift_down = [&](uint32_t (&w)[4], uint32_t next) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 3; ++i) w[i] = __builtin_amdgcn_alignbit(w[i + 1], w[i], shift);
    w[3] = __builtin_amdgcn_alignbit(next, w[3], shift);
  };
  uint32_t w[6][4];
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    const v4u_t v = *reinterpret_cast<const v4u_t*>(i < 4 ? b + 64 * h + 16 * i : b + 64 + 32 * h + 16 * i);
#pragma unroll
    for (int j = 0; j < 4; ++j) w[i][j] = v[j];
  }
  const uint32_t ql_end = lds_word(b + 64 * h + 64), qh_end = lds_word(b + 160 + 32 * h);
  const uint2 sc = *reinterpret_cast<const uint2*>(b + 192 + 8 * h);
  const uint32_t sc_end = lds_word(b + 200 + 8 * h);
  r.d = *reinterpret_cast<const uint16_t*>(p + 208);
#pragma unroll
  for (int i = 0; i < 6; ++i) shift_down(w[i], i == 3 ? ql_end : i == 5 ? qh_end : w[i + 1][0]);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
#pragma unroll
    for (int i = 0; i < 4; ++i) r.ql[i][j] = w[i][j];
#pragma unroll
    for (int i = 0; i < 2; ++i) r.qh[i][j] = w[4 + i][j];
  }
  r.sc = make_uint2(__builtin_amdgcn_alignbit(sc.y, sc.x, shift), __builtin_amdgcn_alignbit(sc_end, sc.y, shift));
  opaque(r);  // (shifted here: put off until they are used, the words take more registers)
}
// (any even address, rows an odd number of words apart: word by word)
__device__ __forceinline__ void sb_read_words(const uint8_t* p, int h, SbRaw<kQ6K>& r) {
  const uint32_t at = (uint32_t)(uintptr_t)p, shift = (at & 2u) << 3;
  const uint8_t* const b = p - (at & 2u);
  uint32_t ql[17], qh[9], sc[3];
#pragma unroll
  for (int i = 0; i < 17; ++i) ql[i] = lds_word(b + 64 * h + 4 * i);
#pragma unroll
  for (int i = 0; i < 9; ++i) qh[i] = lds_word(b + 128 + 32 * h + 4 * i);
#pragma unroll
  for (int i = 0; i < 3; ++i) sc[i] = lds_word(b + 192 + 8 * h + 4 * i);
  r.d = *reinterpret_cast<const uint16_t*>(p + 208);
#pragma unroll
  for (int i = 0; i < 16; ++i) r.ql[i / 4][i % 4] = __builtin_amdgcn_alignbit(ql[i + 1], ql[i], shift);
#pragma unroll
  for (int i = 0; i < 8; ++i) r.qh[i / 4][i % 4] = __builtin_amdgcn_alignbit(qh[i + 1], qh[i], shift);
  r.sc = make_uint2(__builtin_amdgcn_alignbit(sc[1], sc[0], shift), __builtin_amdgcn_alignbit(sc[2], sc[1], shift));
  opaque(r);
}
__device__ __forceinline__ void sb_read(const uint8_t* p, int h, SbRaw<kQ8_0>& r) {  // (`p` on an 8-byte boundary)
#pragma unroll
  for (int i = 0; i < 17; ++i) {
    const uint2 t = *reinterpret_cast<const uint2*>(p + 136 * h + 8 * i);
    r.v[2 * i] = t.x;
    r.v[2 * i + 1] = t.y;
  }
}

__device__ __forceinline__ void sb_read_slot(const uint8_t* p, int h, SbRaw<kQ8_0>& r) { sb_read(p, h, r); }
__device__ __forceinline__ void sb_read_words(const uint8_t* p, int h, SbRaw<kQ8_0>& r) { sb_read(p, h, r); }

// Codes of group (s, l) as int8.  Q6_K codes come out times four, as signed bytes: the six bits sit at the byte's top with
// the code's top bit flipped (c - 32 in two's complement), which costs no more than unpacking them in place; the quarter
// is folded into the superblock's scale.
__device__ __forceinline__ void sb_codes(const SbRaw<kQ6K>& r, int s, int l, v4i_t& c) {
  const v4u_t a = r.ql[(s & 1) * 2 + l], q = r.qh[l];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // two shifts, one select of the two high bits from qh and the rest from ql, one mask and flip: four instructions per
    // four codes, spelled out because the compiler makes five of the plain expression
    const uint32_t lo = s < 2 ? a[i] << 2 : a[i] >> 2;
    const uint32_t hi = s == 0 ? q[i] << 6 : s == 1 ? q[i] << 4 : s == 2 ? q[i] << 2 : q[i];
    const uint32_t t = __builtin_amdgcn_bitop3_b32(hi, lo, 0xc0c0c0c0u, 0xE4);   // (hi & m) | (lo & ~m)
    c[i] = (int)__builtin_amdgcn_bitop3_b32(t, 0xfcfcfcfcu, 0x80808080u, 0x6A);  // (t & b) ^ c
  }
}
__device__ __forceinline__ void sb_codes(const SbRaw<kQ8_0>& r, int s, int l, v4i_t& c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int b = 34 * s + 2 + 16 * l + 4 * i;
    c[i] = (b & 2) ? (int)__builtin_amdgcn_alignbit(r.v[b / 4 + 1], r.v[b / 4], 16) : (int)r.v[b / 4];
  }
}
// The scale of group (s, l), as the product with d and, for Q6_K, by itself and without it.
__device__ __forceinline__ int sb_int_scale(const SbRaw<kQ6K>& r, int s, int l) {
  int v = (int8_t)((s < 2 ? r.sc.x : r.sc.y) >> (16 * (s & 1) + 8 * l));
  asm("" : "+v"(v));  // (one instruction here; as a byte operand of six products it would keep them from taking the sum in)
  return v;
}
__device__ __forceinline__ float sb_quarter(const SbRaw<kQ6K>& r) { return f16_bits_to_f32(r.d) * 0.25f; }
__device__ __forceinline__ float sb_scale(const SbRaw<kQ6K>& r, int s, int l) {
  return sb_quarter(r) * (float)(int8_t)((s < 2 ? r.sc.x : r.sc.y) >> (16 * (s & 1) + 8 * l));
}
__device__ __forceinline__ float sb_scale(const SbRaw<kQ8_0>& r, int s, int) {
  const int db = 34 * s;
  return f16_bits_to_f32((db & 2) ? r.v[db / 4] >> 16 : r.v[db / 4] & 0xffffu);
}

// The joined digit sums of a group (six exact integers, most significant first) as the group's sum, in units of the top
// pair: |digit sum| <= 2^18, so a pair is below 2^27.
__device__ __forceinline__ float join_digits(int d0, int d1, int d2, int d3, int d4, int d5) {
  const int hi = (d0 << 8) + d1, mid = (d2 << 8) + d3, lo = (d4 << 8) + d5;
  return __builtin_fmaf(__builtin_fmaf((float)lo, 0x1p-16f, (float)mid), 0x1p-16f, (float)hi);
}

// One more group's digit sum (at most 2^18 in magnitude) times its integer scale into the half superblock's.
__device__ __forceinline__ void add_scaled(int& sum, int scale, int digits) {
  sum = __mul24(scale, digits) + sum;
  asm("" : "+v"(sum));  // (a multiply-add each; the compiler would regroup them as products and three-way additions)
}
// join_digits for sums that went through a half superblock with their integer scales (six exact integers below 2^29).
__device__ __forceinline__ float join_sums(const int (&d)[6]) {
  float f = (float)d[5];
#pragma unroll
  for (int k = 4; k >= 1; --k) f = __builtin_fmaf(f, 0x1p-8f, (float)d[k]);
  return __builtin_fmaf((float)d[0], 256.0f, f);
}

// The lane's half superblock by plain fp32 multiply-adds in the order of the groups, weights dequantised exactly: what
// a half superblock with a mark goes through.  `x`: the superblock's activations, of which the half's 128 are taken, the same
// for the lanes of a DPP row; each of its sixteen lanes loads eight of them (one trip to memory) and the
// others take them from there.  `lane`: the pair forms pass fresh_lane(), whose registers are full (kept for this branch,
// which marked superblocks alone take, the lane's offset was spilled by every wavefront of the block's down launch: 13 / 32 /
// 45 tokens 432 / 488 / 608 us of blocks, 421 / 467 / 586 without); sb_dot, whose registers are not, passes the number it has
// (made anew 40 tokens of the dense sibling took 431 us instead of 429).
// (The registers go through an empty statement first and the groups are kept apart: the compiler would otherwise keep the
// codes it unpacked for the matrix instruction for this branch, or unpack all of them at once.)
__device__ __forceinline__ void opaque(SbRaw<kQ8_0>& r) {
#pragma unroll
  for (int i = 0; i < 34; ++i) asm volatile("" : "+v"(r.v[i]));
}
// elements 8 K .. 8 K + 7 of the half, which lane K of the row holds
template <int QUANT, int K>
__device__ __forceinline__ void half_fp32_eight(const SbRaw<QUANT>& r, const float (&own)[8], float& out) {
  constexpr int s = K / 4, l = (K >> 1) & 1;
  asm volatile("" : "+v"(out));
  v4i_t c;
  sb_codes(r, s, l, c);
  const float ws = sb_scale(r, s, l);
#pragma unroll
  for (int i = 0; i < 8; ++i)
    out = __builtin_fmaf(dpp_f<0x150 + K>(own[i]), ws * (float)(int8_t)(c[2 * (K & 1) + i / 4] >> (8 * (i % 4))), out);  // (row_newbcast:K)
}
template <int QUANT, int... K>
__device__ __forceinline__ float half_fp32_all(const SbRaw<QUANT>& r, const float (&own)[8], std::integer_sequence<int, K...>) {
  float out = 0.0f;
  (half_fp32_eight<QUANT, K>(r, own, out), ...);
  return out;
}
using HalfOrder = std::integer_sequence<int, 0, 1, 4, 5, 8, 9, 12, 13, 2, 3, 6, 7, 10, 11, 14, 15>;  // (l outermost)
__device__ __forceinline__ void half_own(const float* __restrict__ x, int half, int lane, float (&own)[8]) {
  const uint8_t* const at = reinterpret_cast<const uint8_t*>(x) + (uint32_t)(half * 512 + (lane & 15) * 32);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float4 v = reinterpret_cast<const float4*>(at)[i];
    own[4 * i] = v.x, own[4 * i + 1] = v.y, own[4 * i + 2] = v.z, own[4 * i + 3] = v.w;
  }
}
template <int QUANT>
__device__ __forceinline__ float half_fp32(SbRaw<QUANT>& r, const float* __restrict__ x, int half, int lane) {
  float own[8];
  half_own(x, half, lane, own);
  opaque(r);
  return half_fp32_all<QUANT>(r, own, HalfOrder{});
}

// The lane's eight group sums of one superblock for NT tokens: out[t] = the half's sum.
//   high_of(s, l, tg): operand A of group (s, l) for tokens 4 tg .. 4 tg + 3, or both tokens (zeros past NT)
//   low_of(s, l, tg): the low digits' operand (three tokens and more); l: which group's registers come first
//   e_of(t, l):     token t's scale of the superblock, or the four group scales (s = 0..3) in half `lane >> 5`
//   x_of(t):        token t's 256 fp32 activations (read where a scale is a mark)
//   live:           the lanes that hold a row (another lane's bytes may be anything, and its sum is not looked at)
//   dead:           this half of the superblock lies past the end of the row (its codes are other data's bytes)
// The work goes by units of (group, four tokens), or (block, four tokens): a unit's matrix instructions are issued before
// the sums of the unit before it are taken up, which covers their latency with two sets of result registers in rotation.
constexpr bool digits_in_one(int nt) { return nt <= 2; }
// (both groups of a block in one accumulator: the scale is the block's)
template <int QUANT, bool WHOLE>
constexpr bool kAddsGroups = WHOLE && QUANT == kQ8_0;

template <int QUANT, bool WHOLE, int NT, bool TAIL = false, typename HighOf, typename LowOf, typename EOf, typename XOf>
__device__ __forceinline__ void sb_dot(SbRaw<QUANT>& r, HighOf high_of, LowOf low_of, EOf e_of, XOf x_of, float (&out)[NT],
                                       uint64_t live, bool dead = false) {
  constexpr bool kOne = digits_in_one(NT), kPairs = kAddsGroups<QUANT, WHOLE>, kInts = WHOLE && QUANT == kQ6K;
  constexpr int TG = (NT + 3) / 4, kUnits = (kPairs ? 4 : 8) * TG;
#pragma unroll
  for (int t = 0; t < NT; ++t) out[t] = 0.0f;
  v16i_t d[2], z[2];
  v4i_t c[kPairs ? 2 : 1];
  float ws[2];                // the group's (block's) scale
  int sc[2];                  // kInts: its integer scale
  int sum[kInts ? NT : 1][6];
  float4 xe[WHOLE ? 1 : NT];
  if constexpr (kInts) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int k = 0; k < 6; ++k) sum[t][k] = 0;
  }
  auto issue = [&](int u) __attribute__((always_inline)) {
    const int j = u / TG, tg = u % TG, s = kPairs ? j : j & 3, l = kPairs ? 0 : j >> 2;
    if (tg == 0) {
      sb_codes(r, s, l, c[0]);
      if constexpr (kPairs) sb_codes(r, s, 1, c[1]);
      if constexpr (kInts) sc[j & 1] = sb_int_scale(r, s, l);
      else ws[j & 1] = TAIL && dead ? 0.0f : sb_scale(r, s, l);
    }
    const v16i_t zero = {0};
    v16i_t& dd = d[u & 1];
    dd = __builtin_amdgcn_mfma_i32_32x32x32_i8(high_of(s, l, tg), c[0], zero, 0, 0, 0);
    if constexpr (kPairs) dd = __builtin_amdgcn_mfma_i32_32x32x32_i8(high_of(s, 1, tg), c[1], dd, 0, 0, 0);
    if constexpr (!kOne) {
      v16i_t& zz = z[u & 1];
      zz = __builtin_amdgcn_mfma_i32_32x32x32_i8(low_of(s, 0, tg), c[0], zero, 0, 0, 0);
      if constexpr (kPairs) zz = __builtin_amdgcn_mfma_i32_32x32x32_i8(low_of(s, 1, tg), c[1], zz, 0, 0, 0);
    }
  };
  issue(0);
#pragma unroll
  for (int u = 0; u < kUnits; ++u) {
    const int j = u / TG, tg = u % TG, s = j & 3, l = kPairs ? 0 : j >> 2;
    if (u + 1 < kUnits) issue(u + 1);
    if constexpr (!WHOLE) {
      if (s == 0 && tg == 0) {
#pragma unroll
        for (int t = 0; t < NT; ++t) xe[t] = e_of(t, l);
      }
    }
#pragma unroll
    for (int t = 4 * tg; t < 4 * tg + 4 && t < NT; ++t) {
      const v16i_t& dd = d[u & 1];
      const v16i_t& zz = kOne ? dd : z[u & 1];
      const int k = kOne ? 8 * t : 4 * (t & 3), kz = kOne ? k + 4 : k + 2 * l;
      if constexpr (kInts) {
#pragma unroll
        for (int i = 0; i < 4; ++i) add_scaled(sum[t][i], sc[j & 1], dd[k + i]);
#pragma unroll
        for (int i = 0; i < 2; ++i) add_scaled(sum[t][4 + i], sc[j & 1], zz[kz + i]);
      } else {
        const float f = join_digits(dd[k], dd[k + 1], dd[k + 2], dd[k + 3], zz[kz], zz[kz + 1]);
        if constexpr (WHOLE) {
          out[t] = __builtin_fmaf(f, ws[j & 1], out[t]);
        } else {
          const float e = s == 0 ? xe[t].x : s == 1 ? xe[t].y : s == 2 ? xe[t].z : xe[t].w;
          out[t] = __builtin_fmaf(f, ws[j & 1] * e, out[t]);
        }
      }
    }
  }
  if constexpr (WHOLE) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if constexpr (kInts) out[t] = join_sums(sum[t]) * (sb_quarter(r) * e_of(t, 0));
      else out[t] *= e_of(t, 0);
    }
  }
  uint32_t marked = 0;
#pragma unroll
  for (int t = 0; t < NT; ++t)
    if (__builtin_amdgcn_ballot_w64(out[t] != out[t]) & live) marked |= 1u << t;
  if (__builtin_expect(marked != 0, 0)) {
#pragma unroll 1
    for (; marked; marked &= marked - 1) {
      const int m = __builtin_ctz(marked);
      const float plain = half_fp32(r, x_of(m), TAIL && dead ? 0 : (int)__lane_id() >> 5, (int)__lane_id());
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (t == m && out[t] != out[t]) out[t] = TAIL && dead ? 0.0f : plain;
    }
  }
}

// Where a lane finds its row of the operands A of tokens 4 tg .. 4 tg + 3 (or of both tokens), relative to group (s, 0) of
// token 0, in a pass of NT tokens that lie `stride` bytes apart: the high one's (group (s, 1) lies kGroupBytes further
// on) and the low one's.  Negative: the row is zero.
template <int NT>
__device__ __forceinline__ int high_digit_at(int lane, int tg, int stride) {
  const int h = lane >> 5, m = lane & 31, i = 4 * (m >> 3) + (m & 3);  // the row's register in half h
  const int t = digits_in_one(NT) ? i >> 3 : 4 * tg + (m >> 3), digit = digits_in_one(NT) ? i & 7 : m & 3;
  return ((m >> 2) & 1) == h && t < NT && digit < 6 ? t * stride + 2 * h * kGroupBytes + digit * 16 : -1;
}
template <int NT>
__device__ __forceinline__ int low_digit_at(int lane, int l, int tg, int stride) {
  const int h = lane >> 5, m = lane & 31, t = 4 * tg + (m >> 3);
  return ((m >> 2) & 1) == h && t < NT ? t * stride + (2 * h + (((m >> 1) & 1) ^ l)) * kGroupBytes + (4 + (m & 1)) * 16 : -1;
}

// Operands A and the group scales out of LDS; `zeros`: kZeroBytes of zero bytes that the lanes without a digit read.
constexpr int kSbLdsBytes = kSbDigitBytes + kSbScaleBytes;  // 400 words: four tokens' rows start 16 banks apart
template <int NT, int STRIDE, bool SWAPPED>  // SWAPPED: the low operand with the second group first is wanted, too
struct LdsDigits {
  static constexpr int kQuads = (NT + 3) / 4;
  const uint8_t *a[kQuads], *z[SWAPPED ? 2 : 1][kQuads];
  const uint8_t* e;
  // `digits`, `scales`: token 0's, the other tokens' STRIDE and E_STRIDE bytes apart
  __device__ __forceinline__ void point(const uint8_t* digits, const uint8_t* scales, const uint8_t* zeros) {
    const int lane = (int)__lane_id();
#pragma unroll
    for (int tg = 0; tg < kQuads; ++tg) {
      const int at = high_digit_at<NT>(lane, tg, STRIDE);
      a[tg] = at >= 0 ? digits + at : zeros;
#pragma unroll
      for (int l = 0; l < (SWAPPED ? 2 : 1); ++l) {
        const int low = low_digit_at<NT>(lane, l, tg, STRIDE);
        z[l][tg] = low >= 0 ? digits + low : zeros;
      }
    }
    e = scales + (lane >> 5) * 32;
  }
  __device__ __forceinline__ v4i_t high(int s, int l, int tg) const {
    return *reinterpret_cast<const v4i_t*>(a[tg] + (4 * s + l) * kGroupBytes);
  }
  __device__ __forceinline__ v4i_t low(int s, int l, int tg) const {
    return *reinterpret_cast<const v4i_t*>(z[SWAPPED ? l : 0][tg] + 4 * s * kGroupBytes);
  }
  template <int E_STRIDE>
  __device__ __forceinline__ float4 scale(int t, int l) const { return *reinterpret_cast<const float4*>(e + t * E_STRIDE + l * 16); }
};

template <int N>
__device__ __forceinline__ void wait_but() {  // all but the last N requests of this wavefront are there
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}


// What the pieces of the window that starts at byte `start` of a tensor and ends with it could not hold, two bytes at a time,
// to the window at `slot`.  SPAN: the bytes wanted from `start` on.
template <int QUANT, int SPAN = SbRaw<QUANT>::kBytes>
__device__ __forceinline__ void patch_window(const uint8_t* w, size_t start, uint8_t* slot) {
  int lane = (int)__lane_id();
  asm volatile("" : "+v"(lane));  // (once per launch: its arithmetic stays here, out of the registers of the loop around)
  const size_t from = start & ~(size_t)SbRaw<QUANT>::kStart, whole = (start + SPAN - from) & ~(size_t)15;
  if (2 * lane < (int)(start + SPAN - from - whole))
    *reinterpret_cast<uint16_t*>(slot + whole + 2 * lane) = *reinterpret_cast<const uint16_t*>(w + from + whole + 2 * lane);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------------
// A wavefront's private LDS slot for one superblock of 32 rows (two runs of 16 rows each, from one matrix or from
// two), filled by global -> LDS DMA.  Each row's window is requested as whole 16-byte pieces: a lane that reads its
// fields out of global memory touches every cache line of the rows with each of its eight loads, and the vector L1
// stalls on lines that are still pending (130 us against 85 for a one-token pass over the 248 320-row Q6_K matrix).
// One slot is enough: it is free again as soon as its bytes are in registers, so the next request is in flight
// while this superblock is multiplied.
// ---------------------------------------------------------------------------------
template <int QUANT, int PIECES = SbRaw<QUANT>::kPieces>
struct SliceDma {
  static constexpr int kP = PIECES;
  static constexpr int kInstr = (16 * kP + 63) / 64;  // DMA instructions per run
  static constexpr int kLast = 16 * kP - 64 * (kInstr - 1);  // lanes the last of them is for
  static constexpr int kRunBytes = 16 * kP * 16;
  static constexpr int kSlotBytes = 2 * kRunBytes;
  uint32_t row_bytes;
  uint32_t row_off[kInstr], col[kInstr];

  // `rows`: live rows of a run (1..16); the others repeat the last
  __device__ __forceinline__ void init(uint32_t row_bytes_, int rows) {
    row_bytes = row_bytes_;
    const int lane = (int)__lane_id();
#pragma unroll
    for (int i = 0; i < kInstr; ++i) {
      const int pc = min(64 * i + lane, 16 * kP - 1);
      row_off[i] = (uint32_t)min(pc / kP, rows - 1) * row_bytes;
      col[i] = (uint32_t)(pc % kP) * 16;
    }
  }
  // Requests superblock `sb` of the run whose first row starts `run_off` bytes into the tensor at `w` (16-byte aligned,
  // `w_bytes` long) into LDS at `dst` (byte address).  Pieces that would reach past the tensor repeat its end.
  __device__ __forceinline__ void request(const uint8_t* w, size_t w_bytes, size_t run_off, int sb, uint32_t dst) const {
    constexpr uint32_t kStart = SbRaw<QUANT>::kStart;
    const uint8_t* base = w + (run_off & ~(size_t)15);
    const uint32_t mis = (uint32_t)run_off & 15u;
    const size_t left = w_bytes - (run_off & ~(size_t)15);
    const uint32_t last = (uint32_t)min(left >= 16 ? (left - 16) & ~(size_t)kStart : (size_t)0, (size_t)0xfffffff0u);
#pragma unroll
    for (int i = 0; i < kInstr; ++i) {
      const uint32_t voff = min(((mis + row_off[i] + (uint32_t)(sb * SbRaw<QUANT>::kBytes)) & ~kStart) + col[i], last);
      if (i + 1 < kInstr || kLast == 64 || (int)__lane_id() < kLast) lds_dma_16(base, voff, dst + i * 1024);
    }
  }
  // The run's `live` rows end the tensor, and `sb` is their last superblock: the bytes that no piece inside the tensor
  // held go to the slot two by two.
  __device__ __forceinline__ bool ends_apart(size_t w_bytes) const { return QUANT == kQ6K || (w_bytes & 15) != 0; }
  __device__ __forceinline__ void patch_tail(const uint8_t* w, size_t run_off, int live, int sb, uint8_t* run_slot) const {
    const size_t start = run_off + (size_t)(live - 1) * row_bytes + (size_t)sb * SbRaw<QUANT>::kBytes;
    patch_window<QUANT>(w, start, run_slot + (live - 1) * (kP * 16));
  }
  // the address of the lane's row inside the run's slot
  __device__ __forceinline__ const uint8_t* row_at(const uint8_t* run_slot, size_t run_off, int row, int sb) const {
    const uint32_t mis = ((uint32_t)run_off + (uint32_t)row * row_bytes + (uint32_t)(sb * SbRaw<QUANT>::kBytes)) & SbRaw<QUANT>::kStart;
    return run_slot + row * (kP * 16) + mis;
  }
};

// ---------------------------------------------------------------------------------
// Sixteen rows of two superblocks, one token: the one-token form of the core, on v_mfma_i32_16x16x64_i8.  Lane 16 q + r
// holds row r and half q & 1 of superblock q >> 1 of the pair; operand A's row m is digit m & 3 in quarter m >> 2 of K
// and zero elsewhere, so that the four result registers of a lane are the digit sums of the sixteen elements the lane
// itself unpacked.  The same exact sums and the same fp32 operations per half superblock as sb_dot's, with no operand
// rows spent on other tokens: for a single token 32 rows x 1 superblock and this shape carry the same bytes, and this
// one needs no zeros in LDS, four result registers instead of sixteen, and fits rows of one or two superblocks (a pair
// is then one row or two).  A caller may as well give quarters 2 and 3 sixteen other rows of the same superblock.
// ---------------------------------------------------------------------------------
// N byte offsets below 65536, two to a register: what a lane adds per DMA instruction, unpacked where it is used.
template <int N>
struct PackedOffsets {
  uint32_t p[(N + 1) / 2];
  __device__ __forceinline__ void set(int i, uint32_t v) { p[i / 2] = i & 1 ? p[i / 2] | v << 16 : v; }
  __device__ __forceinline__ uint32_t get(int i) const { return i & 1 ? p[i / 2] >> 16 : p[i / 2] & 0xffffu; }
  // (before a round of get: the compiler would unpack all of them ahead of the loop otherwise)
  __device__ __forceinline__ void opaque() {
#pragma unroll
    for (int i = 0; i < (N + 1) / 2; ++i) asm volatile("" : "+v"(p[i]));
  }
};

// PACKED: the last instruction is for the lanes with a piece only, and slots lie without padding between them.
template <int QUANT, int PIECES = QUANT == kQ6K ? 29 : 35, bool PACKED = false>
struct PairDma {
  static constexpr int kP = PIECES;  // 420 bytes from a word boundary, rows four words apart modulo the banks; 35 likewise
  static constexpr int kInstr = (16 * kP + 63) / 64, kSlotBytes = PACKED ? 16 * kP * 16 : kInstr * 1024;  // (otherwise the last instruction pads)
  PackedOffsets<kInstr> off;  // the lane's piece of each instruction, relative to the tile's first row
  // sixteen rows of `row_bytes` (16 row_bytes are whole pieces, and fewer than 65536), superblocks sb0 and sb0 + 1
  __device__ __forceinline__ void init(uint32_t row_bytes, int sb0) {
    const int lane = (int)__lane_id();
#pragma unroll
    for (int i = 0; i < kInstr; ++i) {
      const int pc = min(64 * i + lane, 16 * kP - 1);
      off.set(i, (((uint32_t)(pc / kP) * row_bytes + (uint32_t)(sb0 * SbRaw<QUANT>::kBytes)) & ~SbRaw<QUANT>::kStart) + (uint32_t)(pc % kP) * 16);
    }
  }
  // `tile`: offset of the tile's first row in the tensor at `w` (16-byte aligned, `w_bytes` long, like the tile); pieces
  // that would reach past the tensor repeat its end (Q6_K: see patch_tail; otherwise they are padding)
  __device__ __forceinline__ void request(const uint8_t* w, size_t w_bytes, size_t tile, uint32_t dst) {
    const uint32_t last = (uint32_t)min((w_bytes & ~(size_t)15) - 16 - tile, (size_t)0xfffffff0u);
    off.opaque();
#pragma unroll
    for (int i = 0; i < kInstr; ++i)
      if (!PACKED || i + 1 < kInstr || (int)__lane_id() < 16 * kP - 64 * (kInstr - 1)) lds_dma_16(w + tile, min(off.get(i), last), dst + i * 1024);
  }
  // (the tile's last row, this pair its last one, ends the tensor; Q6_K)
  static __device__ __forceinline__ void patch_tail(const uint8_t* w, size_t w_bytes, uint8_t* slot) {
    patch_window<QUANT, 2 * SbRaw<QUANT>::kBytes>(w, w_bytes - 2 * SbRaw<QUANT>::kBytes, slot + 15 * (kP * 16));
  }
  static __device__ __forceinline__ const uint8_t* row_at(const uint8_t* slot, uint32_t row_bytes, int row, int sb0) {
    return slot + row * (kP * 16) + (((uint32_t)row * row_bytes + (uint32_t)(sb0 * SbRaw<QUANT>::kBytes)) & SbRaw<QUANT>::kStart);
  }
};

// The same slot where the sixteen pairs follow one another in memory (rows of one or two superblocks) from a 16-byte
// boundary: 6720 or 8704 bytes, whole pieces, requested as they lie.  Q6_K pairs keep their 420-byte stride (105 words:
// no two rows on one bank); Q8_0 pairs of 544 bytes get a piece between them.
template <int QUANT>
struct PairRunDma {
  static constexpr int kPairPieces = 2 * SbRaw<QUANT>::kBytes / 16;  // (Q8_0: 34; Q6_K pairs are not whole pieces)
  static constexpr int kRowStride = QUANT == kQ6K ? 2 * kQ6KBytes : (kPairPieces + 1) * 16;
  static constexpr int kPieces = 16 * kRowStride / 16;
  static constexpr int kInstr = (kPieces + 63) / 64, kSlotBytes = kInstr * 1024;
  PackedOffsets<kInstr> off;
  __device__ __forceinline__ void init() {
    const uint32_t lane = __lane_id();
#pragma unroll
    for (int i = 0; i < kInstr; ++i) {
      const uint32_t pc = min((uint32_t)(64 * i) + lane, (uint32_t)kPieces - 1);  // (a slot's padding repeats its last piece)
      off.set(i, QUANT == kQ6K ? pc * 16 : (pc / (kPairPieces + 1) * kPairPieces + min(pc % (kPairPieces + 1), (uint32_t)kPairPieces - 1)) * 16);
    }
  }
  __device__ __forceinline__ void request(const uint8_t* run, uint32_t dst) {
    off.opaque();
#pragma unroll
    for (int i = 0; i < kInstr; ++i) lds_dma_16(run, off.get(i), dst + i * 1024);
  }
};

// Operands A and the scales of the lane's half superblock, straight from memory.
template <bool WHOLE>
struct PairDigits {
  v4i_t a[8];                // [4 l + s]: digits 0..3
  v4i_t z[4];                // [s]: digits 4 and 5 of l = 0, then of l = 1
  float4 e[WHOLE ? 1 : 2];   // the superblock's in .x, or [l], s = 0..3
  // `xd`, `xe`: digits and scales of the activation superblock the lane's weights lie in (SCALES false: the digits
  // only; one function, because with the scales' loads in another the block's down launch spilled 9 more registers and 13
  // tokens took 3 % longer)
  template <bool SCALES = true>
  __device__ __forceinline__ void load(const uint8_t* xd, const float* xe) {
    const int lane = (int)__lane_id(), q = lane >> 4, m = lane & 15, h = q & 1;
    const bool mine = (m >> 2) == q;
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] = v4i_t{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; ++s) z[s] = v4i_t{0, 0, 0, 0};
    if (mine) {  // (one region for all twelve loads)
      const uint8_t* p = xd + 2 * h * kGroupBytes;
      const uint8_t *pa = p + (m & 3) * 16, *pz = p + ((m >> 1) & 1) * kGroupBytes + (4 + (m & 1)) * 16;
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = *reinterpret_cast<const v4i_t*>(pa + (4 * (j & 3) + (j >> 2)) * kGroupBytes);
#pragma unroll
      for (int s = 0; s < 4; ++s) z[s] = *reinterpret_cast<const v4i_t*>(pz + 4 * s * kGroupBytes);
    }
    if constexpr (SCALES && WHOLE) {
      e[0].x = *xe;
    } else if constexpr (SCALES) {
#pragma unroll
      for (int l = 0; l < 2; ++l) e[l] = reinterpret_cast<const float4*>(xe)[2 * h + l];
    }
  }
};

// `x_of(quarter)`: the 256 fp32 activations of the superblock that quarter `lane >> 4` of the wavefront holds, read where
// a scale is a mark.  `dead`: the lane's half lies past the end of the row (its codes are other data's bytes).
template <int QUANT, bool WHOLE, bool TAIL = false, typename XOf>
__device__ __forceinline__ float pair_dot(SbRaw<QUANT>& r, const PairDigits<WHOLE>& x, XOf x_of, bool dead = false) {
  constexpr bool kPairs = kAddsGroups<QUANT, WHOLE>, kInts = WHOLE && QUANT == kQ6K;
  constexpr int kUnits = kPairs ? 4 : 8;
  float out = 0.0f, ws[2];
  int sc[2], sum[6] = {0, 0, 0, 0, 0, 0};
  v4i_t d[2], z[2];
  auto issue = [&](int j) __attribute__((always_inline)) {
    const int s = kPairs ? j : j & 3, l = kPairs ? 0 : j >> 2;
    const v4i_t zero = {0, 0, 0, 0};
    v4i_t c;
    sb_codes(r, s, l, c);
    if constexpr (kInts) sc[j & 1] = sb_int_scale(r, s, l);
    else ws[j & 1] = sb_scale(r, s, l);
    d[j & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.a[4 * l + s], c, zero, 0, 0, 0);
    z[j & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.z[s], c, zero, 0, 0, 0);
    if constexpr (kPairs) {
      sb_codes(r, s, 1, c);
      d[j & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.a[4 + s], c, d[j & 1], 0, 0, 0);
      const v4i_t second = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.z[s], c, zero, 0, 0, 0);
      z[j & 1][2] = second[2];  // (the first group's sums stay in the first two registers)
      z[j & 1][3] = second[3];
    }
  };
  issue(0);
#pragma unroll
  for (int j = 0; j < kUnits; ++j) {
    if (j + 1 < kUnits) issue(j + 1);
    const v4i_t &dd = d[j & 1], &zz = z[j & 1];
    const int s = kPairs ? j : j & 3, l = kPairs ? 0 : j >> 2;
    if constexpr (kInts) {
#pragma unroll
      for (int i = 0; i < 4; ++i) add_scaled(sum[i], sc[j & 1], dd[i]);
#pragma unroll
      for (int i = 0; i < 2; ++i) add_scaled(sum[4 + i], sc[j & 1], zz[2 * l + i]);
    } else if constexpr (WHOLE) {
      out = __builtin_fmaf(join_digits(dd[0], dd[1], dd[2], dd[3], zz[0] + zz[2], zz[1] + zz[3]), ws[j & 1], out);
    } else {
      const float4& e = x.e[l];
      out = __builtin_fmaf(join_digits(dd[0], dd[1], dd[2], dd[3], zz[2 * l], zz[2 * l + 1]),
                           ws[j & 1] * (s == 0 ? e.x : s == 1 ? e.y : s == 2 ? e.z : e.w), out);
    }
  }
  if constexpr (kInts) out = join_sums(sum) * (sb_quarter(r) * x.e[0].x);
  else if constexpr (WHOLE) out *= x.e[0].x;
  if (TAIL && dead) out = 0.0f;
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(out != out) != 0, 0)) {
    const int lane = fresh_lane(), quarter = lane >> 4;
    const float plain = half_fp32(r, x_of(quarter), TAIL && dead ? 0 : quarter & 1, lane);
    if (out != out) out = plain;
  }
  return out;
}

// The same for the rows' codes against one or two tokens (whole superblocks, Q6_K), the digits in LDS: the codes are unpacked
// once, the sums are pair_dot's.  Where a lane finds its rows of the two operands, relative to its superblock's digits
// (negative: the row is zero, and the lane reads zeros).
__device__ __forceinline__ int pair_high_at(int lane) {
  const int q = lane >> 4, m = lane & 15;
  return (m >> 2) == q ? 2 * (q & 1) * kGroupBytes + (m & 3) * 16 : -1;
}
__device__ __forceinline__ int pair_low_at(int lane) {
  const int q = lane >> 4, m = lane & 15;
  return (m >> 2) == q ? (2 * (q & 1) + ((m >> 1) & 1)) * kGroupBytes + (4 + (m & 1)) * 16 : -1;
}
template <int NT, typename XOf>
__device__ __forceinline__ void pair_dot_lds(SbRaw<kQ6K>& r, const uint8_t* const (&high)[NT], const uint8_t* const (&low)[NT],
                                             const float (&e)[NT], XOf x_of, float (&out)[NT]) {
  int sum[NT][6];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int k = 0; k < 6; ++k) sum[t][k] = 0;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    v4i_t z[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) z[t] = *reinterpret_cast<const v4i_t*>(low[t] + 4 * s * kGroupBytes);
#pragma unroll
    for (int l = 0; l < 2; ++l) {
      const v4i_t zero = {0, 0, 0, 0};
      v4i_t c;
      sb_codes(r, s, l, c);
      const int sc = sb_int_scale(r, s, l);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const v4i_t a = *reinterpret_cast<const v4i_t*>(high[t] + (4 * s + l) * kGroupBytes);
        const v4i_t dd = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, c, zero, 0, 0, 0);
        const v4i_t zz = __builtin_amdgcn_mfma_i32_16x16x64_i8(z[t], c, zero, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) add_scaled(sum[t][i], sc, dd[i]);
#pragma unroll
        for (int i = 0; i < 2; ++i) add_scaled(sum[t][4 + i], sc, zz[2 * l + i]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    out[t] = join_sums(sum[t]) * (sb_quarter(r) * e[t]);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(out[t] != out[t]) != 0, 0)) {
      const int lane = fresh_lane(), quarter = lane >> 4;
      const float plain = half_fp32(r, x_of(t, quarter), quarter & 1, lane);
      if (out[t] != out[t]) out[t] = plain;
    }
  }
}

}  // namespace xabe
