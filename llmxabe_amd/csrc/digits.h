// Quantized rows times fp32 activations on the int8 matrix instruction, at fp32 grade: the contraction every fp32
// regime of this library goes through (decode, dispatch-table and dense widths, the LM head).
//
// A Q6_K or Q8_0 weight is an integer code times a scale per 16 or 32 elements, so inside one group of 16 elements the
// product with the activations is an integer-weighted sum.  An activation is written as a 32-bit fixed-point number
// relative to its group of 16 (a power-of-two scale that puts the group's largest magnitude between 2^29 and 2^30) and
// that number as four signed base-256 digits.  Codes and digits are int8, so the four digit sums of a group come out
// of v_mfma_i32_32x32x32_i8 exact; what is left for the vector ALU is seven instructions per (row, group, token):
// two shift-adds that pair the digit sums, two conversions, one fused multiply-add that joins the pairs, the product
// of the weight's and the activation's scale, and the fused multiply-add into the row's fp32 sum.
//
// Precision: a value within a factor of 2^6 of its group's largest keeps all 24 bits of its fp32 significand, a smaller
// one is off by at most 2^-31 of that largest; the sums inside a group are exact, where sixteen fp32 multiply-adds
// round sixteen times.  Measured against a float64 reference: 1e-7 of the outputs' peak, the fp32 lane sums this
// replaced 1.7e-7.
//
// Why this form: one conversion and one multiply-add per weight and token on a 16-lane SIMD (4.9 vector instructions
// per weight in all) bound every batch wider than a few tokens.  Here a weight costs ~1.3 instructions to unpack
// (none for Q8_0, whose codes are the operand as they lie) and 7/16 per token.  LM head, 2048 -> 248 320 Q8_0, eight
// tokens: 303 -> 120 us; Q6_K, one token: 104 -> 85 us.
//
// The matrix instruction's layout: operand A (activations) row m = lane & 31, operand B (weights) column = lane & 31,
// both with the sixteen K positions of half `lane >> 5` in the lane's four registers; the result's column is the
// lane's own, its row 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3) for register i.  A's row m is digit m & 3 of token
// m >> 3, and only the half (m >> 2) & 1 of it is nonzero: a result register of half h then holds the digit sum over
// the sixteen elements that half h of the wavefront unpacked, so scales and codes meet in one lane.
//
// Order of operations (the numerics contract: a row's value depends on the row and the token only).  A superblock of
// 256 elements is split between the wavefront's halves: half h takes elements 128 h + 32 s + 16 l + [0, 16), s = 0..3,
// l = 0, 1, and sums its eight groups from zero, l outermost.  Superblock sums are added in the order a kernel states.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"

namespace xabe {

typedef int v4i_t __attribute__((ext_vector_type(4)));
typedef int v16i_t __attribute__((ext_vector_type(16)));
typedef uint32_t v4u_t __attribute__((ext_vector_type(4)));

constexpr int kSbElems = 256;
// One superblock of one token: digit planes [s][2 h + l][digit, most significant first][16 elements], then the group
// scales [2 h + l][s] as floats.
constexpr int kSbDigitBytes = 1024, kSbScaleBytes = 64;

// Digits and scale of one group of 16 activations.  A group holding an infinity or a NaN gets a NaN scale.
__device__ __forceinline__ void digitize16(const float (&x)[16], v4u_t (&plane)[4], float& scale) {
  uint32_t mag = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) mag = max(mag, __builtin_bit_cast(uint32_t, x[i]) & 0x7fffffffu);
  const int e = (int)(mag >> 23);
  const int s = min(156 - e, 126);  // |x| 2^s < 2^30
  uint32_t y[16];
#pragma unroll
  for (int i = 0; i < 16; ++i)  // (x + 0x80 per lower byte, minus it again byte by byte: signed digits)
    y[i] = ((uint32_t)(int)__builtin_rintf(__builtin_ldexpf(x[i], s)) + 0x00808080u) ^ 0x00808080u;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const uint32_t a = y[4 * w], b = y[4 * w + 1], c = y[4 * w + 2], d = y[4 * w + 3];
    const uint32_t ab_hi = __builtin_amdgcn_perm(b, a, 0x07030602u), cd_hi = __builtin_amdgcn_perm(d, c, 0x07030602u);
    const uint32_t ab_lo = __builtin_amdgcn_perm(b, a, 0x05010400u), cd_lo = __builtin_amdgcn_perm(d, c, 0x05010400u);
    plane[0][w] = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x07060302u);
    plane[1][w] = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x05040100u);
    plane[2][w] = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x07060302u);
    plane[3][w] = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x05040100u);
  }
  scale = e == 255 ? __builtin_nanf("") : __builtin_ldexpf(1.0f, 16 - s);  // (x = digits' value 2^-16 times this)
}

// Where group `pos` (elements 16 pos .. 16 pos + 15 of its superblock) lies among the digit planes and the scales.
__device__ __forceinline__ int digit_group_offset(int pos) {
  const int h = pos >> 3, s = (pos >> 1) & 3, l = pos & 1;
  return s * 256 + (2 * h + l) * 64;
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
  static constexpr int kPieces = 15;  // 16-byte pieces of a row's window: 210 bytes at any even offset, and one more
                                      // that spreads the rows of a tile over the LDS banks
};
template <>
struct SbRaw<kQ8_0> {
  uint32_t v[34];  // blocks 4 h .. 4 h + 3, 34 bytes each
  static constexpr int kBytes = 8 * kQ8Bytes;
  static constexpr int kPieces = 17;  // 272 bytes, 16-byte aligned where rows are whole superblocks (18 otherwise)
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
__device__ __forceinline__ void sb_read(const uint8_t* p, int h, SbRaw<kQ8_0>& r) {  // (`p` on an 8-byte boundary)
#pragma unroll
  for (int i = 0; i < 17; ++i) {
    const uint2 t = *reinterpret_cast<const uint2*>(p + 136 * h + 8 * i);
    r.v[2 * i] = t.x;
    r.v[2 * i + 1] = t.y;
  }
}

// Codes of group (s, l) as int8 and the scale that goes with them.  Q6_K codes come out times four, as signed bytes:
// the six bits sit at the byte's top with the code's top bit flipped (c - 32 in two's complement), which costs no more
// than unpacking them in place; the quarter is folded into d.
__device__ __forceinline__ void sb_group(const SbRaw<kQ6K>& r, int s, int l, v4i_t& c, float& ws) {
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
  const uint32_t sw = s < 2 ? r.sc.x : r.sc.y;
  ws = (f16_bits_to_f32(r.d) * 0.25f) * (float)(int8_t)(sw >> (16 * (s & 1) + 8 * l));
}
__device__ __forceinline__ void sb_group(const SbRaw<kQ8_0>& r, int s, int l, v4i_t& c, float& ws) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int b = 34 * s + 2 + 16 * l + 4 * i;
    c[i] = (b & 2) ? (int)__builtin_amdgcn_alignbit(r.v[b / 4 + 1], r.v[b / 4], 16) : (int)r.v[b / 4];
  }
  const int db = 34 * s;
  ws = f16_bits_to_f32((db & 2) ? r.v[db / 4] >> 16 : r.v[db / 4] & 0xffffu);
}

// The lane's eight group sums of one superblock for NT tokens: out[t] = the half's sum, from zero.
//   a_of(s, l, tg): operand A of group (s, l) for tokens 4 tg .. 4 tg + 3 (zeros for tokens past NT)
//   e_of(t, l):     the four group scales (s = 0..3) of token t in half `lane >> 5`
//   dead:           this half of the superblock lies past the end of the row (its codes are other data's bytes)
// The work goes by units of (group, four tokens): a unit's matrix instruction is issued before the sums of the unit
// before it are taken up, which covers its latency with two result registers in rotation.
template <int QUANT, int NT, bool TAIL = false, typename AOf, typename EOf>
__device__ __forceinline__ void sb_dot(const SbRaw<QUANT>& r, AOf a_of, EOf e_of, float (&out)[NT], bool dead = false) {
  constexpr int TG = (NT + 3) / 4, kUnits = 8 * TG;
#pragma unroll
  for (int t = 0; t < NT; ++t) out[t] = 0.0f;
  v16i_t d[2];
  v4i_t c;
  float ws[2];
  float4 xe[NT];
  auto issue = [&](int u) __attribute__((always_inline)) {
    const int j = u / TG, tg = u % TG;
    if (tg == 0) {
      sb_group(r, j & 3, j >> 2, c, ws[j & 1]);
      if (TAIL && dead) ws[j & 1] = 0.0f;
    }
    const v16i_t zero = {0};
    d[u & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a_of(j & 3, j >> 2, tg), c, zero, 0, 0, 0);
  };
  issue(0);
#pragma unroll
  for (int u = 0; u < kUnits; ++u) {
    const int j = u / TG, tg = u % TG, s = j & 3, l = j >> 2;
    if (u + 1 < kUnits) issue(u + 1);
    if (s == 0 && tg == 0) {
#pragma unroll
      for (int t = 0; t < NT; ++t) xe[t] = e_of(t, l);
    }
#pragma unroll
    for (int t = 4 * tg; t < 4 * tg + 4 && t < NT; ++t) {
      const v16i_t& dd = d[u & 1];
      const int k = 4 * (t & 3);
      const int hi = (dd[k] << 8) + dd[k + 1], lo = (dd[k + 2] << 8) + dd[k + 3];
      const float f = __builtin_fmaf((float)lo, 0x1p-16f, (float)hi);
      const float e = s == 0 ? xe[t].x : s == 1 ? xe[t].y : s == 2 ? xe[t].z : xe[t].w;
      out[t] = __builtin_fmaf(f, ws[j & 1] * e, out[t]);
    }
  }
}

// Operand A and the group scales out of LDS, tokens of a superblock kSbBytes apart (digits, then scales); `zeros`: a
// kilobyte of zero bytes that the lanes without a digit read.
constexpr int kSbLdsBytes = kSbDigitBytes + kSbScaleBytes;  // 272 words: four tokens' rows start 16 banks apart
template <int NT, int STRIDE>
struct LdsDigits {
  static constexpr int kQuads = (NT + 3) / 4;
  const uint8_t* a[kQuads];
  const uint8_t* e;
  // `digits`, `scales`: token 0's, the other tokens' STRIDE and E_STRIDE bytes apart
  __device__ __forceinline__ void point(const uint8_t* digits, const uint8_t* scales, const uint8_t* zeros) {
    const int lane = (int)__lane_id(), h = lane >> 5, m = lane & 31;
    const bool mine = ((m >> 2) & 1) == h;
#pragma unroll
    for (int tg = 0; tg < kQuads; ++tg) {
      const int t = 4 * tg + (m >> 3);
      a[tg] = mine && t < NT ? digits + t * STRIDE + h * 128 + (m & 3) * 16 : zeros;
    }
    e = scales + h * 32;
  }
  __device__ __forceinline__ v4i_t digit(int s, int l, int tg) const { return *reinterpret_cast<const v4i_t*>(a[tg] + s * 256 + l * 64); }
  template <int E_STRIDE>
  __device__ __forceinline__ float4 scale(int t, int l) const { return *reinterpret_cast<const float4*>(e + t * E_STRIDE + l * 16); }
};

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
  static constexpr int kInstr = (16 * kP + 63) / 64;     // DMA instructions per run
  static constexpr int kRunBytes = kInstr * 1024;        // (a run's last instruction pads)
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
  // `w_bytes` long) into LDS at `dst` (byte address).  Pieces past the tensor's last whole one repeat it.
  __device__ __forceinline__ void request(const uint8_t* w, size_t w_bytes, size_t run_off, int sb, uint32_t dst) const {
    const uint8_t* base = w + (run_off & ~(size_t)15);
    const uint32_t mis = (uint32_t)run_off & 15u;
    const size_t left = w_bytes - (run_off & ~(size_t)15);
    const uint32_t last = (uint32_t)min(left >= 16 ? (left & ~(size_t)15) - 16 : (size_t)0, (size_t)0xfffffff0u);
#pragma unroll
    for (int i = 0; i < kInstr; ++i) {
      const uint32_t voff = min(((mis + row_off[i] + (uint32_t)(sb * SbRaw<QUANT>::kBytes)) & ~15u) + col[i], last);
      lds_dma_16(base, voff, dst + i * 1024);
    }
  }
  // A tensor that ends inside a 16-byte piece: its last bytes, which no whole piece holds, go to the slot two by two
  // (the run's `live` rows end the tensor, and `sb` is the rows' last superblock).
  __device__ __forceinline__ void patch_tail(const uint8_t* w, size_t w_bytes, size_t run_off, int live, int sb, uint8_t* run_slot) const {
    const int lane = (int)__lane_id();
    const size_t tail = w_bytes & ~(size_t)15, start = run_off + (size_t)(live - 1) * row_bytes + (size_t)sb * SbRaw<QUANT>::kBytes;
    uint8_t* p = run_slot + (live - 1) * (kP * 16) + (start & 15) + (tail - start);
    if (2 * lane < (int)(w_bytes & 15)) *reinterpret_cast<uint16_t*>(p + 2 * lane) = *reinterpret_cast<const uint16_t*>(w + tail + 2 * lane);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // the address of the lane's row inside the run's slot
  __device__ __forceinline__ const uint8_t* row_at(const uint8_t* run_slot, size_t run_off, int row, int sb) const {
    const uint32_t mis = ((uint32_t)run_off + (uint32_t)row * row_bytes + (uint32_t)(sb * SbRaw<QUANT>::kBytes)) & 15u;
    return run_slot + row * (kP * 16) + mis;
  }
};

// ---------------------------------------------------------------------------------
// Sixteen rows of two superblocks, one token: the one-token form of the core, on v_mfma_i32_16x16x64_i8.  Lane 16 q + r
// holds row r and half q & 1 of superblock q >> 1 of the pair; operand A's row m is digit m & 3 in quarter m >> 2 of K
// and zero elsewhere, so that the four result registers of a lane are the digit sums of the sixteen elements the lane
// itself unpacked.  The same exact sums and the same fp32 operations per half superblock as sb_dot's, with no operand
// rows spent on other tokens: for a single token 32 rows x 1 superblock and this shape carry the same bytes, and this
// one needs no kilobyte of zeros in LDS and fits rows of one or two superblocks (a pair is then one row or two).
// ---------------------------------------------------------------------------------
template <int QUANT>
struct PairDma {  // 29 pieces: 420 bytes at any even offset, rows four words apart modulo the banks; 35 likewise
  using Dma = SliceDma<QUANT, QUANT == kQ6K ? 29 : 35>;
  static constexpr int kSlotBytes = Dma::kRunBytes;
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
  static __device__ __forceinline__ void request(const uint8_t* run, uint32_t dst) {
    const uint32_t lane = __lane_id();
#pragma unroll
    for (int i = 0; i < kInstr; ++i) {
      const uint32_t pc = min((uint32_t)(64 * i) + lane, (uint32_t)kPieces - 1);  // (a slot's padding repeats its last piece)
      const uint32_t voff = QUANT == kQ6K ? pc * 16 : (pc / (kPairPieces + 1) * kPairPieces + min(pc % (kPairPieces + 1), (uint32_t)kPairPieces - 1)) * 16;
      lds_dma_16(run, voff, dst + i * 1024);
    }
  }
};

// Operand A and the group scales of the lane's half superblock, straight from memory.
struct PairDigits {
  v4i_t a[8];   // [4 l + s]
  float4 e[2];  // [l], s = 0..3
  // `xd`, `xe`: digits and scales of the activation superblock the lane's weights lie in
  __device__ __forceinline__ void load(const uint8_t* xd, const float* xe) {
    const int lane = (int)__lane_id(), q = lane >> 4, m = lane & 15, h = q & 1;
    const bool mine = (m >> 2) == q;
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] = v4i_t{0, 0, 0, 0};
    if (mine) {  // (one region for all eight loads)
      const uint8_t* p = xd + h * 128 + (m & 3) * 16;
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = *reinterpret_cast<const v4i_t*>(p + (j & 3) * 256 + (j >> 2) * 64);
    }
#pragma unroll
    for (int l = 0; l < 2; ++l) e[l] = reinterpret_cast<const float4*>(xe)[2 * h + l];
  }
};

template <int QUANT>
__device__ __forceinline__ float pair_dot(const SbRaw<QUANT>& r, const PairDigits& x) {
  float out = 0.0f, ws[2];
  v4i_t d[2];
  auto issue = [&](int j) __attribute__((always_inline)) {
    v4i_t c;
    sb_group(r, j & 3, j >> 2, c, ws[j & 1]);
    const v4i_t zero = {0, 0, 0, 0};
    d[j & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.a[j], c, zero, 0, 0, 0);
  };
  issue(0);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (j + 1 < 8) issue(j + 1);
    const v4i_t& dd = d[j & 1];
    const int hi = (dd[0] << 8) + dd[1], lo = (dd[2] << 8) + dd[3], s = j & 3;
    const float f = __builtin_fmaf((float)lo, 0x1p-16f, (float)hi);
    const float4& e = x.e[j >> 2];
    out = __builtin_fmaf(f, ws[j & 1] * (s == 0 ? e.x : s == 1 ? e.y : s == 2 ? e.z : e.w), out);
  }
  return out;
}

}  // namespace xabe
