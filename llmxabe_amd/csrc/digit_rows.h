// Interface of the digit row contractions (digit_rows.hip) and the device helpers that write digits.
#pragma once

#include "digits.h"

struct xabe_moe_kernels;

namespace xabe {

struct ExpertArgs;

constexpr int kRowsBlock = 1;   // one dispatch block per unit: one expert, its run of tokens
constexpr int kRowsShared = 2;  // every live token, one matrix
constexpr int kRowsMaxTiles = 5;  // tiles of one wavefront's share whose sums it keeps in registers

inline __host__ __device__ size_t digit_superblocks(size_t K) { return (K + kSbElems - 1) / kSbElems; }

struct RowsArgs {
  const uint8_t* w0;         // gate stack (nm = 2) or the one matrix
  const uint8_t* w1;         // up stack (nm = 2)
  size_t w_bytes;            // length of each stack
  size_t expert_bytes;       // bytes of one expert in a stack (0: a single matrix)
  const float* x;            // the activation rows, [row][K] (what a marked group goes back to)
  const uint8_t* xd;         // digits of the activation rows, [row][superblock][kSbDigitBytes] (pairs' gate/up makes its own)
  const float* xe;           // their scales: gate/up [row][superblock], down [row][superblock][16] (by group; or as gate/up)
  float* out;                // [row][n_rows]
  uint8_t* out_d;            // nm = 2: digits of the output rows (null: not written)
  float* out_e;
  const float* norm;         // launch_digit_up: x is normalised with this weight, and goes to `normed`
  float* normed;
  float eps;
  const float* residual;     // with l_out: l_out = out + residual
  float* l_out;
  const int* valid_tokens;
  const int* topk_ids;
  const float* topk_weights;
  const int* sorted_token_ids;
  const int* expert_ids;
  int K, n_rows, top_k, block_size;
  int unit0;  // the first pair, block or (a single matrix, whose pointers are that token's) token of this launch; digits of
              // intermediate rows are counted from its rows
  // filled in by launch_digit_rows
  int nsb, out_nsb, classes, tile_rows, n_tiles;
  int units, shares, xcd_units;  // pairs (xcd_units: units of one share side by side, one per XCD; 0: plain order)
  int tokens;                      // launch_digit_columns: rows of a plane of `parts`
  float* parts;                    // [quarter][token][n_rows]
  int shared_wgs, shared_rps;      // pairs with the shared expert: its workgroups per chunk of two tokens, rows per step
  uint32_t row_bytes;
};

// The digits of a group that sixteen consecutive lanes (a DPP row) hold one element each: lane's value `v` is element
// `row` of the row whose digits start at xd.  Returns whether this lane's element is not held exactly.
__device__ __forceinline__ bool store_digit_lane(float v, int shift, int row, uint8_t* xd, bool live) {
  uint32_t y, z;
  bool inexact = false;
  digits_of(v, shift, y, z, inexact);
  // four lanes transpose their digits: lane q of a quad stores digit q of the quad's elements as one word, lanes 0 and 1
  // digits 4 and 5 as well
  const uint32_t y0 = dpp_i<0x00>((int)y), y1 = dpp_i<0x55>((int)y), y2 = dpp_i<0xAA>((int)y), y3 = dpp_i<0xFF>((int)y);
  const uint32_t z0 = dpp_i<0x00>((int)z), z1 = dpp_i<0x55>((int)z), z2 = dpp_i<0xAA>((int)z), z3 = dpp_i<0xFF>((int)z);
  const int gi = row >> 4, j = row & 15, q = row & 3;
  const uint32_t sel = (uint32_t)((7 - q) << 8 | (3 - q)), sel_z = (uint32_t)((5 - (q & 1)) << 8 | (1 - (q & 1)));
  const uint32_t w = __builtin_amdgcn_perm(__builtin_amdgcn_perm(y3, y2, sel), __builtin_amdgcn_perm(y1, y0, sel), 0x05040100u);
  const uint32_t wz = __builtin_amdgcn_perm(__builtin_amdgcn_perm(z3, z2, sel_z), __builtin_amdgcn_perm(z1, z0, sel_z), 0x05040100u);
  if (!live) return inexact;
  uint8_t* d = xd + (size_t)(gi >> 4) * kSbDigitBytes + digit_group_offset(gi & 15) + 16 * q + (j & ~3);
  *reinterpret_cast<uint32_t*>(d) = w;
  if (q < 2) *reinterpret_cast<uint32_t*>(d + 64) = wz;
  return inexact;
}

// The same with the scale of the group, [superblock][16] at xe.
__device__ __forceinline__ void store_digit_group(float v, int row, uint8_t* xd, float* xe, bool live) {
  const uint32_t mag = row16_max(__builtin_bit_cast(uint32_t, v) & 0x7fffffffu);
  const int e = digit_exponent(mag), gi = row >> 4;
  const bool inexact = row16_any(store_digit_lane(v, digit_shift(e), row, xd, live));
  if (live && (row & 15) == 0) xe[(gi >> 4) * 16 + scale_group_index(gi & 15)] = digit_scale(mag, e, inexact);
}

// host side
int digit_rows_configure();
// (`rests`: with negative scales, which down of `shared_whole` matrices takes: digit_rests)
int launch_digitize_rows(hipStream_t s, const float* x, size_t K, size_t rows, uint8_t* xd, float* xe, bool rests = false);
int launch_digitize_groups(hipStream_t s, const float* x, size_t K, size_t rows, uint8_t* xd, float* xe);
// `units`: dispatch blocks, or the tokens of a single matrix
int launch_digit_rows(const xabe_moe_kernels* k, int mode, int quant, int nm, RowsArgs a, size_t units, hipStream_t s);
// What the launches have in common: superblocks, classes and tiles of the matrix.
void rows_shape(RowsArgs& a, int quant, int nm);

// Down of a large single Q6_K matrix, whose activations are scaled by superblocks (digit_columns.hip): classes are superblock
// mod 32, class c in quarter c / 8; a quarter adds its classes in order, each half of the superblocks by itself, then the two
// halves; the quarters are added in pairs.  Values that the digits of a superblock do not hold exactly, a few of them, are added to
// the class ahead of the superblock's sum (digit_rests).
constexpr int kWholeQuarters = 4;
constexpr int kWholeMaxSb = 21, kWholeMinInterSb = 24;  // superblocks of the hidden size at most, of the intermediate size at least
int digit_columns_configure();
int digit_narrow_configure();
// Gate and up for one or two tokens, from a.x alone.
int launch_digit_up(const xabe_moe_kernels* k, RowsArgs a, size_t tokens, hipStream_t s);
// Down for up to four tokens.  One, and each by itself under force_community: from a.x alone; otherwise from its digits.
bool digit_down_makes(const xabe_moe_kernels* k, size_t tokens);
int launch_digit_down(const xabe_moe_kernels* k, RowsArgs a, size_t tokens, hipStream_t s);
// Any number of tokens, of such a matrix or of gate/up's.  nm = 1 with a.parts, kWholeQuarters * tokens * n_rows floats.
int launch_digit_columns(const xabe_moe_kernels* k, int nm, RowsArgs a, size_t tokens, hipStream_t s);
// One (token, k) pair per unit, straight from topk_ids: pairs a.unit0 .. a.unit0 + units - 1.  `shared`: the shared
// expert's rows of the same shape (whole superblocks, at most 2048 elements) ride along.
int launch_digit_pairs(const xabe_moe_kernels* k, int quant, int nm, RowsArgs a, size_t units, hipStream_t s,
                       const ExpertArgs* shared = nullptr, int shared_quant = -1);

}  // namespace xabe
