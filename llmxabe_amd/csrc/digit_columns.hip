// Passes of five to sixteen tokens over a large single Q6_K matrix (the dense sibling's), activations scaled by whole
// superblocks.
//
// Up to four tokens k_digit_rows holds a superblock's digits in registers; eight used to be read out of LDS for every 32
// rows, with six multiply-adds per (row, group, token).  Here, as in the LM head (lm_head_tiles.hip), the group's scale goes
// to the code first: two int8 planes per weight (planes.h), so that the matrix instruction carries a digit's sum through half
// a superblock, and the operands of eight tokens stay in registers for all rows of a share.
//
// A workgroup is eight wavefronts, one per class of superblocks, over the sets of sixteen rows of its share: eight gate and the
// eight matching up rows, or sixteen rows of one matrix.  34816 rows of gate and up are 2176 sets, eight or nine for each of 256
// compute units (tiles of 32 rows: four or five).  Weights come by DMA into one of two half slots per wavefront, the set after
// next requested when a set is in registers.  LDS has room for one superblock's digits of eight tokens per wavefront beside
// them: a pass of eight requests them a superblock ahead; one of sixteen keeps the second eight's there for all sets, once the
// first eight's are in registers.
//
// Gate/up: classes are superblock mod 8, the whole contraction in a workgroup, as in k_digit_rows: the same order and the same
// bits.  Down has few rows and a long contraction (5120 of 17408): a share of twenty rows would bring 12 KB of digits per
// superblock for 4 KB of weights.  There a share is four times as many rows and a quarter of the classes, which are superblock
// mod 32: quarter q of the workgroups has classes 8 q .. 8 q + 7, neighbours in memory (spread over the workgroups, and so over
// the L2s, the launch took 59 us instead of 33), and leaves sums for a small launch that adds the quarters in pairs, and the
// residual.
//
// Hidden 5120, intermediate 17408 (146 and 73 MB, 27 and 13 us at the rate of a large copy), us, k_digit_rows of eight tokens / this:
// seven tokens gate/up 57.5 / 43, down 46.5 / 31.5 and 9 for the digits and the quarters; sixteen tokens 115 / 63 and 93 / 41;
// the block 102 -> 80, 183 -> 109, 32 tokens 349 -> 190, 63 685 -> 365.  What bounds
// it: vector instructions, the unpacking at eight tokens, joining the digits' sums at sixteen.
#include <algorithm>

#include "device_once.h"
#include "digit_rows.h"
#include "host_common.h"
#include "planes.h"

namespace xabe {

using ColDma = SliceDma<kQ6K>;                                  // (its slot's layout: rows of fifteen pieces)
constexpr int kColRow = ColDma::kP * 16, kColSet = 16 * kColRow;
constexpr int kColSlots = 8 * 2 * kColSet, kColDigits = 8 * kSbDigitBytes;
constexpr int kColScales = kColSlots + 8 * kColDigits, kColLds = kColScales + 8 * 256;
template <int NO>
constexpr int kColSets = NO == 1 ? 9 : 5;                       // sets whose sums a wavefront holds
static_assert(kColSets<1> * 8 * 8 * 32 * 4 <= 8 * kColDigits && kColSets<2> * 8 * 16 * 32 * 4 <= 8 * kColDigits, "the classes' sums lie where the digits did");

// NM 2: gate and up and SwiGLU; 1: one matrix, a quarter of its classes.
template <int NM, int NO>
__global__ void __launch_bounds__(512, 2) k_digit_columns(RowsArgs a) {
  constexpr int MT = kColSets<NO>, NT = 8 * NO, kQuarters = NM == 1 ? kWholeQuarters : 1;
  extern __shared__ __attribute__((aligned(16))) uint8_t s_cols[];
  const int lane = (int)__lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4;
  const int slot0 = (int)blockIdx.y * NT, n_tok = min(NT, *a.valid_tokens - a.unit0 - slot0);
  if (n_tok <= 0) return;
  const int quarter = (int)blockIdx.x % kQuarters, share = (int)blockIdx.x / kQuarters, shares = (int)gridDim.x / kQuarters;
  const int n_sets = a.n_rows * NM / 16;
  const int set_lo = (int)((long long)n_sets * share / shares), set_hi = (int)((long long)n_sets * (share + 1) / shares);
  const int nsb = a.nsb, cls = 8 * quarter + wave;
  constexpr int kStride = 8 * kQuarters;  // from one superblock of a class to the next
  const uint32_t row_bytes = a.row_bytes;
  uint8_t* const slot = s_cols + (size_t)wave * 2 * kColSet;
  uint8_t* const dig = s_cols + kColSlots + (size_t)wave * kColDigits;
  float* const scales = reinterpret_cast<float*>(s_cols + kColScales) + 64 * wave;  // of the pass's tokens
  const uint32_t slot_lds = lds_address(slot), dig_lds = lds_address(dig), scales_lds = lds_address(scales);
  float* const red = reinterpret_cast<float*>(s_cols + kColSlots);  // [class][set][token][half, row]

  // ---- requests
  // Half a set is eight consecutive rows, 120 pieces.
  constexpr int kWInstr = 4, kXInstr = 13;  // (of a set; of eight tokens' digits with the scales)
  uint32_t w_off[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int pc = min(64 * i + lane, 8 * ColDma::kP - 1);
    w_off[i] = (uint32_t)(pc / ColDma::kP) * row_bytes + (uint32_t)(pc % ColDma::kP) * 16;
  }
  auto rows_of = [&](int u) __attribute__((always_inline)) { return NM == 2 && u ? a.w1 : a.w0; };
  auto row_of = [&](int set, int u) __attribute__((always_inline)) { return NM == 2 ? 8 * set : 16 * set + 8 * u; };
  // (windows start on words; pieces that would reach past the tensor repeat its end)
  auto request_w = [&](int set, int sb, int half_slot) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const size_t off = (size_t)row_of(set, u) * row_bytes, left = a.w_bytes - (off & ~(size_t)15);
      const uint8_t* base = rows_of(u) + (off & ~(size_t)15);
      const uint32_t from = ((uint32_t)off & 15u) + (uint32_t)(sb * kQ6KBytes), last = (uint32_t)min((left - 16) & ~(size_t)3, (size_t)0xfffffff0u);
      const uint32_t dst = slot_lds + half_slot * kColSet + u * 8 * kColRow;
      lds_dma_16(base, min((from + w_off[0]) & ~3u, last), dst);
      if (lane < 8 * ColDma::kP - 64) lds_dma_16(base, min((from + w_off[1]) & ~3u, last), dst + 1024);
    }
  };
  // Eight tokens' digits of a superblock, 96 pieces each, three instructions per two tokens; places are permuted (planes.h).
  uint32_t d_off[3][2];  // [instruction][tokens 0, 1 and 4, 5 of eight, or 2, 3 and 6, 7]
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int pc = 64 * i + lane, t = pc / 96;
      d_off[i][p] = (uint32_t)planes_piece(pc % 96, 2 * p + t) * 16;
    }
  const uint32_t e_off = (uint32_t)((slot0 + min(lane, n_tok - 1)) * nsb) * 4u;
  auto request_x = [&](int sb, int o) __attribute__((always_inline)) {
    if (o == 0) lds_dma_4(a.xe + sb, e_off, scales_lds);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int t = 8 * o + 2 * p;  // (tokens past the live ones repeat one of them)
      const uint8_t* from = a.xd + ((size_t)(slot0 + min(t, n_tok - 1)) * nsb + sb) * kSbDigitBytes;
      const uint32_t second = t + 1 < n_tok ? (uint32_t)(nsb * kSbDigitBytes) : 0;
#pragma unroll
      for (int i = 0; i < 3; ++i)
        lds_dma_16(from, d_off[i][p & 1] + (64 * i + lane >= 96 ? second : 0), dig_lds + (2 * p) * kSbDigitBytes + i * 1024);
    }
  };

  struct Step {
    int sb, set;  // (of the group set0 .. set0 + MT - 1)
  };
  const uint32_t shift[2] = {4u - 2u * (uint32_t)(g >> 1), 2u * (uint32_t)(g >> 1)};
  PlanesOperands operands;
  operands.init();
  v4i_t op[4][3];  // of the first eight tokens, [2 half + step]
  float e[NO][2];    // scales of tokens g and 4 + g of each eight
  bool dead[NO][2];  // their superblock is marked

  for (int set0 = set_lo; set0 < set_hi; set0 += MT) {
    const int sets = min(MT, set_hi - set0);
    float acc[MT][2][2 * NO];  // [set][half][token 8 o + 4 u + g as 2 o + u]
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < 2 * NO; ++t) acc[i][h][t] = 0.0f;
    if (set0 != set_lo) __syncthreads();  // (the sums before have been read)
    auto advance = [&](Step& p) __attribute__((always_inline)) {
      if (++p.set == sets) p.set = 0, p.sb += kStride;
    };
    Step now = {cls, 0}, next = now;
    advance(next);
    Step third = next;  // the one to request
    if (cls < nsb) {
      if (NO == 1) request_x(cls, 0);
      request_w(set0, cls, 0);
      if (next.sb < nsb) request_w(set0 + next.set, next.sb, 1);
      advance(third);
    }
    int half_slot = 0;
    bool ahead = false;  // digits have been requested behind the next set's rows
#pragma unroll 1
    while (now.sb < nsb) {
      const int sb = now.sb, set = set0 + now.set;
      if (now.set == 0) {
        // (eight tokens: the digits were requested ahead of these rows)
        if constexpr (NO == 1) {
          if (next.sb < nsb) wait_but<kWInstr>();
          else wait_but<0>();
        } else {
          request_x(sb, 0);
          wait_but<0>();
        }
        bool marked = false;
#pragma unroll
        for (int o = 0; o < NO; ++o)
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const float scale = scales[8 * o + 4 * u + g];
            e[o][u] = __builtin_fabsf(scale);
            dead[o][u] = scale != scale;
            marked |= !(scale >= 0.0f);
          }
        // Tokens whose superblock is marked: its halves' plain sums into the sums of every set here, and zero for what the
        // matrix instructions make of it.  (Not where a set is multiplied: a branch there cost fifty spilled registers.)
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(marked) != 0, 0)) {
#pragma unroll 1
          for (int t = 0; t < n_tok; ++t) {
            const float scale = scales[t];
            if (scale >= 0.0f) continue;
            // A few values' rests, a weight of every row for each.  (Dense block of 7 / 16 / 63 tokens, 0.4 % of SwiGLU's values
            // a thousand times the others, us: 136 / 178 / 585 where such superblocks were summed again whole, 87 / 125 / 448 like this;
            // normal rows 80 / 114 / 384, 80 / 110 / 366.)
            if (NM == 1 && scale < 0.0f) {
              const float4 f = reinterpret_cast<const float4*>(a.x + (size_t)(slot0 + t) * a.K + sb * kSbElems)[lane];
              const float q4[4] = {f.x, f.y, f.z, f.w};
              float rest[4];
              digit_rests(q4, scale, rest);
              for_rests(rest, [&](int p, float value) __attribute__((always_inline)) {
                const uint8_t* at = a.w0 + (size_t)(16 * set0) * row_bytes + (size_t)(sb * kQ6KBytes);
                uint32_t off = (uint32_t)r * row_bytes;
                asm volatile("" : "+s"(at), "+v"(off));  // (made here, not ahead of the loops and spilled)
                float own[2][2 * NO];  // zero but for the token's and the half's sums
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                  for (int u = 0; u < 2 * NO; ++u) own[h][u] = t == 4 * u + g && h == p >> 7 ? value : 0.0f;
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                  const float w = q6k_weight(at, off, p);
                  const float finite = __builtin_isfinite(w) ? w : 0.0f;
                  if (i + 1 < sets) at += 16 * row_bytes;
#pragma unroll
                  for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int u = 0; u < 2 * NO; ++u) acc[i][h][u] = __builtin_fmaf(finite, own[h][u], acc[i][h][u]);
                }
              });
              continue;
            }
            // (a lane per row and half: lane 32 h + r; the next set's rows are on their way while one is summed)
            float own[8];
            half_own(a.x + (size_t)(slot0 + t) * a.K + sb * kSbElems, lane >> 5, lane, own);
            SbRaw<kQ6K> raw[2];
            auto fetch = [&](int i) __attribute__((always_inline)) {
              int row = row_of(set0 + min(i, sets - 1), r >> 3) + (r & 7);
              asm volatile("" : "+v"(row));  // (the rows' offsets are made here, not ahead of the loops: fifty registers)
              sb_read(rows_of(r >> 3) + (size_t)row * row_bytes + (size_t)sb * kQ6KBytes, lane >> 5, raw[i & 1]);
            };
            fetch(0);
#pragma unroll
            for (int i = 0; i < MT; ++i) {
              if (i + 1 < MT) fetch(i + 1);
              if (i >= sets) continue;
              opaque(raw[i & 1]);
              const float plain = half_fp32_all<kQ6K>(raw[i & 1], own, HalfOrder{});
              const float half[2] = {__shfl(plain, r, 64), __shfl(plain, 32 + r, 64)};
#pragma unroll
              for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int u = 0; u < 2 * NO; ++u)
                  if (t == 4 * u + g) acc[i][h][u] += half[h];
            }
          }
          wait_loads();
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) operands.read(dig, j >> 1, j & 1, op[j]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if constexpr (NO == 1) {
          ahead = sb + kStride < nsb;
          if (ahead) request_x(sb + kStride, 0);
        } else {
          request_x(sb, 1);
        }
      } else if (next.sb >= nsb) {
        wait_but<0>();
      } else if (ahead) {
        wait_but<kWInstr + kXInstr>();
        ahead = false;
      } else {
        wait_but<kWInstr>();
      }
      if (sb == nsb - 1) {  // (the tensor's last bytes, which no whole piece held)
#pragma unroll
        for (int u = 0; u < 2; ++u)
          if (row_of(set, u) + 8 == a.n_rows)
            patch_window<kQ6K>(rows_of(u), a.w_bytes - kQ6KBytes, slot + half_slot * kColSet + (8 * u + 7) * kColRow);
      }
      Q6Quarter w;
      w.read(slot + half_slot * kColSet + r * kColRow,
             ((uint32_t)(row_of(set, r >> 3) + (r & 7)) * row_bytes + (uint32_t)(sb * kQ6KBytes)) & 3u, g);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (third.sb < nsb) request_w(set0 + third.set, third.sb, half_slot);
      float out[2][2 * NO];
      const float d = f16_bits_to_f32(w.d) * 0.25f;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        v4i_t hi[2], lo[2];
        w.planes(h, shift, hi, lo);
#pragma unroll
        for (int o = 0; o < NO; ++o) {
          float v[2];
          const float eo[2] = {dead[o][0] ? 0.0f : d * e[o][0], dead[o][1] ? 0.0f : d * e[o][1]};  // (d may be infinite)
          if (o == 0) {
            planes_dot(op[2 * h], op[2 * h + 1], hi, lo, eo, v);
          } else {
            if (h == 0 && now.set == 0) {  // (the second eight's digits, behind which the set after next was requested)
              if (third.sb < nsb) wait_but<kWInstr>();
              else wait_but<0>();
            }
            v4i_t x[2][3];
#pragma unroll
            for (int j = 0; j < 2; ++j) operands.read(dig, h, j, x[j]);
            planes_dot(x[0], x[1], hi, lo, eo, v);
          }
#pragma unroll
          for (int u = 0; u < 2; ++u) out[h][2 * o + u] = v[u];
        }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {  // (the sums stay in registers: the set's own by a uniform branch, not by an index)
        if (i != now.set) continue;
        asm volatile("");
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int u = 0; u < 2 * NO; ++u) acc[i][h][u] += out[h][u];
      }
      now = next;
      next = third;
      advance(third);
      half_slot ^= 1;
    }

    // ---- classes meet in LDS (over the digits, which everyone is done with)
    __syncthreads();
    if (cls < nsb) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        if (i >= sets) continue;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int u = 0; u < 2 * NO; ++u) red[((size_t)(wave * MT + i) * NT + 4 * u + g) * 32 + 16 * h + r] = acc[i][h][u];
      }
    }
    __syncthreads();
    const int live = NM == 2 ? 8 : max(1, min(8, nsb - 8 * quarter));  // wavefronts with a superblock
    auto total = [&](int tl, int t, int col) __attribute__((always_inline)) {
      float h[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float* p = red + ((size_t)tl * NT + t) * 32 + 16 * q + col;
        float part[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) part[c] = p[(size_t)min(c, live - 1) * MT * NT * 32];
        float v = part[0];
#pragma unroll
        for (int c = 1; c < 8; ++c) v = c < live ? v + part[c] : v;
        h[q] = v;
      }
      return h[0] + h[1];
    };
    constexpr int kCols = NM == 2 ? 8 : 16;
    for (int i = threadIdx.x; i < sets * n_tok * kCols; i += 512) {
      const int col = i % kCols, tl = i / kCols % sets, t = i / (kCols * sets), row = (set0 + tl) * kCols + col;
      if constexpr (NM == 2) a.out[(size_t)(slot0 + t) * a.n_rows + row] = silu_f(total(tl, t, col)) * total(tl, t, col + 8);
      else a.parts[((size_t)quarter * a.tokens + slot0 + t) * a.n_rows + row] = total(tl, t, col);
    }
  }
}

// Down's output rows, the quarters added in pairs, and with the residual.  (n_rows is a multiple of 256.)
__global__ void __launch_bounds__(256) k_columns_out(RowsArgs a) {
  const int t = blockIdx.x, j = ((int)blockIdx.y * 256 + (int)threadIdx.x) * 4;
  if (t >= min(a.tokens, *a.valid_tokens - a.unit0) || j >= a.n_rows) return;
  const size_t at = (size_t)t * a.n_rows + j, plane = (size_t)a.tokens * a.n_rows;
  const bool whole = ((reinterpret_cast<uintptr_t>(a.out) | reinterpret_cast<uintptr_t>(a.residual) | reinterpret_cast<uintptr_t>(a.l_out)) & 15) == 0;
  float4 q[kWholeQuarters], x = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < kWholeQuarters; ++i) q[i] = *reinterpret_cast<const float4*>(a.parts + i * plane + at);
  if (whole && a.l_out) x = *reinterpret_cast<const float4*>(a.residual + at);
#pragma unroll
  for (int i = 1; i < kWholeQuarters; ++i)
    if (8 * i >= a.nsb) q[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const float4 v = make_float4((q[0].x + q[1].x) + (q[2].x + q[3].x), (q[0].y + q[1].y) + (q[2].y + q[3].y),
                               (q[0].z + q[1].z) + (q[2].z + q[3].z), (q[0].w + q[1].w) + (q[2].w + q[3].w));
  if (whole) {
    *reinterpret_cast<float4*>(a.out + at) = v;
    if (a.l_out) *reinterpret_cast<float4*>(a.l_out + at) = make_float4(v.x + x.x, v.y + x.y, v.z + x.z, v.w + x.w);
    return;
  }
  const float o[4] = {v.x, v.y, v.z, v.w};
  for (int c = 0; c < 4; ++c) {  // (rows that start on any float)
    a.out[at + c] = o[c];
    if (a.l_out) a.l_out[at + c] = o[c] + a.residual[at + c];
  }
}

// ------------------------------------------------------------------ host side
template <int NM, int NO>
static int columns_limit() {
  XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_digit_columns<NM, NO>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, kColLds));
  return XABE_OK;
}
static int columns_set_limits() {
  XABE_TRY((columns_limit<1, 1>()));
  XABE_TRY((columns_limit<1, 2>()));
  XABE_TRY((columns_limit<2, 1>()));
  return columns_limit<2, 2>();
}
int digit_columns_configure() {
  static DeviceOnce once;
  int dev = 0;
  XABE_HIP_TRY(hipGetDevice(&dev));
  return once.run(dev, columns_set_limits);
}

template <int NM, int NO>
static int columns_go(const RowsArgs& a, unsigned workgroups, size_t passes, hipStream_t s) {
  hipLaunchKernelGGL((k_digit_columns<NM, NO>), dim3(workgroups, (unsigned)passes), dim3(512), kColLds, s, a);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}
// Passes of sixteen; for what is left one of eight, or up to four tokens as they go by themselves (launch_digit_rows,
// launch_digit_down; three and four tokens' gate/up there 36 us, down 29, one and two 30 and 19, a pass of eight 43 and 31, of
// sixteen 63 and 41).  Dense sibling, us, passes of sixteen only / of eight, too / these: 17 tokens 184 / 172 / 155, 20 188 / 177 /
// 166, 24 190 / 181 / -, 33 270 / 255 / 239, 49 354 / 338 / 324.
int launch_digit_columns(const xabe_moe_kernels* k, int nm, RowsArgs a, size_t tokens, hipStream_t s) {
  rows_shape(a, XABE_QUANT_Q6K, nm);
  a.tokens = (int)tokens;
  const int quarters = nm == 1 ? kWholeQuarters : 1, sets = a.n_rows * nm / 16;
  const unsigned workgroups = (unsigned)(std::min(sets, std::max(1, k->num_cus / quarters)) * quarters);
  const size_t wide = (tokens + 7) / 16, done = std::min(tokens, 16 * wide), left = tokens - done;
  const bool eight = left > 4;
  RowsArgs rest = a;  // of tokens done, done + 1, ..
  rest.unit0 += (int)done;
  rest.x += done * a.K;
  rest.xd += done * a.nsb * kSbDigitBytes;
  rest.xe += done * a.nsb;
  rest.out += done * a.n_rows;
  if (nm == 1) rest.parts += done * a.n_rows;
  if (a.l_out) rest.residual += done * a.n_rows, rest.l_out += done * a.n_rows;
  if (nm == 2) {
    if (wide) XABE_TRY((columns_go<2, 2>(a, workgroups, wide, s)));
    if (eight) return columns_go<2, 1>(rest, workgroups, 1, s);
    return left ? launch_digit_rows(k, kRowsShared, XABE_QUANT_Q6K, 2, rest, left, s) : XABE_OK;
  }
  if (wide) XABE_TRY((columns_go<1, 2>(a, workgroups, wide, s)));
  if (eight) XABE_TRY((columns_go<1, 1>(rest, workgroups, 1, s)));
  hipLaunchKernelGGL(k_columns_out, dim3((unsigned)(eight ? tokens : done), (unsigned)((a.n_rows + 1023) / 1024)), dim3(256), 0, s, a);
  XABE_HIP_TRY(hipGetLastError());
  return left && !eight ? launch_digit_down(k, rest, left, s) : XABE_OK;
}

}  // namespace xabe
