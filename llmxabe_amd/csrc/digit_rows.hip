// The fp32 regimes' row contractions on the digit core (digits.h): quantized rows of one matrix, or of a gate/up pair
// with SwiGLU between them, against the tokens of a work unit.  Replaces the reference's flat and tiled fp32
// families (crates/xabe-cuda/src/kernels/moe.rs:2403-3124, :3425-3725, :4082-4227).
//
// A workgroup is eight wavefronts over the row tiles of its share (32 rows, or 16 gate and the 16 matching up rows).
// The contraction is split between the wavefronts by superblock class (superblock mod 8; rows of fewer than eight
// superblocks leave several wavefronts per class, which take the tiles in turn), so that a wavefront meets few
// superblocks of activations and reuses their digits for every tile of its share.
//
// Order of operations per (row, token), whatever the launch shape: a class sums its superblocks in order, each half of
// the wavefront its own groups; the classes are added in order, then half 0 + half 1.  A token's row is therefore the
// same bits alone, in a batch, in any mode.
#include <string.h>

#include <algorithm>

#include "decode_kernels.h"
#include "device_once.h"
#include "digit_rows.h"
#include "host_common.h"

namespace xabe {

// Digits of fp32 rows, scaled by superblocks: a wavefront per superblock; elements past the end of the row are zeros.
// (A thread per group of sixteen took 4.7 us for a single row, this 2.)
template <bool RESTS>
__global__ void __launch_bounds__(256) k_digitize_rows(const float* __restrict__ x, int K, int nsb, int rows, uint8_t* __restrict__ xd,
                                                       float* __restrict__ xe) {
  const int i = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)__lane_id();
  if (i >= rows * nsb) return;
  const int row = i / nsb, sb = i % nsb, at = sb * 64 + lane;
  const float4 f = reinterpret_cast<const float4*>(x + (size_t)row * K)[min(at, K / 4 - 1)];
  const bool in = 4 * at < K;
  const float v[4] = {in ? f.x : 0.0f, in ? f.y : 0.0f, in ? f.z : 0.0f, in ? f.w : 0.0f};
  const float scale = digitize_quads<RESTS>(v, xd + (size_t)i * kSbDigitBytes);
  if (lane == 0) xe[i] = scale;
}

// Digits of fp32 rows, scaled by groups of sixteen (what a gate/up launch writes where the scratch holds all of its rows).
__global__ void __launch_bounds__(256) k_digitize_groups(const float* __restrict__ x, int K, int nsb, int rows, uint8_t* __restrict__ xd,
                                                         float* __restrict__ xe) {
  const int i = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)__lane_id();
  if (i >= rows * nsb) return;
  const int row = i / nsb, sb = i % nsb, at = sb * 64 + lane;
  const float4 f = reinterpret_cast<const float4*>(x + (size_t)row * K)[min(at, K / 4 - 1)];
  const bool in = 4 * at < K;
  const float v[4] = {in ? f.x : 0.0f, in ? f.y : 0.0f, in ? f.z : 0.0f, in ? f.w : 0.0f};
  digitize_quads_by_group(v, xd + (size_t)i * kSbDigitBytes, xe + (size_t)i * 16);
}

// Tiles per wavefront of a dispatch block, the next one's rows in flight while one is multiplied.
constexpr int kRowsRoutedTiles = 4;

template <int MODE, int QUANT, int NM, int NT, bool TAIL>
struct RowsLds {
  static constexpr bool kFromLds = NT > 4;  // a superblock's digits are read from LDS as they are used
  // (14 pieces are enough for 210 bytes from the word boundary below)
  using Dma = SliceDma<QUANT, TAIL ? 18 : kFromLds && NM == 1 ? 14 : SbRaw<QUANT>::kPieces>;
  static constexpr int kDigits = NT * kSbDigitBytes, kScales = NM == 1 ? NT * kSbScaleBytes : 0;
  static constexpr int kPerWave = Dma::kSlotBytes + kDigits + (kFromLds ? 1 : 2) * kScales;
};

// Up to four tokens hold a superblock's digits in registers for every tile of the share.  Eight do not fit there: Q6_K
// passes of eight read them from LDS as the matrix instructions take them (the slot is busy until the last tile is done, so
// the next superblock's digits are requested only then; down's weight windows give up the piece that spreads rows over
// the banks, and scales their second buffer, to make room).  Q8_0's weight slots leave no such room: two TEAMS of four
// wavefronts, each with four tokens of its own and twice the classes; both request and unpack every row.  Dense sibling,
// eight tokens, us, two teams / one: gate/up 69.5 / 64.5, down 61 / 49.5; 32 tokens 475 / 417.
template <int MODE, int QUANT, int NM, int NT, int TEAMS, int MT, bool TAIL>
__global__ void __launch_bounds__(512, 2) k_digit_rows(RowsArgs a) {
  constexpr bool kFromLds = RowsLds<MODE, QUANT, NM, NT, TAIL>::kFromLds;
  constexpr int kTeam = 8 / TEAMS, kRounds = TEAMS, kTokens = NT * TEAMS;
  using L = RowsLds<MODE, QUANT, NM, NT, TAIL>;
  // gate and up read rows whose scales are whole superblocks', down the intermediate rows, scaled by groups
  constexpr bool kScale = NM == 2 ? kWhole : kGroups, kSwapped = kAddsGroups<QUANT, kScale> && !digits_in_one(NT);
  using Dma = typename L::Dma;
  constexpr int TG = (NT + 3) / 4;
  extern __shared__ __attribute__((aligned(16))) uint8_t s_rows[];
  const int lane = (int)__lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int valid = *a.valid_tokens - (MODE == kRowsShared ? a.unit0 : 0);
  // ---- the unit's weights and token rows
  size_t e_off = 0;
  int n_tok;
  const int* slots = nullptr;
  size_t slot0 = 0;
  if constexpr (MODE == kRowsBlock) {
    const int block = a.unit0 + (int)blockIdx.y, e = a.expert_ids[block];
    if (e < 0) return;
    e_off = (size_t)e * a.expert_bytes;
    slot0 = (size_t)block * a.block_size;
    slots = a.sorted_token_ids + slot0;
    n_tok = a.block_size;
  } else {
    slot0 = (size_t)blockIdx.y * kTokens;
    if ((int)slot0 >= valid) return;
    n_tok = min(kTokens, valid - (int)slot0);
  }
  const int sentinel = valid * a.top_k;
  // rows are counted from here among the digits
  const int d_row0 = MODE == kRowsBlock && NM == 1 ? a.unit0 * a.block_size : 0;

  // ---- this wavefront's class and tiles
  const int team = wave / kTeam, member = wave % kTeam, t0 = team * NT;             // (the team's tokens: t0 ..)
  const int classes = a.classes, side = min(classes, kTeam), per_class = kTeam / side;  // `side` classes at a time
  const int cls = member % side, sub = member / side, rounds = classes / side;        // (at most kRounds)
  const int tile_lo = (int)((long long)a.n_tiles * (int)blockIdx.x / (int)gridDim.x);
  const int n_wg = (int)((long long)a.n_tiles * ((int)blockIdx.x + 1) / (int)gridDim.x) - tile_lo;  // <= MT * per_class
  const int n_mine = (n_wg - sub + per_class - 1) / per_class;
  const int nsb = a.nsb;
  const uint32_t row_bytes = a.row_bytes;
  uint8_t* const s_zero = s_rows;
  uint8_t* const w_slot = s_rows + kZeroBytes + (size_t)wave * L::kPerWave;
  uint8_t* const d_slot = w_slot + Dma::kSlotBytes;
  uint8_t* const e_slot = d_slot + L::kDigits;
  auto lds_addr = [](uint8_t* p) __attribute__((always_inline)) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)p);
  };
  const uint32_t w_lds = lds_addr(w_slot), d_lds = lds_addr(d_slot), e_lds = lds_addr(e_slot);
  for (int i = threadIdx.x; i < kZeroBytes / 16; i += 512) reinterpret_cast<v4u_t*>(s_zero)[i] = v4u_t{0, 0, 0, 0};

  // rows of tile i of this wavefront: run 0 and run 1 (NM == 2: gate and up, the same 16 rows of each)
  const int tile_rows = NM == 2 ? 16 : a.tile_rows;
  auto tile_of = [&](int i) __attribute__((always_inline)) { return tile_lo + sub + per_class * i; };
  auto run_row = [&](int i, int u) __attribute__((always_inline)) {
    const int row = tile_of(i) * tile_rows + (NM == 2 ? 0 : 16 * u);
    return min(row, a.n_rows - 1);
  };
  Dma dma[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) dma[u].init(row_bytes, NM == 2 ? 16 : min(max(tile_rows - 16 * u, 1), 16));
  const uint64_t live_lanes = __builtin_amdgcn_ballot_w64((lane & 31) < (NM == 2 ? 32 : tile_rows));
  auto request_w = [&](int i, int sb) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
      dma[u].request(NM == 2 && u ? a.w1 : a.w0, a.w_bytes, e_off + (size_t)run_row(i, u) * row_bytes, sb, w_lds + u * Dma::kRunBytes);
  };
  // A wavefront's steps: for every superblock of its classes in order, every one of its tiles.
  struct Step {
    int sb, i, round;
  };
  auto advance = [&](Step& p) __attribute__((always_inline)) {
    if (++p.i < n_mine) return;
    p.i = 0;
    p.sb += classes;
    if (kRounds > 1 && p.sb >= nsb && ++p.round < rounds) p.sb = cls + p.round * side;
  };
  const int u_lane = (lane >> 4) & 1, r_lane = lane & 15, half = lane >> 5;

  for (int first = 0; first < n_tok; first += kTokens) {
    // the chunk's tokens: activation rows (tokens past the live ones repeat the last of them and are never stored)
    int x_row[NT], n_live = 0;
    if constexpr (MODE == kRowsBlock) {
#pragma unroll
      for (int t = 0; t < kTokens; ++t) n_live += n_live == t && first + t < n_tok && slots[first + t] < sentinel;
      if (n_live == 0) break;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int at = first + min(t0 + t, n_live - 1);
        x_row[t] = NM == 2 ? slots[at] / a.top_k : (int)slot0 + at;
      }
    } else {
      n_live = n_tok;
#pragma unroll
      for (int t = 0; t < NT; ++t) x_row[t] = (int)slot0 + min(t0 + t, n_live - 1);
    }
    int x_row_l = x_row[NT - 1];
#pragma unroll
    for (int t = 0; t < NT; ++t)
      if ((lane >> 2) == t) x_row_l = x_row[t];
    float e_now[NT], e_next[NT];  // (whole superblocks' scales)
    auto request_x = [&](int sb, int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const uint8_t* from = a.xd + ((size_t)(x_row[t] - d_row0) * nsb + sb) * kSbDigitBytes;
        lds_dma_16(from, (uint32_t)lane * 16, d_lds + t * kSbDigitBytes);
        if (lane < 32) lds_dma_16(from + 1024, (uint32_t)lane * 16, d_lds + t * kSbDigitBytes + 1024);
      }
      if constexpr (kScale == kGroups) {
        if (lane < 4 * NT)  // (64 bytes per token)
          lds_dma_16(a.xe, ((uint32_t)(x_row_l - d_row0) * nsb + sb) * kSbScaleBytes + (lane & 3) * 16, e_lds + buf * L::kScales);
      } else {
#pragma unroll
        for (int t = 0; t < NT; ++t) e_next[t] = a.xe[(size_t)x_row[t] * nsb + sb];
      }
    };

    float acc[kRounds][MT][NT];
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][i][t] = 0.0f;
    if (first == 0) __syncthreads();  // the zeros are there
    // Requests run one step ahead, rows and digits: both leave LDS for registers before the next ones are requested.
    Step now = {cls, 0, 0};
    const bool any = cls < nsb && n_mine > 0 && t0 < n_live;
    if (any) {
      request_w(0, cls);
      request_x(cls, 0);
    }
    int buf = 0;
    if (any) {
      v4i_t ax[kFromLds ? 1 : 8][TG], az[kFromLds ? 1 : kSwapped ? 8 : 4][TG];
      LdsDigits<NT, kSbDigitBytes, kSwapped> x;
#pragma unroll 1
      while (now.sb < nsb) {
        const int sb = now.sb, i = now.i;
        Step next = now;
        advance(next);
        wait_loads();
        if (i == 0) {
          if constexpr (kScale == kWhole) {
#pragma unroll
            for (int t = 0; t < NT; ++t) e_now[t] = e_next[t];
          }
          x.point(d_slot, e_slot + buf * L::kScales, s_zero);
          if constexpr (!kFromLds) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
              for (int tg = 0; tg < TG; ++tg) ax[j][tg] = x.high(j & 3, j >> 2, tg);
#pragma unroll
            for (int j = 0; j < (kSwapped ? 8 : 4) && !digits_in_one(NT); ++j)
#pragma unroll
              for (int tg = 0; tg < TG; ++tg) az[j][tg] = x.low(j & 3, j >> 2, tg);
          }
        }
        if (sb == nsb - 1 && dma[0].ends_apart(a.w_bytes)) {
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const size_t off = e_off + (size_t)run_row(i, u) * row_bytes;
            const int live = min(min(tile_rows - (NM == 2 ? 0 : 16 * u), 16), a.n_rows - (tile_of(i) * tile_rows + (NM == 2 ? 0 : 16 * u)));
            if (live >= 1 && off + (size_t)live * row_bytes == a.w_bytes) dma[u].patch_tail(NM == 2 && u ? a.w1 : a.w0, off, live, sb, w_slot + u * Dma::kRunBytes);
          }
        }
        SbRaw<QUANT> raw;
        sb_read_slot(dma[0].row_at(w_slot + u_lane * Dma::kRunBytes, e_off + (size_t)run_row(i, u_lane) * row_bytes, r_lane, sb), half, raw);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (next.sb < nsb) request_w(next.i, next.sb);
        if (!kFromLds && next.sb < nsb && next.i == 0) request_x(next.sb, buf ^ 1);
        float v[NT];
        auto x_of = [&](int t) __attribute__((always_inline)) {
          int row = x_row[0];
#pragma unroll
          for (int j = 1; j < NT; ++j) row = t == j ? x_row[j] : row;
          return a.x + (size_t)row * a.K + sb * kSbElems;
        };
        auto e_of = [&](int t, int l) __attribute__((always_inline)) {
          if constexpr (kScale == kWhole) return e_now[t];
          else return x.template scale<kSbScaleBytes>(t, l);
        };
        sb_dot<QUANT, kScale, NT, TAIL>(
            raw,
            [&](int s, int l, int tg) __attribute__((always_inline)) {
              if constexpr (kFromLds) return x.high(s, l, tg);
              else return ax[4 * l + s][tg];
            },
            [&](int s, int l, int tg) __attribute__((always_inline)) {
              if constexpr (kFromLds) return x.low(s, l, tg);
              else return az[kSwapped ? 4 * l + s : s][tg];
            },
            e_of, x_of, v, live_lanes,
            TAIL && half == 1 && (sb * kSbElems + 128) >= a.K);
#pragma unroll
        for (int m = 0; m < kRounds * MT; ++m) {  // (the sums stay in registers: the tile's own by a uniform branch, not by an index)
          if (kRounds * MT > 1 && m != now.round * MT + i) continue;
          if (kRounds * MT > 1) asm volatile("");
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[m / MT][m % MT][t] += v[t];
        }
        if (next.i == 0 && !kFromLds) buf ^= 1;
        if (kFromLds && next.sb < nsb && next.i == 0) {  // (the last tile is done with the slot)
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          request_x(next.sb, buf);
        }
        now = next;
      }
    }

    // ---- classes meet in LDS (over the slots, which everyone is done with)
    __syncthreads();
    float* const red = reinterpret_cast<float*>(s_rows + kZeroBytes);  // [class][tile of the workgroup][token][64]
    const int span = MT * per_class;
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      if (r >= rounds) continue;
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        if (i >= n_mine) continue;
#pragma unroll
        for (int t = 0; t < NT; ++t) red[(((size_t)(cls + r * side) * span + sub + per_class * i) * kTokens + t0 + t) * 64 + lane] = acc[r][i][t];
      }
    }
    __syncthreads();
    const int live_classes = min(classes, nsb);
    auto total = [&](int tl, int t, int col) __attribute__((always_inline)) {
      float h[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float* p = red + ((size_t)tl * kTokens + t) * 64 + 32 * q + col;
        float v = p[0];
        for (int c = 1; c < live_classes; ++c) v += p[(size_t)c * span * kTokens * 64];
        h[q] = v;
      }
      return h[0] + h[1];
    };
    constexpr int kCols = NM == 2 ? 16 : 32;
    for (int i = threadIdx.x; i < n_wg * kTokens * kCols; i += 512) {
      const int col = i % kCols, t = i / kCols % kTokens, tl = i / (kCols * kTokens);
      const int row = (tile_lo + tl) * tile_rows + col;
      const bool live = t < n_live && col < tile_rows && row < a.n_rows;
      size_t o_row = 0;
      float scale = 1.0f;
      if constexpr (MODE == kRowsBlock) {
        if (NM == 2) {
          o_row = slot0 + first + t;
        } else {
          const int f = slots[min(first + t, n_tok - 1)];
          o_row = live ? (size_t)f : 0;
          if (live) scale = a.topk_weights[f];
        }
      } else {
        o_row = slot0 + t;
      }
      if constexpr (NM == 2) {
        const float v = silu_f(total(tl, t, col)) * total(tl, t, col + 16);
        if (live) a.out[o_row * a.n_rows + row] = v;
        // sixteen consecutive threads hold one group of the next contraction's activations
        if (a.out_d) store_digit_group(v, row, a.out_d + o_row * a.out_nsb * kSbDigitBytes, a.out_e + o_row * a.out_nsb * 16, live);
      } else {
        const float v = scale * total(tl, t, col);
        if (live) {
          a.out[o_row * a.n_rows + row] = v;
          if (a.l_out) a.l_out[o_row * a.n_rows + row] = v + a.residual[o_row * a.n_rows + row];
        }
      }
    }
    if (first + kTokens < n_tok) __syncthreads();  // (before the next chunk's requests land in the slots)
  }
}

// ------------------------------------------------------------------------------------------------
// Routed experts, one (token, k) pair per unit: what the step-by-step entry points run below the matrix-core widths (the
// block as a whole goes through decode_block.hip, whose second and third launch have the same core) and the exact regime
// at any width.
//
// Same classes, tiles and order of operations as above on the one-token core (pair_dot: four result registers where
// sb_dot has sixteen, two workgroups on a CU), quarters 0, 1 of the wavefront on a tile's first sixteen rows and 2, 3 on
// the others.  gate/up makes the digits of its activation superblocks itself, four elements per lane, in the weight slot
// between a tile's bytes and the next one's: a launch of its own for them cost 4.7 us and its boundary.  Sums wait in LDS.
// What bounds it: at a few tokens the chain of round trips of two launches; from 13 tokens on the vector instructions of
// one unpacking per pair, and one expert read once per pair and XCD.  (k_digit_rows unpacks once per four or eight tokens
// of a dispatch block, but below the matrix-core widths most blocks hold one or two, and its registers leave one
// workgroup per CU.)
// Routed experts of the model geometry, us: one token 31 -> 16, three 33 -> 26, 45 213 -> 171 (k_digit_rows -> this).
// ------------------------------------------------------------------------------------------------
constexpr int kPairTiles = 4;  // tiles a wavefront takes at most
// From this width on the workgroups that read the same rows run side by side on one XCD (kXcdGroupMinTokens in
// decode_block.hip says why).  Shares that do not divide evenly over the eight XCDs keep the plain order: padded to eight
// they left half of the chip idle (four shares: 126 against 84 us for the down launch of 64 tokens).
constexpr size_t kPairsXcdMinTokens = 24;

// SliceDma's slot for tiles that start on 16-byte boundaries (sixteen rows of an expert are whole pieces, and so are the
// rows before them): the lane's offsets are the same for every tile of a superblock and kept in units of what windows start
// on, two to a register (longer rows, Q6_K's of 16 KB: worked out again for every tile).
template <int QUANT, int PIECES>
struct TileDma {
  static constexpr int kP = PIECES, kInstr = (16 * kP + 63) / 64, kLast = 16 * kP - 64 * (kInstr - 1);
  static constexpr int kRunBytes = 16 * kP * 16, kSlotBytes = 2 * kRunBytes;
  static constexpr uint32_t kStart = SbRaw<QUANT>::kStart, kUnit = kStart + 1;
  PackedOffsets<kInstr> off;
  static __device__ __forceinline__ uint32_t piece(int i, uint32_t row_bytes, int sb) {
    const uint32_t pc = min((uint32_t)(64 * i) + __lane_id(), 16u * kP - 1);
    return (pc / kP * row_bytes + (uint32_t)(sb * SbRaw<QUANT>::kBytes)) / kUnit + pc % kP * (16 / kUnit);
  }
  __device__ __forceinline__ void init(uint32_t row_bytes, int sb) {
#pragma unroll
    for (int i = 0; i < kInstr; ++i) off.set(i, piece(i, row_bytes, sb) & 0xffffu);
  }
  // pieces that would reach past the tensor repeat its end (Q6_K: see patch_tail; otherwise they are padding)
  __device__ __forceinline__ void request(const uint8_t* w, size_t w_bytes, size_t tile, uint32_t row_bytes, int sb, uint32_t dst) {
    const uint32_t last = (uint32_t)min(w_bytes - 16 - tile, (size_t)0xfffffff0u);
    const bool fits = row_bytes <= 65536 / 16 * kUnit - kP;  // (16 rows and a window are at most 65535 units)
    off.opaque();
#pragma unroll
    for (int i = 0; i < kInstr; ++i) {
      uint32_t o = off.get(i);
      if (__builtin_expect(!fits, 0)) o = piece(i, row_bytes, sb);
      if (i + 1 < kInstr || kLast == 64 || (int)__lane_id() < kLast) lds_dma_16(w + tile, min(o * kUnit, last), dst + i * 1024);
    }
  }
  // (the run's last row ends the tensor, and this is its last superblock; Q6_K)
  static __device__ __forceinline__ void patch_tail(const uint8_t* w, size_t w_bytes, uint8_t* run_slot) {
    patch_window<QUANT>(w, w_bytes - SbRaw<QUANT>::kBytes, run_slot + 15 * (kP * 16));
  }
  static __device__ __forceinline__ const uint8_t* row_at(const uint8_t* run_slot, uint32_t row_bytes, int row, int sb) {
    return run_slot + row * (kP * 16) + (((uint32_t)row * row_bytes + (uint32_t)(sb * SbRaw<QUANT>::kBytes)) & kStart);
  }
};

template <int QUANT, bool TAIL, bool DIRECT>
struct PairRowsLds {
  using Dma = TileDma<QUANT, TAIL ? 18 : SbRaw<QUANT>::kPieces>;
  static constexpr int kTiles = DIRECT ? 1 : kPairTiles, kSlot = DIRECT ? kSbDigitBytes : Dma::kSlotBytes;
  static constexpr size_t kSlots = 8 * (size_t)kSlot, kBytes = kSlots + (size_t)8 * kTiles * 64 * sizeof(float);
};

// DIRECT (one tile and one superblock per wavefront): its rows go straight into registers; there is no next tile whose
// bytes a slot would receive meanwhile, and the digits of gate/up are made while they are on their way.
// SQ >= 0: the workgroups past the pairs' are the shared expert's row tiles on the lanes' fp32 sums, two tiles of
// k_expert_shared each (`sh`): at a few tokens a launch of their own is mostly its boundary.
template <int QUANT, int NM, bool TAIL, bool DIRECT, int SQ>
__global__ void __launch_bounds__(512, DIRECT ? 2 : 4) k_digit_pairs(RowsArgs a, ExpertArgs sh) {
  using L = PairRowsLds<QUANT, TAIL, DIRECT>;
  using Dma = typename L::Dma;
  constexpr int kTiles = L::kTiles;
  constexpr bool kScale = NM == 2 ? kWhole : kGroups;
  constexpr int tile_rows = NM == 2 ? 16 : 32;
  extern __shared__ __attribute__((aligned(16))) uint8_t s_pair[];
  const int lane = (int)__lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if constexpr (SQ >= 0) {
    const int pair_wgs = a.units * a.shares;
    if ((int)blockIdx.x >= pair_wgs) {
      const int n = (int)blockIdx.x - pair_wgs, chunk = n / a.shared_wgs, tile = 2 * (n % a.shared_wgs) + (wave >> 2);
      switch (a.shared_rps) {
        case 8: shared_body<SQ, 1, 8, NM>(sh, chunk, tile); break;
        case 4: shared_body<SQ, 1, 4, NM>(sh, chunk, tile); break;
        case 2: shared_body<SQ, 1, 2, NM>(sh, chunk, tile); break;
        default: shared_body<SQ, 1, 1, NM>(sh, chunk, tile); break;
      }
      return;
    }
  }
  int u = (int)blockIdx.x / a.shares, share = (int)blockIdx.x % a.shares;
  if (a.xcd_units) {  // one XCD's workgroups: one share at a time, all its units next to each other
    const int xcd = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3;
    if (a.xcd_units == 1) {
      share = xcd + 8 * (j / a.units);
      u = j % a.units;
    } else {
      share = xcd % a.shares;
      u = j * a.xcd_units + xcd / a.shares;
      if (u >= a.units) return;
    }
  }
  const int pair = a.unit0 + u;
  const int id = a.topk_ids ? a.topk_ids[pair] : 0;  // (none: a single expert, a token per unit)
  const float weight = NM == 1 && a.topk_ids ? a.topk_weights[pair] : 1.0f;
  const int classes = a.classes, per_class = 8 / classes;
  const int cls = wave % classes, sub = wave / classes;
  const int tile_lo = (int)((long long)a.n_tiles * share / a.shares);
  const int n_wg = (int)((long long)a.n_tiles * (share + 1) / a.shares) - tile_lo;  // <= kTiles * per_class
  const int n_mine = (n_wg - sub + per_class - 1) / per_class;
  const int nsb = a.nsb;
  const uint32_t row_bytes = a.row_bytes;
  const bool any = cls < nsb && n_mine > 0;
  uint8_t* const w_slot = s_pair + (size_t)wave * L::kSlot;
  const uint32_t w_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)w_slot);
  float* const red = reinterpret_cast<float*>(s_pair + L::kSlots);  // [class][tile of the workgroup][half, row]
  const int run = lane >> 5, half = (lane >> 4) & 1;

  // the pair's activations, requested before its expert is known
  const size_t x_row = NM == 2 ? (size_t)(pair / a.top_k) : (size_t)pair;
  const float* const x_f = a.x + x_row * a.K;
  PairDigits<kScale> x;
  float4 quad = {0.0f, 0.0f, 0.0f, 0.0f};
  auto load_x = [&](int sb) __attribute__((always_inline)) {
    if constexpr (NM == 2) quad = reinterpret_cast<const float4*>(x_f)[min(sb * 64 + lane, a.K / 4 - 1)];
    else x.load(a.xd + ((size_t)u * nsb + sb) * kSbDigitBytes, a.xe + ((size_t)u * nsb + sb) * 16);
  };
  Dma dma;  // (its lane offsets are ready before the expert is known)
  if (any) {
    load_x(cls);
    if constexpr (!DIRECT) dma.init(row_bytes, cls);
  }
  if (pair >= *a.valid_tokens * a.top_k) return;
  const size_t e_off = (size_t)__builtin_amdgcn_readfirstlane(id) * a.expert_bytes;
  auto request_w = [&](int i, int sb) __attribute__((always_inline)) {
    const size_t tile = e_off + (size_t)(tile_lo + sub + per_class * i) * tile_rows * row_bytes;
#pragma unroll
    for (int r = 0; r < 2; ++r)
      dma.request(NM == 2 && r ? a.w1 : a.w0, a.w_bytes, NM == 2 ? tile : tile + (size_t)(16 * r) * row_bytes, row_bytes, sb,
                  w_lds + r * Dma::kRunBytes);
  };
  SbRaw<QUANT> raw;
  if constexpr (DIRECT) {
    const bool dead = TAIL && half == 1 && cls * kSbElems + 128 >= a.K;  // (a half past the row's end: its bytes are never looked at)
    const size_t row = (size_t)(tile_lo + sub) * tile_rows + (NM == 2 ? 0 : 16 * run) + (lane & 15);
    if (any) sb_read((NM == 2 && run ? a.w1 : a.w0) + e_off + row * row_bytes + (size_t)cls * SbRaw<QUANT>::kBytes, dead ? 0 : half, raw);
  } else {
    if (any) request_w(0, cls);
  }
  int sb = any ? cls : nsb, i = 0;
#pragma unroll 1
  while (sb < nsb) {
    const bool last = i + 1 >= n_mine;
    const int next_i = last ? 0 : i + 1, next_sb = last ? sb + classes : sb;
    if constexpr (!DIRECT) {
      wait_loads();
      if (QUANT == kQ6K && sb == nsb - 1) {
        const size_t end = e_off + ((size_t)(tile_lo + sub + per_class * i) * tile_rows + tile_rows) * row_bytes;
        if (end == a.w_bytes) {  // (NM == 2: both matrices end here)
          if constexpr (NM == 2) Dma::patch_tail(a.w0, a.w_bytes, w_slot);
          Dma::patch_tail(NM == 2 ? a.w1 : a.w0, a.w_bytes, w_slot + Dma::kRunBytes);
        }
      }
      sb_read_slot(Dma::row_at(w_slot + run * Dma::kRunBytes, row_bytes, lane & 15, sb), half, raw);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    if constexpr (NM == 2) {
      if (i == 0) {
        const bool in = !TAIL || sb * kSbElems + 4 * lane < a.K;
        const float q[4] = {in ? quad.x : 0.0f, in ? quad.y : 0.0f, in ? quad.z : 0.0f, in ? quad.w : 0.0f};
        x.e[0].x = digitize_quads(q, w_slot);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        x.template load<false>(w_slot, nullptr);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
    }
    if (!DIRECT && next_sb < nsb) {
      if (next_sb != sb) dma.init(row_bytes, next_sb);
      request_w(next_i, next_sb);
    }
    const float v = pair_dot<QUANT, kScale, TAIL>(
        raw, x, [&](int) __attribute__((always_inline)) { return x_f + sb * kSbElems; }, TAIL && half == 1 && sb * kSbElems + 128 >= a.K);
    float* const r = red + (((size_t)cls * (kTiles * per_class) + sub + per_class * i) * 64 + half * 32 + run * 16 + (lane & 15));
    *r = (sb == cls ? 0.0f : *r) + v;
    if (DIRECT) break;
    if (last && next_sb < nsb) load_x(next_sb);
    sb = next_sb;
    i = next_i;
  }
  __syncthreads();
  const int live_classes = min(classes, nsb), class_stride = kTiles * per_class * 64;
  auto total = [&](int tl, int col) __attribute__((always_inline)) {
    float h[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const float* p = red + (size_t)tl * 64 + 32 * q + col;
      float v = p[0];
      for (int c = 1; c < live_classes; ++c) v += p[(size_t)c * class_stride];
      h[q] = v;
    }
    return h[0] + h[1];
  };
  for (int n = threadIdx.x; n < n_wg * tile_rows; n += 512) {
    const int col = n % tile_rows, tl = n / tile_rows, row = (tile_lo + tl) * tile_rows + col;
    if constexpr (NM == 2) {
      const float v = silu_f(total(tl, col)) * total(tl, col + 16);
      a.out[(size_t)pair * a.n_rows + row] = v;
      // sixteen consecutive threads hold one group of the next contraction's activations
      if (a.out_d) store_digit_group(v, row, a.out_d + (size_t)u * a.out_nsb * kSbDigitBytes, a.out_e + (size_t)u * a.out_nsb * 16, true);
    } else {
      a.out[(size_t)pair * a.n_rows + row] = weight * total(tl, col);
    }
  }
}

// ------------------------------------------------------------------ host side
template <int QUANT, int NM, bool TAIL, bool DIRECT, int SQ>
static int pairs_go(dim3 grid, hipStream_t s, const RowsArgs* a, const ExpertArgs& sh) {
  constexpr size_t smem = PairRowsLds<QUANT, TAIL, DIRECT>::kBytes;
  if (!a) {
    XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_digit_pairs<QUANT, NM, TAIL, DIRECT, SQ>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    return XABE_OK;
  }
  hipLaunchKernelGGL((k_digit_pairs<QUANT, NM, TAIL, DIRECT, SQ>), grid, dim3(512), smem, s, *a, sh);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}
// `sq`: the format of the shared expert's rows (negative: not in this launch)
template <int QUANT, int NM, bool TAIL>
static int pairs_form(bool direct, int sq, dim3 grid, hipStream_t s, const RowsArgs* a, const ExpertArgs& sh) {
  if constexpr (!TAIL) {
    if (sq == XABE_QUANT_Q6K) return pairs_go<QUANT, NM, false, true, kQ6K>(grid, s, a, sh);
    if (sq == XABE_QUANT_Q8_0) return pairs_go<QUANT, NM, false, true, kQ8_0>(grid, s, a, sh);
  }
  return direct ? pairs_go<QUANT, NM, TAIL, true, -1>(grid, s, a, sh) : pairs_go<QUANT, NM, TAIL, false, -1>(grid, s, a, sh);
}
template <int NM>
static int pairs_quant(int quant, bool tail, bool direct, int sq, dim3 grid, hipStream_t s, const RowsArgs* a, const ExpertArgs& sh) {
  if (quant == XABE_QUANT_Q6K) return pairs_form<kQ6K, NM, false>(direct, sq, grid, s, a, sh);
  return tail ? pairs_form<kQ8_0, NM, true>(direct, sq, grid, s, a, sh) : pairs_form<kQ8_0, NM, false>(direct, sq, grid, s, a, sh);
}

template <int MODE, int QUANT, int NM, int NT, int TEAMS, int MT, bool TAIL>
static size_t rows_lds() {
  const size_t slots = (size_t)8 * RowsLds<MODE, QUANT, NM, NT, TAIL>::kPerWave, red = (size_t)8 * MT * NT * TEAMS * 64 * sizeof(float);
  return kZeroBytes + std::max(slots, red);
}

template <int MODE, int QUANT, int NM, int NT, int TEAMS, int MT, bool TAIL>
static int rows_go(dim3 grid, hipStream_t s, const RowsArgs* a) {
  const size_t smem = rows_lds<MODE, QUANT, NM, NT, TEAMS, MT, TAIL>();
  if (!a) {  // (at handle creation: the LDS limit)
    XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_digit_rows<MODE, QUANT, NM, NT, TEAMS, MT, TAIL>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    return XABE_OK;
  }
  hipLaunchKernelGGL((k_digit_rows<MODE, QUANT, NM, NT, TEAMS, MT, TAIL>), grid, dim3(512), smem, s, *a);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

template <int MODE, int NM, int NT, int TEAMS, int MT>
static int rows_quant(int quant, bool tail, dim3 grid, hipStream_t s, const RowsArgs* a) {
  if (quant == XABE_QUANT_Q6K) return rows_go<MODE, kQ6K, NM, NT, TEAMS, MT, false>(grid, s, a);
  return tail ? rows_go<MODE, kQ8_0, NM, NT, TEAMS, MT, true>(grid, s, a) : rows_go<MODE, kQ8_0, NM, NT, TEAMS, MT, false>(grid, s, a);
}

// (see k_digit_rows)
static bool one_team(int quant) { return quant == XABE_QUANT_Q6K; }

template <int NM, int MT>
static int rows_shared(int nt, int quant, bool tail, dim3 grid, hipStream_t s, const RowsArgs* a) {
  switch (nt) {
    case 1: return rows_quant<kRowsShared, NM, 1, 1, MT>(quant, tail, grid, s, a);
    case 2: return rows_quant<kRowsShared, NM, 2, 1, MT>(quant, tail, grid, s, a);
    case 4: return rows_quant<kRowsShared, NM, 4, 1, MT>(quant, tail, grid, s, a);
    default:
      // (down: the form for several tiles also where there is one: the other's compiled loop spills registers, and waits for
      // them together with the rows it has just requested)
      if (one_team(quant)) return rows_go<kRowsShared, kQ6K, NM, 8, 1, NM == 1 ? kRowsMaxTiles : MT, false>(grid, s, a);
      return rows_quant<kRowsShared, NM, 4, 2, MT>(quant, tail, grid, s, a);
  }
}

template <int NM>
static int rows_mode(int mode, int nt, int mt, int quant, bool tail, dim3 grid, hipStream_t s, const RowsArgs* a) {
  if (mode == kRowsBlock && nt > 4 && one_team(quant)) return rows_go<kRowsBlock, kQ6K, NM, 8, 1, kRowsRoutedTiles, false>(grid, s, a);
  if (mode == kRowsBlock)
    return nt == 4 ? rows_quant<kRowsBlock, NM, 4, 1, kRowsRoutedTiles>(quant, tail, grid, s, a)
                   : rows_quant<kRowsBlock, NM, 4, 2, kRowsRoutedTiles>(quant, tail, grid, s, a);
  return mt == 1 ? rows_shared<NM, 1>(nt, quant, tail, grid, s, a) : rows_shared<NM, kRowsMaxTiles>(nt, quant, tail, grid, s, a);
}

static int digit_rows_set_limits() {
  for (int q : {XABE_QUANT_Q6K, XABE_QUANT_Q8_0})
    for (bool tail : {false, true})
      for (bool direct : {false, true})
        for (int sq : {-1, (int)XABE_QUANT_Q6K, (int)XABE_QUANT_Q8_0}) {
          XABE_TRY(pairs_quant<1>(q, tail, direct, sq, dim3(1), nullptr, nullptr, ExpertArgs{}));
          XABE_TRY(pairs_quant<2>(q, tail, direct, sq, dim3(1), nullptr, nullptr, ExpertArgs{}));
        }
  for (int q : {XABE_QUANT_Q6K, XABE_QUANT_Q8_0})
    for (bool tail : {false, true})
      for (int mode : {kRowsBlock, kRowsShared})
        for (int nt : {1, 2, 4, 8})
          for (int mt : {1, kRowsMaxTiles}) {
            XABE_TRY(rows_mode<1>(mode, nt, mt, q, tail, dim3(1), nullptr, nullptr));
            XABE_TRY(rows_mode<2>(mode, nt, mt, q, tail, dim3(1), nullptr, nullptr));
          }
  return XABE_OK;
}

// at handle creation, for the current device
int digit_rows_configure() {
  static DeviceOnce once;
  int dev = 0;
  XABE_HIP_TRY(hipGetDevice(&dev));
  return once.run(dev, digit_rows_set_limits);
}

int launch_digitize_rows(hipStream_t s, const float* x, size_t K, size_t rows, uint8_t* xd, float* xe, bool rests) {
  const size_t nsb = digit_superblocks(K), n = rows * nsb;
  hipLaunchKernelGGL(rests ? k_digitize_rows<true> : k_digitize_rows<false>, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s, x, (int)K, (int)nsb, (int)rows, xd, xe);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

int launch_digitize_groups(hipStream_t s, const float* x, size_t K, size_t rows, uint8_t* xd, float* xe) {
  const size_t nsb = digit_superblocks(K), n = rows * nsb;
  hipLaunchKernelGGL(k_digitize_groups, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s, x, (int)K, (int)nsb, (int)rows, xd, xe);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

void rows_shape(RowsArgs& a, int quant, int nm) {
  const size_t be = xabe_expert_quant_block_elements(quant), bb = xabe_expert_quant_block_bytes(quant);
  a.nsb = (int)digit_superblocks((size_t)a.K);
  a.row_bytes = (uint32_t)((size_t)a.K / be * bb);
  a.out_nsb = (int)digit_superblocks((size_t)a.n_rows);
  a.classes = a.nsb > 4 ? 8 : a.nsb > 2 ? 4 : a.nsb;
  a.tile_rows = nm == 2 ? 16 : 32;
  a.n_tiles = (a.n_rows + a.tile_rows - 1) / a.tile_rows;
}


int launch_digit_pairs(const xabe_moe_kernels* k, int quant, int nm, RowsArgs a, size_t units, hipStream_t s, const ExpertArgs* shared, int shared_quant) {
  rows_shape(a, quant, nm);
  const int per_class = 8 / a.classes, wg_tiles = (a.n_tiles + per_class - 1) / per_class;
  // tiles per wavefront: as many as leave 384 workgroups (one with the shared expert: those launches have at most 32
  // pairs; us with it, one / two tiles: three tokens 28.1 / 29, four 36.1 / 37)
  int each = 1;
  while (!shared && each < kPairTiles && units * (size_t)wg_tiles >= (size_t)768 * each) each *= 2;
  a.shares = (wg_tiles + each - 1) / each;
  a.units = (int)units;
  const bool direct = each == 1 && a.nsb <= a.classes, tail = a.K % kSbElems != 0;
  // (shares that divide evenly over the XCDs, or the XCDs over them)
  a.xcd_units = k->g.max_tokens < kPairsXcdMinTokens ? 0 : a.shares % 8 == 0 ? 1 : 8 % a.shares == 0 ? 8 / a.shares : 0;
  size_t wgs = a.xcd_units > 1 ? (units + a.xcd_units - 1) / a.xcd_units * 8 : units * a.shares;
  ExpertArgs sh;
  memset(&sh, 0, sizeof(sh));
  if (shared) {
    sh = *shared;
    a.shared_rps = a.K == 256 ? 8 : a.K == 512 ? 4 : a.K == 1024 ? 2 : 1;
    sh.tile_rows = kWavesPerWg * a.shared_rps;
    a.shared_wgs = (a.n_rows / sh.tile_rows + 1) / 2;
    wgs += (k->g.max_tokens + 1) / 2 * a.shared_wgs;
  }
  const dim3 grid((unsigned)wgs);
  const int sq = shared ? shared_quant : -1;
  return nm == 2 ? pairs_quant<2>(quant, tail, direct, sq, grid, s, &a, sh) : pairs_quant<1>(quant, tail, direct, sq, grid, s, &a, sh);
}

int launch_digit_rows(const xabe_moe_kernels* k, int mode, int quant, int nm, RowsArgs a, size_t units, hipStream_t s) {
  rows_shape(a, quant, nm);
  int nt = 1;
  if (mode == kRowsShared) {
    // tokens per pass over the weights: all of them up to eight, equal passes beyond
    // (force_community: one, for comparison: the same bits)
    const size_t t = units, passes = k->force_community ? t : (t + 7) / 8, each = (t + passes - 1) / passes;
    nt = each == 1 ? 1 : each == 2 ? 2 : each <= 4 ? 4 : 8;
    units = (t + nt - 1) / nt;
  } else {
    // tokens of a block per pass over an expert's rows: four, or eight where an expert has six on average (a pass for two,
    // as it was: 256 tokens 797 us, now 530; 1024 tokens 2724, now 1553)
    nt = k->g.max_tokens * k->g.experts_per_token >= 6 * k->g.num_experts ? 8 : 4;
  }
  const bool teams = nt > 4 && !one_team(quant);
  const int per_class = std::max(1, (teams ? 4 : 8) / a.classes);  // (as the kernel has it)
  int mt = 1;
  const int tiles16 = a.n_tiles;
  unsigned grid_x = (unsigned)((tiles16 + per_class - 1) / per_class);
  if (mode == kRowsBlock) {
    // tiles per wavefront: as many as leave two workgroups per CU for the blocks a pass is likely to have
    const size_t pairs = k->g.max_tokens * k->g.experts_per_token, live = std::max(std::min(k->g.num_experts, pairs), pairs / k->g.block_size);
    int each = kRowsRoutedTiles;
    while (each > 1 && live * ((tiles16 + per_class * each - 1) / (per_class * each)) < (size_t)2 * k->num_cus) each /= 2;
    grid_x = (unsigned)((tiles16 + per_class * each - 1) / (per_class * each));
  } else if (per_class == 1 && tiles16 > k->num_cus) {
    // many tiles: one workgroup per CU with an even share of them, so that a superblock's digits serve the whole share
    mt = kRowsMaxTiles;
    const unsigned rounds = (unsigned)((tiles16 + (size_t)k->num_cus * mt - 1) / ((size_t)k->num_cus * mt));
    grid_x = rounds * (unsigned)k->num_cus;
  } else if (nm == 1 && per_class == 1 && tiles16 * 2 > k->num_cus && a.n_rows > k->num_cus) {
    // fewer tiles than CUs, but not by half: narrower tiles, one for every CU (5120 rows: 256 of 20, not 160 of 32)
    a.tile_rows = std::max(1, (a.n_rows + k->num_cus - 1) / k->num_cus);
    a.n_tiles = (a.n_rows + a.tile_rows - 1) / a.tile_rows;
    grid_x = (unsigned)a.n_tiles;
  }
  if (units > 65535) return set_error(XABE_ERR_UNSUPPORTED_GEOMETRY, "%zu work units exceed the 65535 grid.y limit of the fp32 regime", units);
  const bool tail = a.K % kSbElems != 0;
  const dim3 grid(grid_x, (unsigned)units);
  return nm == 2 ? rows_mode<2>(mode, nt, mt, quant, tail, grid, s, &a) : rows_mode<1>(mode, nt, mt, quant, tail, grid, s, &a);
}

}  // namespace xabe
