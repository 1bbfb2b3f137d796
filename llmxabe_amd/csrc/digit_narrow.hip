// Passes of up to four tokens over the dense sibling's large Q6_K matrices, activations scaled by whole superblocks: gate and up for
// one or two, down for up to four (more: digit_columns.hip; gate and up of three and four: k_digit_rows).  The same sums in the
// same order as there.
#include <algorithm>

#include "device_once.h"
#include "digit_rows.h"
#include "host_common.h"

namespace xabe {

constexpr int kMaxLds = 160 * 1024;

// ------------------------------------------------------------------------------------------------
// Gate, up and SwiGLU for one or two tokens, from the fp32 rows; NORM: from the residual rows, normalised on the way.
//
// A workgroup has an equal share of the rows (17408 on 256: 68 of each matrix) in tiles of up to sixteen gate rows and the
// matching up rows.  Its units, a superblock of a tile each, go to the wavefronts in turn, so that those of one moment lie side
// by side in memory and no wavefront has more than one more than another (a class of superblocks per wavefront over tiles of
// sixteen: five tiles to 64 workgroups and four to the others, two or three superblocks of each).  Sums of a unit stay in
// registers until the end, where the classes' are added in their order.
//
// The first units' rows are on their way (29 MB over the chip, 5 us) while the workgroup normalises the tokens' rows and writes
// their digits, for itself: every workgroup does that again, but the launch that does it once takes 5 us by itself.  The rows,
// the norm weight and then the digits take turns in one area of LDS.  Rows come in with each superblock's 64 pieces permuted
// (piece q at q ^ (q / 8 mod 8)): the fold's lanes read pieces eight apart.
// Hidden 5120, intermediate 17408, 146 MB (27 us at the rate of a large copy), us, k_rms_norm_digits and k_digit_rows / this: one
// token 5 and 30.1 / 30.8, two 5 and 30.7 / 33.5.  (Four tokens' digits would leave no room for the rows.)
// ------------------------------------------------------------------------------------------------
constexpr int kUpPieces = 14;  // of a row's window: 210 bytes from the word boundary below
constexpr int kUpRun = 16 * kUpPieces * 16, kUpSlot = 2 * kUpRun, kUpInstr = 2 * 4;
constexpr int kUpMaxSb = 32;  // (scales in LDS)
template <int NT>
constexpr int kUpWaves = NT == 1 ? 16 : 12;
template <int NT>
constexpr int kUpUnits = NT == 1 ? 7 : 9;  // a wavefront has at most
template <int NT>
constexpr int kUpFixed = kZeroBytes + NT * (kUpMaxSb + 1) * 4 + 16 - (NT * (kUpMaxSb + 1) * 4) % 16 + kUpWaves<NT> * kUpSlot;
constexpr int up_area(int nt) { return nt == 1 ? 2048 : 3072; }  // LDS per superblock: digits, or the rows' elements and the weight's
static_assert(kUpFixed<1> + kWholeMaxSb * up_area(1) <= kMaxLds && kUpFixed<2> + kWholeMaxSb * up_area(2) <= kMaxLds, "the rows fit beside the slots");

template <int NT, bool NORM>
__global__ void __launch_bounds__(64 * kUpWaves<NT>, kUpWaves<NT> / 4) k_digit_up(RowsArgs a) {
  constexpr int W = kUpWaves<NT>, kMine = kUpMaxSb / W + (kUpMaxSb % W != 0);
  extern __shared__ __attribute__((aligned(16))) uint8_t s_up[];
  const int lane = (int)__lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), half = lane >> 5;
  const int slot0 = (int)blockIdx.y * NT, n_tok = min(NT, *a.valid_tokens - a.unit0 - slot0);
  const int nsb = a.nsb, row_lo = (int)((long long)a.n_rows * blockIdx.x / gridDim.x);
  const int rows = (int)((long long)a.n_rows * (blockIdx.x + 1) / gridDim.x) - row_lo;
  const int tiles = (rows + 15) / 16, tile_rows = (rows + tiles - 1) / tiles, n_units = tiles * nsb;
  const uint32_t row_bytes = a.row_bytes;
  uint8_t* const s_zero = s_up;
  uint8_t* const slot = s_up + kZeroBytes + (size_t)wave * kUpSlot;
  uint8_t* const area = s_up + kZeroBytes + W * kUpSlot;
  float* const scales = reinterpret_cast<float*>(area + (size_t)nsb * up_area(NT));  // [token][kUpMaxSb], then a token's 1 / rms each
  const uint32_t slot_lds = lds_address(slot), area_lds = lds_address(area);
  const size_t off = (size_t)row_lo * row_bytes, base = off & ~(size_t)15;
  const uint32_t last = (uint32_t)min((a.w_bytes - base - 16) & ~(size_t)3, (size_t)0xfffffff0u);
  // (windows start on words; pieces that would reach past the tensor repeat its end)
  auto request = [&](int tile, int sb) __attribute__((always_inline)) {
    const int live = min(tile_rows, rows - tile * tile_rows);
    const uint32_t from = ((uint32_t)off & 15u) + (uint32_t)(tile * tile_rows) * row_bytes + (uint32_t)(sb * kQ6KBytes);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int pc = 64 * i + lane;
        if (i < 3 || lane < 32)
          lds_dma_16((u ? a.w1 : a.w0) + base, min((from + (uint32_t)min(pc / kUpPieces, live - 1) * row_bytes + (uint32_t)(pc % kUpPieces) * 16) & ~3u, last),
                     slot_lds + u * kUpRun + i * 1024);
      }
  };
  // ---- the tokens' rows (and the norm's weight), then the first unit's
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    const int sb = wave + W * j;
    if (sb >= nsb) continue;
#pragma unroll
    for (int t = 0; t < NT; ++t)
      lds_dma_16(a.x + (size_t)(slot0 + t) * a.K + sb * kSbElems, (uint32_t)(lane ^ (lane >> 3)) * 16, area_lds + (t * nsb + sb) * 1024);
    if (NORM) lds_dma_16(a.norm + sb * kSbElems, (uint32_t)lane * 16, area_lds + (NT * nsb + sb) * 1024);
  }
  int tile = wave / nsb, sb = wave % nsb;
  const bool any = n_tok > 0 && wave < n_units;
  if (any) request(tile, sb);
  for (int i = threadIdx.x; i < kZeroBytes / 16; i += 64 * W) reinterpret_cast<v4u_t*>(s_zero)[i] = v4u_t{0, 0, 0, 0};
  if (any) wait_but<kUpInstr>();
  else wait_but<0>();
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  float4 f[kMine][NT], g[kMine];
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    const int at = min(wave + W * j, nsb - 1);
#pragma unroll
    for (int t = 0; t < NT; ++t) f[j][t] = *reinterpret_cast<const float4*>(area + (t * nsb + at) * 1024 + (lane ^ (lane >> 3)) * 16);
    if (NORM) g[j] = *reinterpret_cast<const float4*>(area + (NT * nsb + at) * 1024 + lane * 16);
  }
  if (NORM && wave < NT) {  // (rms_fold's order)
    float s = 0.0f;
#pragma unroll 1
    for (int c = 0; c < a.K; c += 2048) {
      RmsRaw raw;
      const int q = c / 4 + 8 * lane;  // the lane's first piece
#pragma unroll
      for (int i = 0; i < 8; ++i)
        raw.q[i] = 4 * q < a.K ? *reinterpret_cast<const float4*>(area + wave * nsb * 1024 + (q + (i ^ (lane & 7))) * 16) : make_float4(0.f, 0.f, 0.f, 0.f);
      s = rms_fold(raw, s);
    }
    s = rms_finish(s, a.K, a.eps);
    if (lane == 0) scales[NT * kUpMaxSb + wave] = s;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    const int at = wave + W * j;
    if (at >= nsb) continue;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float inv = NORM ? scales[NT * kUpMaxSb + t] : 1.0f;
      const float4 x = f[j][t], w = g[j];
      const float v[4] = {NORM ? x.x * inv * w.x : x.x, NORM ? x.y * inv * w.y : x.y, NORM ? x.z * inv * w.z : x.z, NORM ? x.w * inv * w.w : x.w};
      const float scale = digitize_quads(v, area + (at * NT + t) * kSbDigitBytes);
      if (lane == 0) scales[t * kUpMaxSb + at] = scale;
      if (NORM && (at % (int)gridDim.x == (int)blockIdx.x || scale != scale)) {
        // (one workgroup writes it; of a marked superblock every one, to read it below)
        *reinterpret_cast<float4*>(a.normed + (size_t)(slot0 + t) * a.K + at * kSbElems + 4 * lane) = make_float4(v[0], v[1], v[2], v[3]);
        // A store of sixteen bytes still reads its registers while the next two instructions run.  The compiler keeps them apart
        // from what writes these registers next, but not across the branch that ends this block: with one instruction in
        // between a quarter of the lanes stored the next token's LDS address.
        asm volatile("s_nop 2" ::: "memory");
        if (scale != scale) wait_but<0>();
      }
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if (n_tok <= 0) return;
  LdsDigits<NT, kSbDigitBytes, false> x;
  x.point(area, area, s_zero);
  const uint32_t step = x.a[0] == s_zero ? 0 : NT * kSbDigitBytes;
  const float* const rows_f = NORM ? a.normed : a.x;
  float acc[kUpUnits<NT>][NT];
#pragma unroll
  for (int i = 0; i < kUpUnits<NT>; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[i][t] = 0.0f;
  const int r = lane & 15, run = (lane >> 4) & 1;
#pragma unroll 1
  for (int u = wave, n = 0; u < n_units; u += W, ++n) {
    wait_but<0>();
    const int live = min(tile_rows, rows - tile * tile_rows);
    if (sb == nsb - 1 && row_lo + tile * tile_rows + live == a.n_rows) {
#pragma unroll
      for (int m = 0; m < 2; ++m)
        patch_window<kQ6K>(m ? a.w1 : a.w0, a.w_bytes - kQ6KBytes, slot + m * kUpRun + (live - 1) * (kUpPieces * 16));
    }
    SbRaw<kQ6K> raw;
    sb_read_slot(slot + run * kUpRun + min(r, live - 1) * (kUpPieces * 16) +
                     (((uint32_t)off + (uint32_t)(tile * tile_rows + min(r, live - 1)) * row_bytes + (uint32_t)(sb * kQ6KBytes)) & 3u), half, raw);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int now = sb;
    sb += W;
    while (sb >= nsb) sb -= nsb, ++tile;
    if (u + W < n_units) request(tile, sb);
    const uint8_t* const digits = x.a[0] + now * step;
    float v[NT], e[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) e[t] = scales[t * kUpMaxSb + now];
    sb_dot<kQ6K, kWhole, NT>(
        raw, [&](int s, int l, int) __attribute__((always_inline)) { return *reinterpret_cast<const v4i_t*>(digits + (4 * s + l) * kGroupBytes); },
        [&](int s, int l, int tg) __attribute__((always_inline)) { return x.low(s, l, tg); },
        [&](int t, int) __attribute__((always_inline)) { return e[t]; },
        [&](int t) __attribute__((always_inline)) { return rows_f + (size_t)(slot0 + min(t, n_tok - 1)) * a.K + now * kSbElems; }, v,
        __builtin_amdgcn_ballot_w64(r < live));
#pragma unroll
    for (int i = 0; i < kUpUnits<NT>; ++i) {  // (the sums stay in registers)
      if (i != n) continue;
      asm volatile("");
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[i][t] = v[t];
    }
  }
  __syncthreads();
  float* const red = reinterpret_cast<float*>(s_up + kZeroBytes);  // [unit][token][half, matrix, row] over the slots
#pragma unroll
  for (int i = 0; i < kUpUnits<NT>; ++i) {
    if (wave + W * i >= n_units) continue;
#pragma unroll
    for (int t = 0; t < NT; ++t) red[((size_t)(wave + W * i) * NT + t) * 64 + lane] = acc[i][t];
  }
  __syncthreads();
  // four threads per row and token: half and matrix
  for (int i0 = 0; i0 < 4 * rows * n_tok; i0 += 64 * W) {
    const int i = i0 + (int)threadIdx.x, t = min(i / (4 * rows), n_tok - 1), row = min((i - t * 4 * rows) >> 2, rows - 1), q = i & 1, m = (i >> 1) & 1;
    const float* p = red + ((size_t)(row / tile_rows * nsb) * NT + t) * 64 + 32 * q + 16 * m + row % tile_rows;
    float h = 0.0f;
#pragma unroll
    for (int c = 0; c < 8; ++c) {  // (at least eight superblocks)
      float v = 0.0f;
#pragma unroll
      for (int s = 0; s < kUpMaxSb / 8; ++s)
        if (c + 8 * s < nsb) v += p[(size_t)(c + 8 * s) * NT * 64];
      h = c == 0 ? v : h + v;
    }
    h += __shfl_xor(h, 1, 64);
    const float other = __shfl_xor(h, 2, 64);
    if ((i & 3) == 0 && i < 4 * rows * n_tok) a.out[(size_t)(slot0 + t) * a.n_rows + row_lo + row] = silu_f(h) * other;
  }
}

// ------------------------------------------------------------------------------------------------
// Down for up to four tokens, the sums of the same classes in the same order.  A workgroup is a tile of rows, as many as give
// every compute unit one (5120 rows: twenty), a wavefront per superblock mod 16, or mod 8 with two superblocks on their way
// where four tokens' digits leave no room for sixteen slots (tiles of more than sixteen rows).  Bound by latency and, with two fifths of the lanes without a row, by vector
// instructions.  One token: the wavefront writes the digits of the superblock that it multiplies itself (100 instructions per
// superblock and workgroup), where a launch for them is 5 us; two tokens: twice as many instructions are more than that.
// Dense sibling's 73 MB, us, k_digit_rows with scales by group / eight wavefronts / sixteen: one token 20.3 / 22.3 / 19.3, two
// 20.5 / 21.6 / 19.4 and 5 for the digits, four 33 / 29.2 / - and 5.  Its block of three tokens 67.5 / 69.5 / 63.5.  Blocks of smaller
// matrices: three tokens, 2048 x 8192 31.1 / 33.5 / 30.6, 3072 x 8192 34.8 / 37.0 / 34.0, 4096 x 11008 47.8 / 48.9 / 44.0; four tokens 30.8 /
// 32.8 / 31.5, 34.2 / 35.7 / 35.0, 47.3 / 48.8 / 47.9.
// ------------------------------------------------------------------------------------------------
constexpr int kDownRows = 21;  // (five instructions bring 320 pieces, a row is 15)
template <int NT, int WAVES, int SLOTS, int ROWS>  // ROWS: of a tile at most
struct DigitDown {
  static constexpr int kInstr = (15 * ROWS + 63) / 64, kSlot = 15 * ROWS * 16;  // DMA instructions of a tile's superblock, 64 pieces each
  static constexpr int kPer = SLOTS * kSlot + NT * kSbDigitBytes, kLds = kZeroBytes + WAVES * kPer;
};
template <int NT, int WAVES, int SLOTS, int ROWS>
__global__ void __launch_bounds__(64 * WAVES, WAVES / 4) k_digit_down(RowsArgs a) {
  using L = DigitDown<NT, WAVES, SLOTS, ROWS>;
  constexpr bool MADE = NT == 1;
  constexpr int kTurns = 32 / WAVES, kRow = 15 * 16, kSlot = L::kSlot, kInstr = L::kInstr;
  extern __shared__ __attribute__((aligned(16))) uint8_t s_down[];
  const int lane = (int)__lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), half = lane >> 5;
  const int slot0 = (int)blockIdx.y * NT, n_tok = min(NT, *a.valid_tokens - a.unit0 - slot0);
  if (n_tok <= 0) return;
  const int nsb = a.nsb, row0 = (int)blockIdx.x * a.tile_rows, rows = min(a.tile_rows, a.n_rows - row0);
  const uint32_t row_bytes = a.row_bytes;
  uint8_t* const s_zero = s_down;
  uint8_t* const slots = s_down + kZeroBytes + (size_t)wave * L::kPer;
  uint8_t* const dig = slots + SLOTS * kSlot;
  const uint32_t slots_lds = lds_address(slots), dig_lds = lds_address(dig);
  const size_t off = (size_t)row0 * row_bytes, base = off & ~(size_t)15;
  const uint32_t last = (uint32_t)min((a.w_bytes - base - 16) & ~(size_t)3, (size_t)0xfffffff0u);
  auto offset = [&](int i, int lane) __attribute__((always_inline)) {
    const int pc = min(64 * i + lane, 15 * rows - 1);
    return ((uint32_t)off & 15u) + (uint32_t)(pc / 15) * row_bytes + (uint32_t)(pc % 15) * 16;
  };
  constexpr bool kHeldOffsets = NT < 4 || WAVES < 16;  // (no registers for them otherwise)
  uint32_t w_off[kHeldOffsets ? kInstr : 1];
  if constexpr (kHeldOffsets) {
#pragma unroll
    for (int i = 0; i < kInstr; ++i) w_off[i] = offset(i, lane);
  }
  // (windows start on words; pieces that would reach past the tensor repeat its end)
  auto request_w = [&](int sb, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kInstr; ++i)
      if (i + 1 < kInstr || lane < 15 * ROWS - 64 * i)
        lds_dma_16(a.w0 + base, min(((kHeldOffsets ? w_off[kHeldOffsets ? i : 0] : offset(i, fresh_lane())) + (uint32_t)(sb * kQ6KBytes)) & ~3u, last), slots_lds + buf * kSlot + i * 1024);
  };
  float4 f[MADE ? NT : 1];
  float e_next[NT];
  auto request_x = [&](int sb) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const size_t x_row = (size_t)(slot0 + min(t, n_tok - 1));
      if constexpr (MADE) {
        f[t] = *reinterpret_cast<const float4*>(a.x + x_row * a.K + sb * kSbElems + lane * 4);
      } else {
        const uint8_t* from = a.xd + (x_row * nsb + sb) * kSbDigitBytes;
        e_next[t] = a.xe[x_row * nsb + sb];
        lds_dma_16(from, (uint32_t)lane * 16, dig_lds + t * kSbDigitBytes);
        if (lane < 32) lds_dma_16(from + 1024, (uint32_t)lane * 16, dig_lds + t * kSbDigitBytes + 1024);
      }
    }
  };
  float acc[kTurns][NT];
#pragma unroll
  for (int q = 0; q < kTurns; ++q)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[q][t] = 0.0f;
  if (wave < nsb) {
    request_x(wave);
    request_w(wave, 0);
  }
  if (SLOTS == 2 && wave + WAVES < nsb) request_w(wave + WAVES, 1);
  for (int i = threadIdx.x; i < kZeroBytes / 16; i += 64 * WAVES) reinterpret_cast<v4u_t*>(s_zero)[i] = v4u_t{0, 0, 0, 0};
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (the zeros are there; the requests need not be)
  LdsDigits<NT, kSbDigitBytes, false> x;
  x.point(dig, dig, s_zero);
  constexpr bool kHeld = WAVES == 8 && !MADE;  // the operands leave LDS for registers, and the next digits are requested with the next rows
  v4i_t ax[kHeld ? 8 : 1], az[kHeld ? 4 : 1];
  const uint64_t live = __builtin_amdgcn_ballot_w64((lane & 31) < rows);
#pragma unroll 1
  for (int sb = wave, n = 0; sb < nsb; sb += WAVES, ++n) {
    const int buf = SLOTS == 2 ? n & 1 : 0;
    float e[NT], v[NT];
    if constexpr (MADE) {  // (the same while the rows are on their way, out of a slot of their own: no faster)
      const float q[4] = {f[0].x, f[0].y, f[0].z, f[0].w};
      e[0] = digitize_quads<true>(q, dig);
    }
    if (SLOTS == 2 && sb + WAVES < nsb) wait_but<kInstr>();
    else wait_but<0>();
    if constexpr (!MADE) {
#pragma unroll
      for (int t = 0; t < NT; ++t) e[t] = e_next[t];
    }
    uint8_t* const slot = slots + buf * kSlot;
    const int row = min((kHeldOffsets ? lane : fresh_lane()) & 31, rows - 1);
    if (sb == nsb - 1 && row0 + rows == a.n_rows) patch_window<kQ6K>(a.w0, a.w_bytes - kQ6KBytes, slot + (rows - 1) * kRow);
    const uint8_t* const bytes = slot + row * kRow + (((uint32_t)off + (uint32_t)row * row_bytes + (uint32_t)(sb * kQ6KBytes)) & 3u);
#pragma unroll
    for (int t = 0; t < NT; ++t) {  // (ahead of the superblock's sum: k_digit_columns' order)
      if (__builtin_expect(e[t] < 0.0f, 0)) {
        float4 own;
        if constexpr (MADE) own = f[t];
        else own = *reinterpret_cast<const float4*>(a.x + (size_t)(slot0 + min(t, n_tok - 1)) * a.K + sb * kSbElems + lane * 4);
        const float q4[4] = {own.x, own.y, own.z, own.w};
        float rest[4], sum = 0.0f;
        digit_rests(q4, e[t], rest);
#pragma unroll
        for (int q = 0; q < kTurns; ++q)
          if (q == n % kTurns) sum = acc[q][t];
        for_rests(rest, [&](int p, float value) __attribute__((always_inline)) {
          const float w = q6k_weight(bytes, 0, p);
          if (p >> 7 == half && __builtin_isfinite(w)) sum = __builtin_fmaf(w, value, sum);
        });
#pragma unroll
        for (int q = 0; q < kTurns; ++q)
          if (q == n % kTurns) acc[q][t] = sum;
        e[t] = -e[t];
      }
    }
    SbRaw<kQ6K> raw;
    sb_read_slot(bytes, half, raw);
    if constexpr (kHeld) {
#pragma unroll
      for (int j = 0; j < 8; ++j) ax[j] = x.high(j & 3, j >> 2, 0);
#pragma unroll
      for (int j = 0; j < 4 && !digits_in_one(NT); ++j) az[j] = x.low(j, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if ((MADE || kHeld) && sb + WAVES < nsb) request_x(sb + WAVES);
    if (sb + SLOTS * WAVES < nsb) request_w(sb + SLOTS * WAVES, buf);
    sb_dot<kQ6K, kWhole, NT>(
        raw, [&](int s, int l, int tg) __attribute__((always_inline)) { return kHeld ? ax[kHeld ? 4 * l + s : 0] : x.high(s, l, tg); },
        [&](int s, int l, int tg) __attribute__((always_inline)) { return kHeld ? az[kHeld ? s : 0] : x.low(s, l, tg); },
        [&](int t, int) __attribute__((always_inline)) { return e[t]; },
        [&](int t) __attribute__((always_inline)) {
          const float* at = a.x + (size_t)(slot0 + min(t, n_tok - 1)) * a.K + sb * kSbElems;
          asm volatile("" : "+s"(at));  // (made here, not ahead of the loop and spilled)
          return at;
        }, v, live);
#pragma unroll
    for (int q = 0; q < kTurns; ++q) {  // (the sums stay in registers)
      if (q != n % kTurns) continue;
      asm volatile("");
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[q][t] += v[t];
    }
    if (!MADE && !kHeld && sb + WAVES < nsb) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      request_x(sb + WAVES);
    }
  }
  __syncthreads();
  float* const red = reinterpret_cast<float*>(s_down + kZeroBytes);  // [class][token][half, row] over the slots
#pragma unroll
  for (int q = 0; q < kTurns; ++q)
#pragma unroll
    for (int t = 0; t < NT; ++t) red[((size_t)(WAVES * q + wave) * NT + t) * 64 + lane] = acc[q][t];
  __syncthreads();
  for (int i = threadIdx.x; i < n_tok * rows; i += 64 * WAVES) {
    const int col = i % rows, t = i / rows;
    float v[kWholeQuarters];
#pragma unroll
    for (int q = 0; q < kWholeQuarters; ++q) {
      const float* p = red + ((size_t)8 * q * NT + t) * 64 + col;
      float h0 = p[0], h1 = p[32];
#pragma unroll
      for (int c = 1; c < 8; ++c)
        if (8 * q + c < nsb) h0 += p[(size_t)c * NT * 64], h1 += p[(size_t)c * NT * 64 + 32];
      v[q] = 8 * q < nsb ? h0 + h1 : 0.0f;
    }
    const float total = (v[0] + v[1]) + (v[2] + v[3]);
    const size_t at = (size_t)(slot0 + t) * a.n_rows + row0 + col;
    a.out[at] = total;
    if (a.l_out) a.l_out[at] = total + a.residual[at];
  }
}

// ------------------------------------------------------------------ host side
template <int NT, int WAVES, int SLOTS, int ROWS = kDownRows>
static int down_limit() {
  XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_digit_down<NT, WAVES, SLOTS, ROWS>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, DigitDown<NT, WAVES, SLOTS, ROWS>::kLds));
  return XABE_OK;
}
template <int NT, bool NORM>
static int up_limit() {
  XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_digit_up<NT, NORM>), hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
  return XABE_OK;
}
static int digit_narrow_set_limits() {
  XABE_TRY((down_limit<1, 16, 1>()));
  XABE_TRY((down_limit<2, 16, 1>()));
  XABE_TRY((down_limit<3, 16, 1>()));
  XABE_TRY((down_limit<4, 8, 2>()));
  XABE_TRY((down_limit<4, 16, 1, 16>()));
  XABE_TRY((up_limit<1, false>()));
  XABE_TRY((up_limit<1, true>()));
  XABE_TRY((up_limit<2, false>()));
  return up_limit<2, true>();
}
template <int NT, int WAVES, int SLOTS, int ROWS = kDownRows>
static int down_go(RowsArgs a, int cus, unsigned passes, hipStream_t s) {
  using L = DigitDown<NT, WAVES, SLOTS, ROWS>;
  const int per_cu = (a.n_rows + cus * ROWS - 1) / (cus * ROWS);
  a.tile_rows = (a.n_rows + cus * per_cu - 1) / (cus * per_cu);
  const unsigned tiles = (unsigned)((a.n_rows + a.tile_rows - 1) / a.tile_rows);
  hipLaunchKernelGGL((k_digit_down<NT, WAVES, SLOTS, ROWS>), dim3(tiles, passes), dim3(64 * WAVES), L::kLds, s, a);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}
bool digit_down_makes(const xabe_moe_kernels* k, size_t tokens) { return tokens == 1 || k->force_community; }
int launch_digit_down(const xabe_moe_kernels* k, RowsArgs a, size_t tokens, hipStream_t s) {
  rows_shape(a, XABE_QUANT_Q6K, 1);
  if (digit_down_makes(k, tokens)) return down_go<1, 16, 1>(a, k->num_cus, (unsigned)tokens, s);
  if (tokens == 2) return down_go<2, 16, 1>(a, k->num_cus, 1, s);
  if (tokens == 3) return down_go<3, 16, 1>(a, k->num_cus, 1, s);
  return a.n_rows <= 16 * k->num_cus ? down_go<4, 16, 1, 16>(a, k->num_cus, 1, s) : down_go<4, 8, 2>(a, k->num_cus, 1, s);
}

template <int NT>
static int up_go(const RowsArgs& a, int cus, unsigned passes, hipStream_t s) {
  int shares = cus;
  auto units = [&] { return ((a.n_rows + shares - 1) / shares + 15) / 16 * a.nsb; };
  while (units() > kUpWaves<NT> * kUpUnits<NT>) shares += cus;
  const dim3 grid((unsigned)std::min(shares, a.n_rows), passes), block(64 * kUpWaves<NT>);
  const size_t lds = (size_t)(kUpFixed<NT> + a.nsb * up_area(NT));
  if (a.norm) hipLaunchKernelGGL((k_digit_up<NT, true>), grid, block, lds, s, a);
  else hipLaunchKernelGGL((k_digit_up<NT, false>), grid, block, lds, s, a);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}
int launch_digit_up(const xabe_moe_kernels* k, RowsArgs a, size_t tokens, hipStream_t s) {
  rows_shape(a, XABE_QUANT_Q6K, 2);
  return digit_down_makes(k, tokens) ? up_go<1>(a, k->num_cus, (unsigned)tokens, s) : up_go<2>(a, k->num_cus, 1, s);
}

int digit_narrow_configure() {
  static DeviceOnce once;
  int dev = 0;
  XABE_HIP_TRY(hipGetDevice(&dev));
  return once.run(dev, digit_narrow_set_limits);
}

}  // namespace xabe
