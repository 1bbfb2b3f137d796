// Matrix-core regime for prefill widths: a grouped GEMM over expert-sorted tokens that
// dequantises Q6_K / Q8_0 weights to fp16 and feeds v_mfma_f32_32x32x16_f16.
// Takes the place of the reference's int8 tensor-core family
// (crates/xabe-cuda/src/kernels/moe.rs:1316-1819, :2901-2943, :3152-3373) and of its
// int8 shared-expert path (moe.rs:6389-6476); one reader per format feeds the same
// MFMA body for gate, up and down, so there is no per-format asymmetry.
//
// One body (mfma_rows_body) in three kernels: k_mfma_rows (routed or unrouted rows), k_mfma_parts (an unrouted contraction in parts) and
// k_mfma_with_shared (routed and shared rows of a narrow pass); and k_mfma_pc, an alternative form of the routed launches (same
// bits) kept for comparison.
// Token tiles of the routed launches come from a device-built list with entries for the run of every *active* expert in
// the dispatch table: experts with no tokens cost nothing, whatever the skew.  Workgroups are persistent and stride over
// (token tile, row tile) items.
//
// Numerics.  Operands are fp16: activations rounded once; weights are (code - offset) exactly,
// times fp16(d * sc * 256) -- the 2^8 keeps small scales out of the fp16 subnormal range and
// is divided out in the epilogue.  Accumulation is fp32 in the MFMA.  Each output element
// depends only on its own token row and weight row in a fixed contraction order, so a token's
// row is the same bits wherever it sits in a batch of this regime.
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "device_common.h"
#include "device_once.h"
#include "digits.h"
#include "host_common.h"
#include "shared_along.h"
#include "tile_list.h"

namespace xabe {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kWScale = 256.0f;
constexpr float kWScaleInv = 1.0f / 256.0f;

struct MfmaArgs {
  const uint8_t* w0;            // gate (NM=2) or down (NM=1) stack
  const uint8_t* w1;            // up stack (NM=2)
  size_t expert_bytes;          // bytes of one expert in a stack
  size_t w_bytes;               // bytes of a whole stack
  const _Float16* a;            // activations, row-major [*][K]
  void* out;                    // NM=2: fp16 [*][n_rows]; NM=1: fp32 [*][n_rows]
  const int* valid_tokens;
  const int* sorted_token_ids;
  const float* topk_weights;
  const int* tile_list;         // [0] = tile count; entry i at 4+4i: expert, first slot, live rows
  int K;                        // contraction length
  int n_rows;                   // output columns per token (rows of one weight matrix)
  int top_k;
  int tile_rows;                // unrouted: token rows of a tile
  int parts;                    // k_mfma_parts: parts the contraction is in, each of whole superblocks and as long
  int resident;                 // workgroups that fit the chip
  float* planes;                // the second part's sums, [*][n_rows], the others' `plane` elements apart; the first's: `out`
  size_t plane;
};

// SwiGLU's gate in the matrix-core regime: x / (1 + e^-x) from the hardware's exp2 and reciprocal (a few ulp of
// fp32; the product is rounded to fp16 right after, 2^-11).  The fp32 regimes keep silu_f, whose bits they pin.
__device__ __forceinline__ float silu_fast(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896340736f * x));
}

__device__ __forceinline__ u32x4 pack8(uint32_t c0, uint32_t c1, half2v off, half2v s) {
  // c0, c1: eight byte codes; returns eight halfs (code + 1024 - off) * s
  uint32_t p[4];
  p[0] = __builtin_amdgcn_perm(0x64646464u, c0, 0x04010400u);
  p[1] = __builtin_amdgcn_perm(0x64646464u, c0, 0x04030402u);
  p[2] = __builtin_amdgcn_perm(0x64646464u, c1, 0x04010400u);
  p[3] = __builtin_amdgcn_perm(0x64646464u, c1, 0x04030402u);
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    half2v v = __builtin_bit_cast(half2v, p[i]);
    v = (v + off) * s;
    o[i] = __builtin_bit_cast(uint32_t, v);
  }
  u32x4 r = {o[0], o[1], o[2], o[3]};
  return r;
}

// Nothing moves across this point, in either direction, when the compiler schedules.
__device__ __forceinline__ void order_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Raw blocks in flight, in the registers the loads deliver them to.  Blocks sit at two-byte alignment (210- and
// 34-byte blocks) and the fields are read where they lie: vector memory loads on this hardware take any
// alignment, which is what the compiler itself relies on for a memcpy from a byte pointer.
// (d stays the sixteen bits the load delivers until the step that consumes it widens them: widened here, the
// compiler carries the narrow value across the item boundary and widens it right after an item's last step,
// waiting there for the loads meant to be in flight under the epilogue)
struct Q6Pend {
  uint2 qa, qb, qh, sc;
  uint16_t dh;
};
struct Q8Pend {
  u32x4 lo, hi;
  uint16_t dh;
};
template <typename T>
__device__ __forceinline__ T load_any(const uint8_t* p) {
  T v;
  __builtin_memcpy(&v, p, sizeof(T));
  return v;
}
// unit l8 of half `half` of the superblock at `blk` (field offsets: crates/xabe-kernels/src/quant.rs:725-729)
__device__ __forceinline__ void q6_issue(const uint8_t* blk, int half, int l8, Q6Pend& r) {
  r.qa = load_any<uint2>(blk + half * 64 + l8 * 8);
  r.qb = load_any<uint2>(blk + half * 64 + 32 + l8 * 8);
  r.qh = load_any<uint2>(blk + 128 + half * 32 + l8 * 8);
  r.sc = load_any<uint2>(blk + 192 + half * 8);
  r.dh = load_any<uint16_t>(blk + 208);
}
__device__ __forceinline__ void q8_issue(const uint8_t* blk, Q8Pend& r) {
  r.dh = load_any<uint16_t>(blk);
  r.lo = load_any<u32x4>(blk + 2);
  r.hi = load_any<u32x4>(blk + 18);
}

// ------------------------------------------------------------------------------------------------------------
// The same grouped GEMM with the wavefronts of a workgroup specialised: an alternative form of the routed launches,
// selected with xabe_moe_kernels_set_mfma_form(k, 2).  Same bits as k_mfma_rows, and behind it everywhere (8192 tokens:
// gate/up 461 against 357 us, down 333 against 287), so it is not the default.  It is kept
// because it is the measured answer to "would wavefronts that only dequantise beside wavefronts that only multiply
// overlap the two kinds of work": less than one wavefront that does both does, instruction by instruction.
//
// A workgroup is sixteen wavefronts with two jobs:
//   consumers (wavefronts 0-7, 2 row halves x 4 column quarters): request the activation tile three steps ahead
//     (global memory -> LDS, no registers) and multiply THIS step's tiles: 64 token rows x 64 weight rows each;
//   producers (wavefronts 8-15): keep the raw weight bytes of the next two 128-element blocks of the contraction in
//     flight and dequantise the next step's weight tile into LDS.
// A step is 64 contraction elements; the weight tile is double-buffered and the activation tile sits in a ring of
// four, so there is ONE barrier per step and nobody waits inside a step for memory it has just asked for: a
// consumer's pieces were requested three steps earlier, a producer's raw bytes two to four steps earlier, and each
// kind of wavefront counts only its own loads (the wait counters are per wavefront).
//
// The tile is 128 token rows x 256 weight rows (gate/up: 128 + 128; with 128 weight rows and an activation tile one step
// ahead the consumers waited for L2 every step: 623 us).
// Per output element the operands and the order of the matrix instructions are k_mfma_rows's (see there which 16 elements
// an instruction takes), so the bits are the same.
// A Q6_K unit (32 codes of one row: 8 at each of four places 32 elements apart) spans two steps: its raw registers
// are loaded once per 128-element block and dequantised a half at a time.
// LDS: rows of 64 halfs (128 bytes: two rows to a 256-byte line of the 64 banks), 16-byte chunks XOR-swizzled by
// pc_swizzle(row) in both tiles.  Fragment reads are served sixteen lanes at a time (sixteen rows, one chunk each): the
// eight rows of either parity must put the chunk at eight different positions, hence a permutation of (row >> 1) & 7;
// the dequantised stores (lanes = rows x the four chunks 4 jj .. 4 jj + 3) need rows two apart to differ in the
// position's high bit, hence the bit order.  (With row & 7 the bank-conflict counter showed every fragment read taking
// twice its cycles.)
constexpr int kPK = 64;        // contraction elements per step
constexpr int kPM = 128;       // token rows per tile
constexpr int kPR = 256;       // weight rows per tile
constexpr int kPARing = 4;     // activation tiles in LDS
constexpr int kPAhead = 3;     // steps between an activation tile's request and its use
constexpr int kPCWaves = 8;    // consumer wavefronts (as many producers)
constexpr int kPAInstr = kPM / (8 * kPCWaves);  // activation-piece instructions per consumer wavefront and step (1 KB = 8 rows each)

__device__ __forceinline__ int pc_swizzle(int row) { return (((row >> 1) & 1) << 2) | ((row >> 2) & 3); }

constexpr size_t mfma_pc_lds_bytes() {
  return (size_t)kPARing * kPM * kPK * sizeof(_Float16) + (size_t)2 * kPR * kPK * sizeof(_Float16) + (size_t)2 * 3 * kPM * sizeof(int);
}

// half HH (codes at places 2 HH and 2 HH + 1) of a Q6_K unit -> chunks (jj * 4 + l8) of the row's 64-element tile row
template <int HH>
__device__ __forceinline__ void q6_half_unit_to_lds(const Q6Pend& r, int l8, _Float16* brow, int swz) {
  const int is8 = (l8 >> 1) * 8;
  const uint32_t sw = (HH ? r.sc.y : r.sc.x) >> is8;
  const float d = f16_bits_to_f32(r.dh) * kWScale;
  const float ds[2] = {d * (float)(int8_t)(sw & 0xff), d * (float)(int8_t)((sw >> 16) & 0xff)};
  uint32_t c[2][2];
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const uint32_t a = w ? r.qa.y : r.qa.x, b = w ? r.qb.y : r.qb.x, h = w ? r.qh.y : r.qh.x;
    if (HH == 0) {
      c[w][0] = (a & 0x0F0F0F0Fu) | ((h << 4) & 0x30303030u);
      c[w][1] = (b & 0x0F0F0F0Fu) | ((h << 2) & 0x30303030u);
    } else {
      c[w][0] = ((a >> 4) & 0x0F0F0F0Fu) | (h & 0x30303030u);
      c[w][1] = ((b >> 4) & 0x0F0F0F0Fu) | ((h >> 2) & 0x30303030u);
    }
  }
  const half2v off = {(_Float16)-1056.0f, (_Float16)-1056.0f};  // 1024 (perm bias) + 32 (code centre)
#pragma unroll
  for (int jj = 0; jj < 2; ++jj) {
    const _Float16 sh = (_Float16)ds[jj];
    const half2v s = {sh, sh};
    *reinterpret_cast<u32x4*>(brow + ((jj * 4 + l8) ^ swz) * 8) = pack8(c[0][jj], c[1][jj], off, s);
  }
}
// a Q8_0 block -> chunks 4 blk .. 4 blk + 3 of the row's 64-element tile row
__device__ __forceinline__ void q8_block_to_lds(const Q8Pend& r, int blk, _Float16* brow, int swz) {
  const _Float16 sh = (_Float16)(f16_bits_to_f32(r.dh) * kWScale);
  const half2v s = {sh, sh};
  const half2v off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
  const uint32_t q[8] = {r.lo[0], r.lo[1], r.lo[2], r.lo[3], r.hi[0], r.hi[1], r.hi[2], r.hi[3]};
#pragma unroll
  for (int w = 0; w < 4; ++w)
    *reinterpret_cast<u32x4*>(brow + ((blk * 4 + w) ^ swz) * 8) = pack8(q[2 * w] ^ 0x80808080u, q[2 * w + 1] ^ 0x80808080u, off, s);
}

template <int QUANT, int NM>
__global__ void __launch_bounds__(1024, 4) k_mfma_pc(MfmaArgs a) {
  constexpr int kTable = 3 * kPM;
  extern __shared__ __attribute__((aligned(16))) uint8_t mfma_smem[];
  _Float16* sA = reinterpret_cast<_Float16*>(mfma_smem);          // [kPARing][128][64]
  _Float16* sB = sA + kPARing * kPM * kPK;                        // [2][256][64]
  int* sArow = reinterpret_cast<int*>(sB + 2 * kPR * kPK);        // [2][3 x 128]: activation row, output row (-1: dead), scale
  int* sOrow = sArow + kPM;
  float* sScale = reinterpret_cast<float*>(sOrow + kPM);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool producer = wave >= kPCWaves;
  const int n_ntiles = a.n_rows / (NM == 2 ? kPR / 2 : kPR);
  const int n_mtiles = a.tile_list[0];
  const int total = n_mtiles * n_ntiles;
  const int nks = a.K / kPK;  // a multiple of four (whole superblocks), at least eight (checked by the host)
  const size_t row_bytes = QUANT == kQ6K ? (size_t)(a.K / 256) * kQ6KBytes : (size_t)(a.K / 32) * kQ8Bytes;

  // which items this workgroup takes (an XCD walks a contiguous eighth of the token tiles)
  const bool by_xcd = (gridDim.x & 7u) == 0 && total >= 2 * (int)gridDim.x && n_mtiles >= 8;
  const int xcd = blockIdx.x & 7;
  const int m_lo = by_xcd ? (int)((long long)n_mtiles * xcd / 8) : 0;
  const int m_hi = by_xcd ? (int)((long long)n_mtiles * (xcd + 1) / 8) : n_mtiles;
  const int first = by_xcd ? (int)(blockIdx.x >> 3) : (int)blockIdx.x;
  const int stride = by_xcd ? (int)(gridDim.x >> 3) : (int)gridDim.x;
  const int local_total = (m_hi - m_lo) * n_ntiles;
  if (first >= local_total) return;
  const int n_items = (local_total - first + stride - 1) / stride;
  const int n_steps = n_items * nks;  // a multiple of four

  struct Item { int e, m0, rows, nt; };
  auto decode = [&](int item) __attribute__((always_inline)) {
    const int mt = m_lo + item / n_ntiles;
    typedef int int4v __attribute__((ext_vector_type(4)));
    int4v ent;
    const int* p = a.tile_list + 4 + 4 * mt;
    asm volatile("s_load_dwordx4 %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(ent) : "s"(p));
    return Item{ent.x, ent.y, ent.z, item % n_ntiles};
  };

  // ---- the first item's row tables, by the consumers' threads; everyone meets at one barrier before the steps
  if (tid < kPM) {
    const Item it = decode(first);
    int arow = 0, orow = -1;
    float sc = 1.0f;
    if (tid < it.rows) {
      const int slot = it.m0 + tid, flat = a.sorted_token_ids[slot];
      if (NM == 2) { arow = flat / a.top_k; orow = slot; }
      else { arow = slot; orow = flat; sc = a.topk_weights[flat]; }
    }
    sArow[tid] = arow;
    sOrow[tid] = orow;
    sScale[tid] = sc;
  }
  __syncthreads();

  if (producer) {
    // ================================================================= producers
    const int ptid = tid - 64 * kPCWaves;
    // Q6_K: units (row rb0 + 128 i, place l8) of the 256-row tile, two per thread, raw registers per 128-element block
    // Q8_0: one 34-byte block per thread and step: row q8row, block q8blk of the step's two
    constexpr int kUnits = QUANT == kQ6K ? 2 : 1;
    const int du = ptid & 3, rb0 = ptid >> 2;
    const int q8row = ptid & 255, q8blk = ptid >> 8;
    const ptrdiff_t up_minus_gate = NM == 2 ? a.w1 - a.w0 : 0;
    const uint8_t* wrow[kUnits];
    auto tile_row = [&](int i) __attribute__((always_inline)) { return QUANT == kQ6K ? rb0 + 128 * i : q8row; };
    auto set_wrow = [&](const Item& it) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < kUnits; ++i) {
        const int rb = tile_row(i);
        const uint8_t* base = a.w0;
        int wr;
        if (NM == 2) {
          // tile rows in groups of 32: gate columns, the matching up columns, the next 32 gate columns, ...
          const int grp = rb >> 6, which = (rb >> 5) & 1, c = rb & 31;
          base += which ? up_minus_gate : (ptrdiff_t)0;
          wr = it.nt * (kPR / 2) + grp * 32 + c;
        } else {
          wr = it.nt * kPR + rb;
        }
        wrow[i] = base + (size_t)it.e * a.expert_bytes + (size_t)wr * row_bytes;
      }
    };
    // raw bytes in flight: Q6_K two blocks of 128 (sets by block parity), Q8_0 four steps (sets by step & 3)
    constexpr int kSets = QUANT == kQ6K ? 2 : 4;
    typename std::conditional<QUANT == kQ6K, Q6Pend, Q8Pend>::type raw[kSets][kUnits];
    // the load stream runs ahead of the dequantisation, across item boundaries: its own item counter and pointers
    int ld_item = 0, ld_k = 0;  // next load: item index (0 .. n_items), and block (Q6_K) or step (Q8_0) within it
    const int ld_per_item = QUANT == kQ6K ? nks / 2 : nks;
    set_wrow(decode(first));
    auto issue = [&](auto set_c) __attribute__((always_inline)) {
      constexpr int S = decltype(set_c)::value;
      // (past the last item the stream re-reads the last item's first blocks and drops them: every fill issues
      // the same loads, so the compiler's count of what is in flight is exact on every path)
#pragma unroll
      for (int i = 0; i < kUnits; ++i) {
        if constexpr (QUANT == kQ6K) {
          // block ld_k covers superblock ld_k >> 1, half ld_k & 1
          q6_issue(wrow[i] + (size_t)(ld_k >> 1) * kQ6KBytes, ld_k & 1, du, raw[S][i]);
        } else {
          q8_issue(wrow[i] + (size_t)(ld_k * 2 + q8blk) * kQ8Bytes, raw[S][i]);
        }
      }
      if (++ld_k == ld_per_item) {
        ld_k = 0;
        if (++ld_item < n_items) set_wrow(decode(first + ld_item * stride));
      }
    };
    // fill of the weight tile of global step T (T & 3 == P): into buffer T & 1
    auto fill = [&](auto p_c) __attribute__((always_inline)) {
      constexpr int P = decltype(p_c)::value;
      _Float16* dst = sB + (P & 1) * kPR * kPK;
      if constexpr (QUANT == kQ6K) {
        constexpr int S = P >> 1, HH = P & 1;
#pragma unroll
        for (int i = 0; i < kUnits; ++i) {
          const int rb = tile_row(i);
          q6_half_unit_to_lds<HH>(raw[S][i], du, dst + rb * kPK, pc_swizzle(rb));
        }
        if constexpr (HH == 1) issue(std::integral_constant<int, S>{});  // the block after next, into the registers just released
      } else {
#pragma unroll
        for (int i = 0; i < kUnits; ++i) {
          const int rb = tile_row(i);
          q8_block_to_lds(raw[P][i], q8blk, dst + rb * kPK, pc_swizzle(rb));
        }
        issue(std::integral_constant<int, P>{});
      }
    };
    order_fence();
    issue(std::integral_constant<int, 0>{});
    order_fence();
    issue(std::integral_constant<int, 1>{});
    order_fence();
    if constexpr (QUANT != kQ6K) {
      issue(std::integral_constant<int, 2>{});
      order_fence();
      issue(std::integral_constant<int, 3>{});
      order_fence();
    }
    fill(std::integral_constant<int, 0>{});
    for (int T = 0; T < n_steps; T += 4) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      fill(std::integral_constant<int, 1>{});
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      fill(std::integral_constant<int, 2>{});
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      fill(std::integral_constant<int, 3>{});
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (T + 4 < n_steps) fill(std::integral_constant<int, 0>{});
    }
    return;
  }

  // ================================================================= consumers
  const int wm = wave >> 2, wq = wave & 3;  // row half (blocks b % 2 == wm), column quarter (64 weight rows)
  // piece q = i * kPCWaves + wave of the tile: rows 8 q .. 8 q + 7; lane: row 8 q + (lane >> 3), position lane & 7, which holds
  // chunk (lane & 7) ^ pc_swizzle(row).  Every piece is requested, dead rows' too (from the tile's first row): the count of
  // requests in flight is then the same at every step, which is what the waits below rely on.
  uint32_t arow_off[kPAInstr], arow_nxt[kPAInstr];
  auto set_arow = [&](int tb, uint32_t (&dst)[kPAInstr]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kPAInstr; ++i) {
      const int row = 8 * (i * kPCWaves + wave) + (lane >> 3), chunk = (lane & 7) ^ pc_swizzle(row);
      dst[i] = (uint32_t)sArow[tb * kTable + row] * (uint32_t)a.K + (uint32_t)chunk * 8u;
    }
  };
  const uint32_t lds_a = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)sA;
  auto move_a = [&](int slot, int ks, const uint32_t (&off)[kPAInstr]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kPAInstr; ++i) {
      const int q = i * kPCWaves + wave;
      const uint32_t voff = (off[i] + (uint32_t)ks * (uint32_t)kPK) * 2u;
      const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_a + (uint32_t)(slot * kPM * kPK * 2) + (uint32_t)q * 1024u);
      lds_dma_16(a.a, voff, dst);
    }
  };

  Item cur = decode(first);
  set_arow(0, arow_off);
#pragma unroll
  for (int i = 0; i < kPAInstr; ++i) arow_nxt[i] = arow_off[i];
  // the first kPAhead tiles (an item has at least eight steps)
#pragma unroll
  for (int t = 0; t < kPAhead; ++t) move_a(t, t, arow_off);
  int step = 0;
  for (int idx = 0; idx < n_items; ++idx) {
    const bool has_next = idx + 1 < n_items;
    const Item nxt = has_next ? decode(first + (idx + 1) * stride) : cur;
    asm volatile("" ::"s"(nxt.e), "s"(nxt.m0), "s"(nxt.rows), "s"(nxt.nt));
    const int tb = idx & 1;
    int n_flat = 0;
    float n_sc = 1.0f;

    float16v acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
    // live 32-row blocks of this consumer row: block b = 2 mi + wm holds rows 32 b ..
    const int nb = min(max((cur.rows - 32 * wm + 63) / 64, 0), 2);

#pragma unroll 1
    for (int ks = 0; ks < nks; ++ks, ++step) {
      // this step's tiles are there: my own pieces of it (requested three steps ago; memory operations retire in
      // order, so all but the two newer tiles' requests covers them) have landed, and past the barrier so have
      // everyone else's and the producers' weight tile.  Near the end of the workgroup's work fewer requests follow.
      order_fence();
      if (step + kPAhead <= n_steps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((kPAhead - 1) * kPAInstr) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      order_fence();
      // the next item's row tables, in three parts spread over this item's steps so that nothing waits for a load
      // it has just issued: flat selection index, output scale, the table itself
      if (has_next && tid < kPM) {
        if (ks == 0) n_flat = a.sorted_token_ids[nxt.m0 + min(tid, nxt.rows - 1)];
        if (NM == 1 && ks == 2) n_sc = a.topk_weights[n_flat];
        if (ks == nks - kPAhead - 2) {
          int arow = 0, orow = -1;
          if (tid < nxt.rows) {
            const int slot = nxt.m0 + tid;
            if (NM == 2) { arow = n_flat / a.top_k; orow = slot; }
            else { arow = slot; orow = n_flat; }
          }
          sArow[(tb ^ 1) * kTable + tid] = arow;
          sOrow[(tb ^ 1) * kTable + tid] = orow;
          sScale[(tb ^ 1) * kTable + tid] = n_sc;
        }
      }
      if (has_next && ks == nks - kPAhead - 1) set_arow(tb ^ 1, arow_nxt);  // (the table was written a step ago)
      // the activation tile of three steps on, into the ring slot everyone finished reading before the barrier above
      if (step + kPAhead < n_steps) {
        const int slot = (step + kPAhead) & (kPARing - 1);
        if (ks + kPAhead < nks) move_a(slot, ks + kPAhead, arow_off);
        else move_a(slot, ks + kPAhead - nks, arow_nxt);
      }
      if (nb > 0) {
        const _Float16* pa = sA + (step & (kPARing - 1)) * kPM * kPK + (32 * wm + (lane & 31)) * kPK;
        const _Float16* pb = sB + (step & 1) * kPR * kPK + (wq * 64 + (lane & 31)) * kPK;
        const int aswz = pc_swizzle(lane), khalf = lane >> 5;    // (block rows start at multiples of 32: the row's low bits are the lane's)
        const int wswz = aswz;
        half8 fa[2][2], fb[2][2];
        auto frags = [&](int kk, int set) __attribute__((always_inline)) {
          const int piece = (kk >> 1) * 4 + khalf * 2 + (kk & 1), apos = (piece ^ aswz) * 8, bpos = (piece ^ wswz) * 8;
#pragma unroll
          for (int mi = 0; mi < 2; ++mi)
            if (mi < nb) fa[set][mi] = *reinterpret_cast<const half8*>(pa + mi * 64 * kPK + apos);
#pragma unroll
          for (int ni = 0; ni < 2; ++ni) fb[set][ni] = *reinterpret_cast<const half8*>(pb + ni * 32 * kPK + bpos);
        };
        frags(0, 0);
#pragma unroll
        for (int kk = 0; kk < kPK / 16; ++kk) {
          const int c = kk & 1;
          if (kk + 1 < kPK / 16) frags(kk + 1, c ^ 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int mi = 0; mi < 2; ++mi) {
            if (mi < nb) {
#pragma unroll
              for (int ni = 0; ni < 2; ++ni)
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[c][mi], fb[c][ni], acc[mi][ni], 0, 0, 0);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }

    // epilogue: acc[mi][ni][v] is tile row 32 (2 mi + wm) + (v / 4) * 8 + (lane / 32) * 4 + v % 4, column lane % 32 of
    // the wavefront's column block ni
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) {
      if (mi >= nb) break;
      int orows[16];
      [[maybe_unused]] float scs[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = 32 * (2 * mi + wm) + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
        orows[v] = sOrow[tb * kTable + r];
        if (NM == 1) scs[v] = sScale[tb * kTable + r];
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int orow = orows[v];
        if (orow < 0) continue;
        if (NM == 2) {
          // column blocks 0 and 1: gate and the matching up columns
          const int col = cur.nt * (kPR / 2) + wq * 32 + (lane & 31);
          const float g = acc[mi][0][v] * kWScaleInv, u = acc[mi][1][v] * kWScaleInv;
          static_cast<_Float16*>(a.out)[(size_t)orow * a.n_rows + col] = (_Float16)(silu_fast(g) * u);
        } else {
#pragma unroll
          for (int ni = 0; ni < 2; ++ni) {
            const int col = cur.nt * kPR + wq * 64 + ni * 32 + (lane & 31);
            static_cast<float*>(a.out)[(size_t)orow * a.n_rows + col] = scs[v] * (acc[mi][ni][v] * kWScaleInv);
          }
        }
      }
    }
    cur = nxt;
#pragma unroll
    for (int i = 0; i < kPAInstr; ++i) arow_off[i] = arow_nxt[i];
  }
}

// ------------------------------------------------------------------------------------------------------------
// The grouped GEMM.  Each wavefront owns 32 weight rows of the tile (gate/up: 16 gate rows and the matching 16 up rows) for
// all of the tile's token rows: it brings those rows' raw bytes into an LDS slot of its own, reads its lanes' share into
// registers, makes halfs of it there, eight at a time as a matrix instruction wants them, and no dequantised weight ever
// goes through LDS or past a barrier.  The activations are what the wavefronts share: steps of 64 contraction elements go
// from global memory straight into a ring in LDS, which leaves one barrier per step.
//
// What bounds it (gate/up of the dense sibling, 2048 x 5120 -> 2 x 17408, 730 GFLOP): the matrix instructions alone take
// 450 us at the 1620 TFLOP/s that the chip holds on random data (it lowers its clock: power, not issue slots), the
// kernel 708 (65 % of its cycles are matrix instructions; 750 and 57 % before these were kept apart, see below), the kernel that
// dequantised 128 x 128 tiles through LDS 969.  Added one by one to the matrix instructions: making halfs 75 us, activation reads 48, raw weight reads 93, the
// requests 162.  Hence
//  - vector instructions between the matrix instructions, up to four of which cost one nothing (five parts of a chunk's
//    weights spread over its NB matrix instructions, w_part);
//  - tall tiles: a weight is made into a half once per 192 rows.  Eight wavefronts of 192 x 32 accumulators fill the
//    registers of a CU's SIMDs; 256 rows measured the same on the dense pass (753 us) and behind on the routed (377
//    against 357 us at 8192 tokens), 128 rows on four wavefronts and two workgroups per CU 652 us;
//  - requests made long before their use and waited for by count, never by draining ("all but the newest n", Requests).  A
//    spilled vector register would undo that (its reload waits for everything requested before it): there is none
//    (tests/test_spilled_registers.py).  With up to seven in eight of the sixteen forms the routed down launch drained
//    its queue once per item, right behind the item's stores.  Scalar registers are kept in lanes of vector ones where there
//    are too many (up to 120, wide routed down of Q6_K; 37 to 70 in k_mfma_with_shared with a Q6_K side, whose routed body alone has 27 and 34): no memory operation, but lane reads in the loop over the superblocks;
//  - what lies between the matrix instructions is kept there (w_part pins its results: the compiler moved the making of a
//    chunk's halfs behind the chunk wherever a branch followed).  Wavefronts of a SIMD that make their requests at different times
//    measured no better than all behind the matrix instructions, and cost a branch per chunk (both builds in turn, with the
//    stores below: published layout 1237 tokens 322 -> 316 us, 1400 659 -> 638 for two layers, two blocks of 8192 with the seam 1896 -> 1852,
//    dense 2048 1159 -> 1122; narrow Q8_0 launches with a workgroup or two per CU lose 1 %);
//  - LDS reads on their own width's boundary (any other takes 64 cycles), rows spread over the banks by the windows' odd
//    count of sixteen bytes, activations by pc_swizzle.
// A short contraction (down of the routed model: two superblocks) is bound by what an item costs besides: its stores, which
// the requests' waits count like any memory operation, 287 us at 8192 tokens against 333 before.
//
// Which elements a matrix instruction takes: chunk c = 2 j + m of a half superblock is elements 32 j + 16 h + 8 m + [0, 8) for
// the lanes of half h, since a lane's sixteen consecutive codes then come out of one 16-byte read; the activations'
// fragments follow (`frag`).  Per output element the order is fixed, whatever the tile.
//
// Forms: wide (six blocks of 32 rows, eight wavefronts, a workgroup per CU) and narrow (two blocks, four wavefronts, three
// workgroups per CU: a tile's start and end are then beside other tiles' steps).  Where the line lies: narrow_tiles,
// unrouted_wide.
constexpr int kSK = 64;                          // contraction elements per activation step
constexpr int kWideRows = 192;                   // token rows of a tile at most, wide form
constexpr int kWRows = 32;                       // weight rows of a wavefront
constexpr int kBlockBytes = 32 * kSK * 2;        // 32 token rows of an activation step in LDS

// A weight row's window in LDS: a superblock of 210 bytes from the word boundary below (Q6_K), four blocks of 34 bytes from a
// 16-byte boundary (Q8_0, whose superblocks of 272 bytes are taken in two windows: 136 = 8 modulo 16).
template <int QUANT, int MI>
struct WWindow {
  // (Q6_K: fourteen pieces hold it, fifteen spread the rows over the LDS banks; the narrow form has no room for the fifteenth)
  static constexpr int kPieces = QUANT == kQ6K ? (MI > 2 ? 15 : 14) : 9;
  static constexpr int kPerSb = QUANT == kQ6K ? 1 : 2, kSpan = QUANT == kQ6K ? kQ6KBytes : 4 * kQ8Bytes;
  static constexpr uint32_t kStart = QUANT == kQ6K ? 3 : 15;  // what windows start on, less one
  static constexpr int kRunBytes = 16 * kPieces * 16;         // sixteen rows
  static constexpr int kRunInstr = (16 * kPieces + 63) / 64;  // DMA instructions of a run
};

// 128 contraction elements of a weight row as a lane of half h holds them: sixteen of every thirty-two, 32 j + 16 h + [0, 16),
// which a matrix instruction's chunk c = 2 j + m takes eight at a time: 32 j + 16 h + 8 m + [0, 8).
template <int QUANT>
struct WHalf;
template <>
struct WHalf<kQ6K> {
  u32x4 qa, qb, qh;
  uint2 sc;
  uint32_t d;
};
template <>
struct WHalf<kQ8_0> {
  u32x4 q[4];
  uint32_t d[4];
};
// Reads on their own boundaries (see sb_read_slot in digits.h), words shifted by the half word that is left where rows do
// not start on words.
__device__ __forceinline__ uint2 lds_pair(const uint8_t* p) { return *static_cast<const uint2*>(__builtin_assume_aligned(p, 8)); }
__device__ __forceinline__ u32x4 lds_quad(const uint8_t* p) { return *static_cast<const u32x4*>(__builtin_assume_aligned(p, 16)); }
__device__ __forceinline__ u32x4 words_from(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3, uint32_t w4, uint32_t shift) {
  const u32x4 r = {__builtin_amdgcn_alignbit(w1, w0, shift), __builtin_amdgcn_alignbit(w2, w1, shift),
                   __builtin_amdgcn_alignbit(w3, w2, shift), __builtin_amdgcn_alignbit(w4, w3, shift)};
  return r;
}
__device__ __forceinline__ u32x4 lds_quad_shifted(const uint8_t* p, uint32_t shift) {
  const u32x4 v = lds_quad(p);
  return words_from(v[0], v[1], v[2], v[3], lds_word(p + 16), shift);
}
// half `half` of the superblock whose window lies at `p`, `mis` (0 or 2) bytes in; `even`: 0 in every lane
__device__ __forceinline__ void w_read(const uint8_t* p, uint32_t mis, bool even, int half, int h, WHalf<kQ6K>& r) {
  const uint8_t *q = p + 64 * half + 16 * h, *qh = p + 128 + 32 * half + 16 * h, *sc = p + 192 + 8 * half;
  if (even) {
    r.qa = lds_quad(q), r.qb = lds_quad(q + 32), r.qh = lds_quad(qh), r.sc = lds_pair(sc);
  } else {
    const uint32_t shift = mis << 3;
    r.qa = lds_quad_shifted(q, shift), r.qb = lds_quad_shifted(q + 32, shift), r.qh = lds_quad_shifted(qh, shift);
    const uint2 v = lds_pair(sc);
    r.sc = make_uint2(__builtin_amdgcn_alignbit(v.y, v.x, shift), __builtin_amdgcn_alignbit(lds_word(sc + 8), v.y, shift));
  }
  r.d = *reinterpret_cast<const uint16_t*>(p + mis + 208);
}
// four blocks from `p` (an 8-byte boundary): their codes start 2, 4, 6 and 0 bytes past one
__device__ __forceinline__ void w_read(const uint8_t* p, uint32_t, bool, int, int h, WHalf<kQ8_0>& r) {
  const uint8_t* q = p + 16 * h;
  const uint2 a = lds_pair(q), b = lds_pair(q + 8), c = lds_pair(q + 40), d = lds_pair(q + 72), e = lds_pair(q + 80);
  r.q[0] = words_from(a.x, a.y, b.x, b.y, lds_word(q + 16), 16);
  r.q[1] = u32x4{lds_word(q + 36), c.x, c.y, lds_word(q + 48)};
  r.q[2] = words_from(lds_word(q + 68), d.x, d.y, e.x, e.y, 16);
  const uint2 f = lds_pair(q + 104), g = lds_pair(q + 112);
  r.q[3] = u32x4{f.x, f.y, g.x, g.y};
#pragma unroll
  for (int j = 0; j < 4; ++j) r.d[j] = *reinterpret_cast<const uint16_t*>(p + 34 * j);
}
// fp16(d sc 2^8) of the lane's sixteens 2 p and 2 p + 1.  `pick`: where the lane finds their scales among four bytes
__device__ __forceinline__ uint32_t w_scale_bytes(int h) { return h ? 0x04030401u : 0x04020400u; }
__device__ __forceinline__ half2v w_scales(const WHalf<kQ6K>& r, int p, uint32_t pick) {
  half2v s = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, (p ? r.sc.y : r.sc.x) ^ 0x80808080u, pick));
  s = s + half2v{(_Float16)-1152.0f, (_Float16)-1152.0f};
  s = s * half2v{(_Float16)kWScale, (_Float16)kWScale};
  const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t)r.d);
  return s * half2v{d, d};
}
__device__ __forceinline__ half2v w_scales(const WHalf<kQ8_0>& r, int p, uint32_t) {
  const half2v d = {__builtin_bit_cast(_Float16, (uint16_t)r.d[2 * p]), __builtin_bit_cast(_Float16, (uint16_t)r.d[2 * p + 1])};
  return d * half2v{(_Float16)kWScale, (_Float16)kWScale};
}
// The lane's eight weights of chunk c in five parts of a few instructions each, for a caller that puts matrix instructions
// between them: part 0 the scales of four chunks, 1 and 2 four codes each, 3 and 4 those as halfs.
struct WChunk {
  half2v scales;
  uint32_t code[2], out[4];
};
constexpr int kWParts = 5;
template <int C>
__device__ __forceinline__ uint32_t w_codes(const WHalf<kQ6K>& r, int w) {
  constexpr int j = C >> 1, m = C & 1;
  const uint32_t a = r.qa[2 * m + w], b = r.qb[2 * m + w], q = r.qh[2 * m + w];
  return j == 0   ? (a & 0x0F0F0F0Fu) | ((q << 4) & 0x30303030u)
         : j == 1 ? (b & 0x0F0F0F0Fu) | ((q << 2) & 0x30303030u)
         : j == 2 ? ((a >> 4) & 0x0F0F0F0Fu) | (q & 0x30303030u)
                  : ((b >> 4) & 0x0F0F0F0Fu) | ((q >> 2) & 0x30303030u);
}
template <int C>
__device__ __forceinline__ uint32_t w_codes(const WHalf<kQ8_0>& r, int w) {
  return r.q[C >> 1][2 * (C & 1) + w] ^ 0x80808080u;
}
template <int C, int PART, int QUANT>
__device__ __forceinline__ void w_part(const WHalf<QUANT>& r, uint32_t pick, WChunk& k) {
  if constexpr (PART == 0) {
    if constexpr ((C & 3) == 0) {
      k.scales = w_scales(r, C >> 2, pick);
      asm volatile("" : "+v"(k.scales));
    }
  } else if constexpr (PART <= 2) {
    k.code[PART - 1] = w_codes<C>(r, PART - 1);
    asm volatile("" : "+v"(k.code[PART - 1]));
  } else {
    constexpr int w = PART - 3;
    const _Float16 off = QUANT == kQ6K ? (_Float16)-1056.0f : (_Float16)-1152.0f;  // (1024 of the byte's placing, and the codes' centre)
    const _Float16 s = (C >> 1) & 1 ? k.scales.y : k.scales.x;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      half2v v = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, k.code[w], i ? 0x04030402u : 0x04010400u));
      v = (v + half2v{off, off}) * half2v{s, s};
      k.out[2 * w + i] = __builtin_bit_cast(uint32_t, v);
    }
    asm volatile("" : "+v"(k.out[2 * w]), "+v"(k.out[2 * w + 1]));
  }
}
template <int C, int PART = 0, int QUANT>
__device__ __forceinline__ void w_parts_from(const WHalf<QUANT>& r, uint32_t pick, WChunk& k) {
  w_part<C, PART>(r, pick, k);
  if constexpr (PART + 1 < kWParts) w_parts_from<C, PART + 1>(r, pick, k);
}
__device__ __forceinline__ half8 w_halfs(const WChunk& k) {
  const u32x4 v = {k.out[0], k.out[1], k.out[2], k.out[3]};
  return __builtin_bit_cast(half8, v);
}

// All but the newest N memory operations of this wavefront have completed.
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// lds_dma_16 for the lanes of `lanes`, which may be none: the instruction is issued and counted all the same, so that the
// number of memory operations in flight does not depend on the data.  (Every lane of the wavefront is active here.)
__device__ __forceinline__ void lds_dma_16_lanes(const void* base, uint32_t voff, uint32_t dst, uint32_t lanes_lo, uint32_t lanes_hi) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %2\n\ts_mov_b32 exec_lo, %3\n\ts_mov_b32 exec_hi, %4\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(voff),
               "s"(base), "s"(__builtin_amdgcn_readfirstlane(dst)), "s"(__builtin_amdgcn_readfirstlane(lanes_lo)),
               "s"(__builtin_amdgcn_readfirstlane(lanes_hi)) : "memory", "m0");
#pragma clang diagnostic pop
}
template <int MI>
constexpr int kRing = MI > 2 ? 4 : 3;  // steps of activations in LDS
// The requests of a superblock's sixteen chunks, in order.  Activations: after the barrier that frees a place in the ring
// (chunks 3, 7, 11, 15), the step that goes there, PI instructions.  Weights: behind them from the barrier on that follows the
// read that empties the slot, two instructions per chunk.  Memory operations complete in order, so a wait for one is
// "all but those made after it".
template <int QUANT, int PI>
struct Requests {
  static constexpr int a_at(int c) { return (c & 3) == 3 ? PI : 0; }
  static constexpr int w_at(int c) { return QUANT == kQ6K ? ((c + 1) & 15) < 4 ? 2 : 0 : ((c + 1) & 7) < 3 ? 2 : 0; }
  // how many are made in chunks [lo, hi)
  static constexpr int between(int lo, int hi) {
    int n = 0;
    for (int c = lo; c < hi; ++c) n += a_at(c + 16) + w_at(c + 16);
    return n;
  }
  // at the start of chunk c: those made after the activations of chunk r, and after the latest weights
  static constexpr int after_a(int r, int c) { return w_at(r + 16) + between(r + 1, c); }
  static constexpr int after_w(int c) {
    int last = c - 1;
    while (w_at(last + 16) == 0) --last;
    return between(last + 1, c);
  }
};
template <int QUANT, int MI, int WAVES>
constexpr size_t mfma_rows_lds() {
  return (size_t)kRing<MI> * MI * kBlockBytes + (size_t)WAVES * 2 * WWindow<QUANT, MI>::kRunBytes + (size_t)2 * 32 * MI * sizeof(int);
}
template <int MI, int WAVES>
constexpr int kWgsPerCu = MI > 2 ? 1 : 3;

// The items first, first + stride, ... below hi; none where first is not below hi.
struct Dealt { int first, hi, stride; };

// Items of a launch: (token tile, row tile) pairs, times the parts of a contraction.
template <int NM, bool ROUTED, int WAVES>
__device__ __forceinline__ int count_items(const MfmaArgs& a, int parts) {
  const int tiles = ROUTED ? a.tile_list[0] : (__builtin_amdgcn_readfirstlane(*a.valid_tokens) + a.tile_rows - 1) / a.tile_rows;
  return tiles * (a.n_rows / (WAVES * kWRows / NM)) * parts;
}

template <int QUANT, int NM, bool ROUTED, int MI, int WAVES, bool kInParts>
__device__ __forceinline__ void mfma_rows_body(const MfmaArgs& a, const Dealt& dealt) {
  const int first = dealt.first, hi = dealt.hi, stride = dealt.stride;
  if (first >= hi) return;
  constexpr int kTM = 32 * MI;                    // token rows of a tile at most
  constexpr int kTR = WAVES * kWRows;             // weight rows of a tile
  constexpr int kSlot = MI * kBlockBytes;         // an activation step in LDS
  constexpr int kRing = xabe::kRing<MI>;
  using Window = WWindow<QUANT, MI>;
  constexpr int kRun = Window::kRunBytes, kRunInstr = Window::kRunInstr;
  constexpr bool kScaled = ROUTED && NM == 1;
  constexpr uint32_t kSbBytes = QUANT == kQ6K ? kQ6KBytes : 8 * kQ8Bytes;
  extern __shared__ __attribute__((aligned(16))) uint8_t mfma_smem[];
  uint8_t* const sA = mfma_smem;
  uint8_t* const sW = sA + kRing * kSlot;
  // flat selection indices of an item's rows: gate/up, this item's and the next one's; down, this item's and their weights
  int* const sId = reinterpret_cast<int*>(sW + WAVES * 2 * kRun);
  [[maybe_unused]] float* const sScale = reinterpret_cast<float*>(sId + kTM);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, col = lane & 31;
  const int valid = __builtin_amdgcn_readfirstlane(*a.valid_tokens);
  const int n_ntiles = a.n_rows / (kTR / NM);
  const int tile_rows = a.tile_rows;
  const int parts = kInParts ? a.parts : 1;
  const int k_part = a.K / parts, nsteps = k_part / kSK, nsb = k_part / 256;
  const uint32_t row_bytes = QUANT == kQ6K ? (uint32_t)(a.K / 256) * kQ6KBytes : (uint32_t)(a.K / 32) * kQ8Bytes;

  // The lane's number for what an item does once: its arithmetic belongs there and not in registers all along, which would
  // be spilled, and what reloads a spilled register waits for every request in flight.
  auto item_lane = [&]() __attribute__((always_inline)) {
    int lane = (int)__lane_id();
    asm volatile("" : "+v"(lane));
    return lane;
  };

  struct Item { int e, m0, rows, nt, part; };
  auto decode = [&](int item) __attribute__((always_inline)) {
    const int row = item / n_ntiles, mt = kInParts ? row / parts : row;
    Item it{0, mt * tile_rows, min(tile_rows, valid - mt * tile_rows), item % n_ntiles, kInParts ? row % parts : 0};
    if (ROUTED) {
      typedef int int4v __attribute__((ext_vector_type(4)));
      int4v ent;
      const int* p = a.tile_list + 4 + 4 * mt;
      asm volatile("s_load_dwordx4 %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(ent) : "s"(p));
      it.e = ent.x;
      it.m0 = ent.y;
      it.rows = min(ent.z, kTM);  // (a list is cut for its launch; LDS holds no more)
    }
    return it;
  };

  // ---- weights: the wavefront's slot
  uint8_t* const slot = sW + wave * 2 * kRun;
  const uint32_t slot_lds = lds_address(slot);
  uint32_t w_off[kRunInstr];  // the lane's piece of each instruction of a run
#pragma unroll
  for (int i = 0; i < kRunInstr; ++i) {
    const int pc = min(64 * i + lane, 16 * Window::kPieces - 1);
    w_off[i] = (uint32_t)(pc / Window::kPieces) * row_bytes + (uint32_t)(pc % Window::kPieces) * 16;
  }
  const uint8_t *w_base0, *w_base1;  // the runs' first rows, of the item the weight stream is in
  // (in parts) how far into its rows an item starts, the weight stream's, and whether it ends them
  auto start_of = [&](const Item& it) __attribute__((always_inline)) { return kInParts ? (uint32_t)(it.part * nsb) * kSbBytes : 0u; };
  [[maybe_unused]] uint32_t w_from = 0;
  [[maybe_unused]] bool w_ends = true;
  uint32_t w_last0, w_last1;         // the last whole piece of the stack from there
  auto set_w = [&](const Item& it) __attribute__((always_inline)) {
    const int r0 = it.nt * (kTR / NM) + wave * (kWRows / NM);
    if constexpr (kInParts) w_from = start_of(it), w_ends = it.part + 1 == parts;
    const size_t off0 = (size_t)it.e * a.expert_bytes + (size_t)r0 * row_bytes;
    const size_t off1 = NM == 2 ? off0 : off0 + (size_t)16 * row_bytes;
    w_base0 = a.w0 + off0;
    w_base1 = (NM == 2 ? a.w1 : a.w0) + off1;
    auto to_last = [&](size_t off) __attribute__((always_inline)) {  // (a run's own pieces lie far below 2^31)
      const size_t n = a.w_bytes - 16 - off;
      return (n >> 31) != 0 ? 0x7fffffffu : (uint32_t)n;  // (scalar: a 64-bit minimum would hold vector registers)
    };
    w_last0 = to_last(off0);
    w_last1 = to_last(off1);
  };
  uint32_t w_at = 0;  // the requested window's start in its rows
  auto request_w = [&](auto i_c) __attribute__((always_inline)) {  // instruction i of either run
    constexpr int i = decltype(i_c)::value, kLastLanes = 16 * Window::kPieces - 64 * (kRunInstr - 1);
    constexpr uint64_t kLast = kLastLanes == 64 ? ~0ull : (1ull << kLastLanes) - 1;
    const uint32_t voff = (w_off[i] + w_at) & ~Window::kStart;
    if (i + 1 < kRunInstr || kLastLanes == 64) {
      lds_dma_16(w_base0, min(voff, w_last0), slot_lds + i * 1024);
      lds_dma_16(w_base1, min(voff, w_last1), slot_lds + kRun + i * 1024);
    } else {
      lds_dma_16_lanes(w_base0, min(voff, w_last0), slot_lds + i * 1024, (uint32_t)kLast, (uint32_t)(kLast >> 32));
      lds_dma_16_lanes(w_base1, min(voff, w_last1), slot_lds + kRun + i * 1024, (uint32_t)kLast, (uint32_t)(kLast >> 32));
    }
  };
  auto request_w_all = [&]() __attribute__((always_inline)) {
    request_w(std::integral_constant<int, 0>{});
    request_w(std::integral_constant<int, 1>{});
    request_w(std::integral_constant<int, 2>{});
    if constexpr (kRunInstr > 3) request_w(std::integral_constant<int, kRunInstr - 1>{});
  };
  const uint32_t my_row = (uint32_t)(col & 15) * row_bytes;
  const bool even_rows = QUANT == kQ6K && (row_bytes & 3) == 0;  // (then a superblock starts on a word in every row or in none)
  const uint8_t* const my_window = slot + (col >> 4) * kRun + (col & 15) * (Window::kPieces * 16);
  // half `u` of the contraction, which starts `from` bytes into its rows, out of the slot
  auto read_w = [&](uint32_t from, int u, int half, WHalf<QUANT>& r) __attribute__((always_inline)) {
    const uint32_t at = (uint32_t)(QUANT == kQ6K ? u >> 1 : u) * Window::kSpan + from, mis = (my_row + at) & Window::kStart;
    if constexpr (QUANT == kQ6K) w_read(my_window, mis, even_rows && (at & 2) == 0, half, h, r);
    else w_read(my_window + mis, 0, false, half, h, r);
  };
  // (Q6_K) the window just landed is the last of its rows: what no piece inside the tensor holds, where a row ends it
  auto patch_w = [&]() __attribute__((always_inline)) {
    if (kInParts && !w_ends) return;
    const size_t run_bytes = (size_t)16 * row_bytes;
    if (w_base0 + run_bytes == a.w0 + a.w_bytes) patch_window<kQ6K>(a.w0, a.w_bytes - kQ6KBytes, slot + 15 * (Window::kPieces * 16));
    if (w_base1 + run_bytes == (NM == 2 ? a.w1 : a.w0) + a.w_bytes)
      patch_window<kQ6K>(NM == 2 ? a.w1 : a.w0, a.w_bytes - kQ6KBytes, slot + kRun + 15 * (Window::kPieces * 16));
  };

  // ---- activations
  // piece q = wave + WAVES i of a step: token rows 8 q .. 8 q + 7; lane: row 8 q + (lane >> 3), position lane & 7, which
  // holds chunk (lane & 7) ^ pc_swizzle(row)
  constexpr int kPI = 4 * MI / WAVES;
  uint32_t a_off[kPI];  // the lane's piece of each instruction
  int a_pieces = 0;     // pieces of live 32-row blocks
  auto set_a = [&](const Item& it, int tb) __attribute__((always_inline)) {
    a_pieces = (it.rows + 31) / 32 * 4;
    const int lane = item_lane();
#pragma unroll
    for (int i = 0; i < kPI; ++i) {
      const int row = 8 * (wave + WAVES * i) + (lane >> 3), live = min(row, it.rows - 1);
      int arow = it.m0 + live;
      if (ROUTED && NM == 2) arow = (int)((uint32_t)sId[tb * kTM + live] / (uint32_t)a.top_k);
      a_off[i] = ((uint32_t)arow * (uint32_t)a.K + (uint32_t)((lane & 7) ^ pc_swizzle(row)) * 8u) * 2u;
      if constexpr (kInParts) a_off[i] += (uint32_t)(it.part * k_part) * 2u;
    }
  };
  const uint32_t lds_a = lds_address(sA) + (uint32_t)wave * 1024u;
  int a_ks = 0;       // the activation stream's step
  uint32_t a_to = 0;  // its place in the ring
  auto request_a = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kPI; ++i) {
      const uint32_t live = WAVES * i < a_pieces ? ~0u : 0u;
      lds_dma_16_lanes(a.a, a_off[i] + (uint32_t)a_ks * (kSK * 2u), lds_a + a_to + 1024u * WAVES * i, live, live);
    }
  };
  auto request_ids = [&](const Item& it, int tb) __attribute__((always_inline)) {
    const int lane = item_lane();
    if (64 * wave < kTM)
      lds_dma_4(a.sorted_token_ids, (uint32_t)(it.m0 + min(64 * wave + lane, it.rows - 1)) * 4u, lds_address(sId + tb * kTM + 64 * wave));
  };
  auto request_scales = [&]() __attribute__((always_inline)) {
    const int lane = item_lane();
    if (64 * wave < kTM) lds_dma_4(a.topk_weights, (uint32_t)sId[64 * wave + lane] * 4u, lds_address(sScale + 64 * wave));
  };
  auto all_landed = [&]() __attribute__((always_inline)) {
    order_fence();
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    order_fence();
  };
  // where the lane finds its row's eight elements of chunk kk of a step: piece 4 (kk >> 1) + 2 h + (kk & 1)
  const uint32_t frag = (uint32_t)col * (kSK * 2) + (uint32_t)(((2 * h) ^ pc_swizzle(col)) * 16);
  const uint32_t pick = w_scale_bytes(h);
  Item cur = decode(first), nxt = cur;
  int tb = 0;              // which of the two tables is this item's
  WHalf<QUANT> raw[QUANT == kQ6K ? 2 : 1];  // the raw weights that an item starts on: a superblock's halves, or its first
  uint32_t ring = 0;       // this step's place in the ring
  auto ring_after = [&](uint32_t r) __attribute__((always_inline)) { return r + kSlot == kRing * kSlot ? 0u : r + kSlot; };
  int w_win = 1;           // the weight stream's next window
  const int n_win = nsb * Window::kPerSb;

  if (ROUTED && NM == 2) {
    request_ids(cur, 0);
    all_landed();
  }
  set_w(cur);
  set_a(cur, 0);
  w_at = w_from;
  request_w_all();
#pragma unroll
  for (a_ks = 0; a_ks < kRing; ++a_ks) {  // (a contraction has at least four steps)
    a_to = (uint32_t)a_ks * kSlot;
    request_a();
  }
  a_ks = kRing - 1;
  all_landed();
  if (QUANT == kQ6K && w_win == n_win) patch_w();
  read_w(start_of(cur), 0, 0, raw[0]);
  if constexpr (QUANT == kQ6K) read_w(start_of(cur), 1, 1, raw[1]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  // (the requests that the chunks before the first would have made: the next window's)
  if (w_win == n_win) {
    w_win = 0;
    if (first + stride < hi) set_w(decode(first + stride));
  }
  w_at = (uint32_t)w_win * Window::kSpan + w_from;
  ++w_win;
  request_w_all();
  wait_vm<0>();

  for (int item = first;; item += stride) {
    const bool has_next = item + stride < hi;
    nxt = has_next ? decode(item + stride) : cur;
    asm volatile("" ::"s"(nxt.e), "s"(nxt.m0), "s"(nxt.rows), "s"(nxt.nt));
    if (ROUTED && nsteps < 8) {  // (no step late enough to find the tables by itself)
      all_landed();                // (the table is free: everyone is past the epilogue that read it)
      if constexpr (NM == 2) request_ids(nxt, tb ^ 1);
      else request_ids(cur, 0);
      all_landed();
      if constexpr (kScaled) {
        request_scales();
        all_landed();
      }
    }

    auto run = [&](auto nb_c) __attribute__((always_inline)) {
      constexpr int NB = decltype(nb_c)::value;
      float16v acc[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][v] = 0.0f;
      half8 fa[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i) fa[i] = *reinterpret_cast<const half8*>(sA + ring + frag + i * kBlockBytes);
      WChunk wc;
      w_parts_from<0>(raw[0], pick, wc);
      half8 fb = w_halfs(wc);
#pragma unroll 1
      for (int sb = 0; sb < nsb; ++sb) {
        WHalf<QUANT> next[2];
        // (Q8_0: the second half, read where it is needed.  It lives in here: outside, its last value would be held all round
        // the loop, since either of two places may write it)
        [[maybe_unused]] WHalf<QUANT> second;
        auto half_of = [&](auto c_c) __attribute__((always_inline)) -> const WHalf<QUANT>& {  // what chunk c's weights come from
          constexpr int c = decltype(c_c)::value;
          if constexpr (c == 0) return next[0];
          else if constexpr (c < 8) return raw[0];
          else if constexpr (QUANT == kQ6K) return raw[1];
          else return second;
        };
        auto chunk = [&](auto c_c) __attribute__((always_inline)) {
          constexpr int C = decltype(c_c)::value, C1 = (C + 1) & 15;
          using Req = Requests<QUANT, kPI>;
          // raw weights out of the slot: the next superblock's (Q6_K), the next half's (Q8_0)
          if constexpr (QUANT == kQ6K) {
            const int u = sb + 1 == nsb ? 0 : 2 * sb + 2;
            const uint32_t from = kInParts ? start_of(sb + 1 == nsb ? nxt : cur) : 0;
            if constexpr (C == 13) {
              wait_vm<Req::after_w(C)>();
              if (w_win == n_win) patch_w();
              read_w(from, u, 0, next[0]);
            }
            if constexpr (C == 14) read_w(from, u + 1, 1, next[1]);
          } else if constexpr ((C & 7) == 6) {
            wait_vm<Req::after_w(C)>();
            read_w(0, C < 8 ? 1 : 0, 0, C < 8 ? second : next[0]);  // (Q8_0 superblocks are whole pieces)
          }
          if constexpr ((C & 3) == 3) {
            constexpr int S = C >> 2;
            // everyone's pieces of the next step have landed, and everyone has read this step's for the last time, and the slot
            order_fence();
            wait_vm<Req::after_a(C - 4 * (kRing - 1), C)>();
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            order_fence();
            if (ROUTED && nsteps >= 8) {
              if (NM == 2 && S == 0 && sb == 0) request_ids(nxt, tb ^ 1);
              if (kScaled && S == 0 && sb == 0) request_ids(cur, 0);
              if (kScaled && S == 0 && sb == 1) request_scales();
            }
            if (++a_ks == nsteps) {
              a_ks = 0;
              set_a(nxt, tb ^ 1);
            }
            a_to = ring;
            if constexpr (S == 3 || (QUANT == kQ8_0 && S == 1)) {
              if (w_win == n_win) {
                w_win = 0;
                // (windows are requested two ahead: a contraction of one window is past the next item with that)
                if (QUANT == kQ6K && n_win == 1) {
                  if (item + 2 * stride < hi) set_w(decode(item + 2 * stride));
                } else {
                  set_w(nxt);
                }
              }
              w_at = (uint32_t)w_win * Window::kSpan + w_from;
              ++w_win;
            }
            ring = ring_after(ring);
          }
          order_fence();
          const WHalf<QUANT>& r1 = half_of(std::integral_constant<int, C1>{});
          const uint8_t* pa = sA + ((frag ^ (64u * ((C1 >> 1) & 1) + 16u * (C1 & 1))) + ring);
#pragma unroll
          for (int i = 0; i < NB; ++i) {
            // (which operand comes first decides what a lane's sums are: a token's for gate/up, a weight row's for down)
            acc[i] = NM == 2 ? __builtin_amdgcn_mfma_f32_32x32x16_f16(fb, fa[i], acc[i], 0, 0, 0)
                             : __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i], fb, acc[i], 0, 0, 0);
            fa[i] = *reinterpret_cast<const half8*>(pa + i * kBlockBytes);
            // the next chunk's weights between the matrix instructions: the two run beside each other (up to four vector
            // instructions cost a matrix instruction nothing)
            if (0 * NB / kWParts == i) w_part<C1 & 7, 0>(r1, pick, wc);
            if (1 * NB / kWParts == i) w_part<C1 & 7, 1>(r1, pick, wc);
            if (2 * NB / kWParts == i) w_part<C1 & 7, 2>(r1, pick, wc);
            if (3 * NB / kWParts == i) w_part<C1 & 7, 3>(r1, pick, wc);
            if (4 * NB / kWParts == i) w_part<C1 & 7, 4>(r1, pick, wc);
            __builtin_amdgcn_sched_barrier(0);
          }
          if constexpr (Req::a_at(C) != 0) request_a();
          if constexpr (Req::w_at(C) != 0) request_w(std::integral_constant<int, QUANT == kQ6K ? (C + 1) & 15 : (C + 1) & 7>{});
          fb = w_halfs(wc);
          if constexpr (C1 == 0) {
            raw[0] = next[0];
            if constexpr (QUANT == kQ6K) raw[1] = next[1];
          }
        };
        chunk(std::integral_constant<int, 0>{});
        chunk(std::integral_constant<int, 1>{});
        chunk(std::integral_constant<int, 2>{});
        chunk(std::integral_constant<int, 3>{});
        chunk(std::integral_constant<int, 4>{});
        chunk(std::integral_constant<int, 5>{});
        chunk(std::integral_constant<int, 6>{});
        chunk(std::integral_constant<int, 7>{});
        chunk(std::integral_constant<int, 8>{});
        chunk(std::integral_constant<int, 9>{});
        chunk(std::integral_constant<int, 10>{});
        chunk(std::integral_constant<int, 11>{});
        chunk(std::integral_constant<int, 12>{});
        chunk(std::integral_constant<int, 13>{});
        chunk(std::integral_constant<int, 14>{});
        chunk(std::integral_constant<int, 15>{});
      }

      // epilogue.  acc[i][v] of block i: gate/up, token lane % 32 and weight row (v / 4) * 8 + h * 4 + v % 4 of the wavefront's, so that
      // a token's gate and up columns are in one lane and leave as sixteen bytes; down, the other way round, so that a store
      // covers 128 bytes of a row (as sixteen bytes per lane, 64 of a row, 1237 tokens took 319 us instead of 309)
      const int lane = item_lane();
      const int h = lane >> 5, col = lane & 31;
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int left = cur.rows - 32 * i;  // live rows from this block on
        if constexpr (NM == 2) {
          // registers 0-7 are gate columns, 8-15 the matching up columns; as halfs, two exchanges between the lane halves give
          // lane h of a token the columns 8 h .. 8 h + 7
          uint32_t p[4];
#pragma unroll
          for (int v = 0; v < 8; v += 2) {
            uint16_t o[2];
#pragma unroll
            for (int w = 0; w < 2; ++w) {
              // (silu_fast(g) * up, both sums' 2^-8 on the gate; halfs one by one: a pair's conversion would round the product twice)
              const float g = acc[i][v + w], e = __builtin_amdgcn_exp2f(g * (-1.44269504088896340736f * kWScaleInv));
              o[w] = __builtin_bit_cast(uint16_t, (_Float16)(g * (kWScaleInv * kWScaleInv) * __builtin_amdgcn_rcpf(1.0f + e) * acc[i][v + w + 8]));
            }
            p[v / 2] = o[0] | (uint32_t)o[1] << 16;
          }
          const auto s0 = __builtin_amdgcn_permlane32_swap(p[0], p[2], false, false), s1 = __builtin_amdgcn_permlane32_swap(p[1], p[3], false, false);
          _Float16* block = static_cast<_Float16*>(a.out) + (size_t)(cur.m0 + 32 * i) * a.n_rows + cur.nt * (kTR / 2) + 16 * wave;
          if (col < left) *reinterpret_cast<u32x4*>(block + (uint32_t)(col * a.n_rows + 8 * h)) = u32x4{s0[0], s1[0], s0[1], s1[1]};
        } else {
          float* out = static_cast<float*>(a.out);
          if (kInParts && cur.part > 0) out = a.planes + (size_t)(cur.part - 1) * a.plane;
          out += cur.nt * kTR + 32 * wave;
          if (!ROUTED) out += (size_t)(cur.m0 + 32 * i) * a.n_rows;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (8 * q >= left) break;
            int4 id = {0, 0, 0, 0};
            float4 w4 = {1.0f, 1.0f, 1.0f, 1.0f};
            if constexpr (ROUTED) {
              id = *reinterpret_cast<const int4*>(sId + 32 * i + 8 * q + 4 * h);
              w4 = *reinterpret_cast<const float4*>(sScale + 32 * i + 8 * q + 4 * h);
            }
            const int ids[4] = {id.x, id.y, id.z, id.w};
            const float ws[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              const int r = 8 * q + 4 * h + w;
              float* to = out + ((size_t)(uint32_t)(ROUTED ? ids[w] : r) * (uint32_t)a.n_rows + (uint32_t)col);
              if (r < left) *to = ws[w] * kWScaleInv * acc[i][4 * q + w];
            }
          }
        }
      }
      // (a join of its own for the last store's branch: run into the item loop's, it makes the weights' scalar addresses vector ones)
      asm volatile("" ::: "memory");
    };
    const int nb = (cur.rows + 31) / 32;
    if constexpr (MI > 2) {
      switch (nb) {
        case 1: run(std::integral_constant<int, 1>{}); break;
        case 2: run(std::integral_constant<int, 2>{}); break;
        case 3: run(std::integral_constant<int, 3>{}); break;
        case 4: run(std::integral_constant<int, 4>{}); break;
        case 5: run(std::integral_constant<int, 5>{}); break;
        default: run(std::integral_constant<int, 6>{}); break;
      }
    } else {
      if (nb == 1) run(std::integral_constant<int, 1>{});
      else run(std::integral_constant<int, 2>{});
    }
    if (!has_next) break;
    cur = nxt;
    tb ^= 1;
  }
  // (nothing may still be on its way into this workgroup's LDS when it ends)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}
// Which items a workgroup takes.  Workgroup ids are dealt round-robin to the eight XCDs, each with its own L2: when
// there is work for every workgroup, XCD x takes a contiguous eighth of the items (token tile major) and its workgroups
// walk that range together, so an activation tile is fetched into one L2 instead of into all eight, and the token tiles
// of one expert reuse its weights from that L2.
// Routed gate/up, narrow: a third round of items would be two thirds full at most, and it begins late on the CUs that a
// launch beside this one still holds when it begins.  There a grid of twice the workgroups that fit (gate_up_twice) deals the
// second half to whatever CU is free first, one or two items each; in fewer rounds, or more, the half that fits does as
// well or better by itself (the others get nothing).
template <bool kTwice>
__device__ __forceinline__ Dealt deal_items(int total, int resident) {
  const bool twice = kTwice && total >= 2 * resident && total < 3 * resident;
  const int wgs = kTwice && !twice ? min((int)gridDim.x, resident) : (int)gridDim.x;
  const bool by_xcd = (wgs & 7) == 0 && (twice || total >= 2 * wgs);
  const int xcd = blockIdx.x & 7;
  const int lo = by_xcd ? (int)((long long)total * xcd / 8) : 0, hi = by_xcd ? (int)((long long)total * (xcd + 1) / 8) : total;
  const int first = lo + (by_xcd ? (int)(blockIdx.x >> 3) : (int)blockIdx.x);
  return {kTwice && (int)blockIdx.x >= wgs ? hi : first, hi, by_xcd ? wgs >> 3 : wgs};
}

template <int QUANT, int NM, bool ROUTED, int MI, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, (kWgsPerCu<MI, WAVES> * WAVES / 4)) k_mfma_rows(MfmaArgs a) {
  constexpr bool kTwice = ROUTED && NM == 2 && MI <= 2;
  mfma_rows_body<QUANT, NM, ROUTED, MI, WAVES, false>(a, deal_items<kTwice>(count_items<NM, ROUTED, WAVES>(a, 1), a.resident));
}
// An unrouted down contraction in parts (down_parts).
template <int QUANT, int MI, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, (kWgsPerCu<MI, WAVES> * WAVES / 4)) k_mfma_parts(MfmaArgs a) {
  mfma_rows_body<QUANT, 1, false, MI, WAVES, true>(a, deal_items<false>(count_items<1, false, WAVES>(a, a.parts), a.resident));
}
// The routed experts' items (QUANT, `a`) and the shared expert's (SQUANT, `s`) of one pass in one launch, narrow form.  Alone a launch of
// the shared expert's is a workgroup per CU or fewer, as long as one item (512 tokens: 27 us and 12); here they fill the last round of
// the routed items: workgroups that have one routed item fewer come first.  By trace, 512 tokens, skewed: gate/up 64 to 70 us without, 70
// with, down 40 and 46, the routing in front 12 and 10, and no fork, join or waiting: a block 168 to 176 and 161 to 162 us.  Shared items first: 512 tokens
// 252.9 -> 255.1.  (The items are dealt as in deal_items, in two kinds: a change of one belongs in the other.)
template <int QUANT, int SQUANT, int NM>
__global__ void __launch_bounds__(256, 3) k_mfma_with_shared(MfmaArgs a, MfmaArgs s) {
  const int routed = count_items<NM, true, 4>(a, 1), shared = count_items<NM, false, 4>(s, 1), total = routed + shared;
  const bool twice = NM == 2 && total >= 2 * a.resident && total < 3 * a.resident;  // (deal_items)
  const int wgs = twice ? (int)gridDim.x : min((int)gridDim.x, a.resident);
  if ((int)blockIdx.x >= wgs) return;
  const bool by_xcd = (wgs & 7) == 0 && (twice || total >= 2 * wgs);
  const int xcd = blockIdx.x & 7, rank = by_xcd ? (int)blockIdx.x >> 3 : (int)blockIdx.x, stride = by_xcd ? wgs >> 3 : wgs;
  auto share = [&](int items, int behind) __attribute__((always_inline)) {  // of the XCD, dealt from its workgroup `behind` on
    const int lo = by_xcd ? (int)((long long)items * xcd / 8) : 0, hi = by_xcd ? (int)((long long)items * (xcd + 1) / 8) : items;
    const int place = rank - behind % stride;
    return Dealt{lo + (place < 0 ? place + stride : place), hi, stride};
  };
  const Dealt mine = share(routed, 0);
  const int before = by_xcd ? (int)((long long)routed * (xcd + 1) / 8) - (int)((long long)routed * xcd / 8) : routed;
  mfma_rows_body<QUANT, NM, true, 2, 4, false>(a, mine);
  // (the bodies share LDS: each ends with its own requests landed, and all wavefronts are past their last reads here)
  __syncthreads();
  mfma_rows_body<SQUANT, NM, false, 2, 4, false>(s, share(shared, before));
}

// fp32 -> fp16 activations for live rows; rows past `valid` are left alone.
__global__ void __launch_bounds__(256) k_to_f16_rows(const float* __restrict__ x, const int* __restrict__ valid_tokens,
                                                      int width, _Float16* __restrict__ out) {
  const int t = blockIdx.x;
  if (t >= *valid_tokens) return;
  const float4* src = reinterpret_cast<const float4*>(x + (size_t)t * width);
  uint2* dst = reinterpret_cast<uint2*>(out + (size_t)t * width);
  for (int j = threadIdx.x; j < width / 4; j += 256) {
    const float4 v = src[j];
    const half2v lo = {(_Float16)v.x, (_Float16)v.y}, hi = {(_Float16)v.z, (_Float16)v.w};
    dst[j] = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
  }
}

// Token-tile list (layout: MfmaArgs), the tiles of each active expert's run at most `bm` rows tall.  One workgroup.
__global__ void __launch_bounds__(256) k_build_tiles(const int* __restrict__ expert_counts, int num_experts, int block_size,
                                                      int capacity, int bm, int* __restrict__ tile_list) {
  __shared__ int s_base[513], s_tiles[513];
  // exclusive prefixes of the padded run lengths and of the tile counts (num_experts <= 512): every thread
  // takes two experts, the pair sums are scanned across the workgroup in eight doubling steps
  __shared__ int s_scan[2][2][256];
  const int t = threadIdx.x;
  int pad[2], til[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int e = 2 * t + j;
    const int c = e < num_experts ? expert_counts[e] : 0;
    pad[j] = (c + block_size - 1) / block_size * block_size;
    til[j] = (c + bm - 1) / bm;
  }
  s_scan[0][0][t] = pad[0] + pad[1];
  s_scan[0][1][t] = til[0] + til[1];
  __syncthreads();
  int cur = 0;
  for (int d = 1; d < 256; d <<= 1) {
#pragma unroll
    for (int a = 0; a < 2; ++a) s_scan[cur ^ 1][a][t] = s_scan[cur][a][t] + (t >= d ? s_scan[cur][a][t - d] : 0);
    cur ^= 1;
    __syncthreads();
  }
  const int base = s_scan[cur][0][t] - (pad[0] + pad[1]), tiles = s_scan[cur][1][t] - (til[0] + til[1]);
  if (2 * t < num_experts) s_base[2 * t] = base, s_tiles[2 * t] = tiles;
  if (2 * t + 1 < num_experts) s_base[2 * t + 1] = base + pad[0], s_tiles[2 * t + 1] = tiles + til[0];
  if (t == 255) tile_list[0] = min(s_scan[cur][1][t], capacity);
  __syncthreads();
  for (int e = threadIdx.x; e < num_experts; e += 256)
    write_tile_entries(e, expert_counts[e], s_base[e], s_tiles[e], bm, capacity, tile_list);
}

// ------------------------------------------------------------------ host side
static size_t stack_row_bytes(int quant, size_t K) {
  return K / xabe_expert_quant_block_elements(quant) * xabe_expert_quant_block_bytes(quant);
}

bool mfma_supported(const xabe_moe_kernels* k, const xabe_moe_buffers* b, int gate_q, int up_q, int down_q, bool routed) {
  const xabe_moe_geometry& g = k->g;
  if (!k->tensor_cores || k->exact_regime || g.max_tokens < kMfmaMinTokens) return false;
  if (!b->x_h || !b->shared_inter_h) return false;
  if (routed && (!b->inter_h || !b->tile_list)) return false;
  if (routed && g.num_experts > 512) return false;  // k_build_tiles scans two experts per thread of one 256-thread workgroup
  auto ok = [](int q) { return q == XABE_QUANT_Q6K || q == XABE_QUANT_Q8_0; };
  if (!ok(gate_q) || !ok(down_q) || gate_q != up_q) return false;
  // whole superblocks of the contraction; gate/up tiles of 128 columns, down tiles of 256
  if (g.hidden % 256 != 0 || g.intermediate % 256 != 0) return false;
  // an activation piece is addressed by a 32-bit byte offset from its tensor's base (fp16 rows of either width, as
  // many as the sorted table has slots)
  const size_t rows = g.max_tokens * g.experts_per_token + g.num_experts * g.block_size;
  if (rows * std::max(g.hidden, g.intermediate) >= ((size_t)1 << 31)) return false;
  return true;
}

static int routed_tile_rows(const xabe_moe_geometry& g, size_t tokens) {
  return narrow_tiles(tokens, g.experts_per_token, g.num_experts) ? kNarrowRows : kWideRows;
}
// Whether narrow gate/up is launched with twice the workgroups that fit: while an expert's share averages one block of 32 rows.
// With the shared expert's items along (k_mfma_with_shared), one layer, us, once / twice: 80 tokens 217 / 222 (the loss that this line
// accepts), 256: 241 / 238, 512: 256 / 254, 700 and 1000 alike; skewed 120 to 700 alike, 1000: 223 / 226.  By itself, the shared expert on a stream beside it, layers of the routed model in a row, us, once / twice: 512 tokens 259.6 / 251.0, 700: 269 / 265, 900: 279.5 / 277.4, 1000: 285.5 / 284.0,
// 1024: 286.3 / 285.1; with the seam 252 / 245, 263 / 258, 275 / 270, 279.2 / 277.4, 279.6 / 278.4; with the published layout 267 / 260, 279 / 274,
// 292 / 286, 296 / 293, 297 / 295.5; 100 and 256 tokens gain as 512 do.  Skewed loads: less than two rounds of items up to 900 tokens, and alike;
// 950: 229 / 220, 1000: 253 / 227, 1024: 229 / 228.  At 1237 tokens, where items are one block or two, 327 / 313, but 314 / 317 in the
// published layout, and skewed 255 / 260.
static bool gate_up_twice(const xabe_moe_geometry& g, size_t tokens) { return share_in_one_block(tokens, g.experts_per_token, g.num_experts); }
// The specialised form (k_mfma_pc) serves both routed launches for contractions of whole superblocks and at least
// eight steps, when asked for: `mfma_form` 2 (0 and 1: k_mfma_rows everywhere; it is the faster at every width
// measured, see k_mfma_pc).
static bool pc_shape_ok(const xabe_moe_geometry& g) {
  return g.hidden % 256 == 0 && g.intermediate % 256 == 0 && g.hidden >= 512 && g.intermediate >= 512;
}
static bool pc_form(const xabe_moe_kernels* k, size_t) { return k->mfma_form == 2 && pc_shape_ok(k->g); }
// The tokens a pass is known to hold when its launches are chosen: the live count last published to the device
// scalar (a 512-token chunk run in buffers sized for 8192 should get the tiles of a 512-token pass), the buffers'
// size before any was.  Every tile height serves any live count and gives the same bits, so a graph captured at one
// count and replayed after another was published is slower at worst.
static size_t pass_tokens(const xabe_moe_kernels* k, const xabe_moe_buffers* b) {
  return b->valid_published > 0 ? std::min<size_t>((size_t)b->valid_published, k->g.max_tokens) : k->g.max_tokens;
}
// Whether the launches of an unrouted pass take the wide form: when whole tiles of it give every CU one, or, as narrow tiles
// dequantise a row of weights once per 64 tokens, as soon as wide ones occupy half of the CUs.  Gate/up: more than 96 tokens of
// matrices whose tiles do that in one row; down in parts: more than 192.  (The shared expert of the routed model stays narrow
// up to 8192 tokens, where it leaves room beside it for the launches it runs along with: 1965 against 1980 us for two blocks.)
// Dense sibling, us per block, both narrow / gate/up wide / both wide: 96 tokens 152 / 149 / 162, 128: 164 / 162 / 177, 192: 203 / 185 /
// 199, 224: 250 / 247 / 239, 256: 263 / 252 / 244, 288: 307 / 272 / 258, 383: 362 / 319 / 292, 450: 463 / 379 / 326.
static bool unrouted_wide(const xabe_moe_kernels* k, size_t tokens) {
  return tokens / kWideRows * (k->g.intermediate / 128) >= (size_t)k->num_cus;
}
static bool unrouted_up_wide(const xabe_moe_kernels* k, size_t tokens) {
  return unrouted_wide(k, tokens) || (tokens > kWideRows / 2 && 2 * (k->g.intermediate / 128) >= (size_t)k->num_cus);
}
static bool unrouted_down_wide(const xabe_moe_kernels* k, size_t tokens, int parts) {
  const size_t items = (tokens + kWideRows - 1) / kWideRows * (k->g.hidden / 256) * parts;
  return unrouted_wide(k, tokens) || (parts > 1 && tokens > kWideRows && 2 * items >= (size_t)k->num_cus);
}
// Token rows of a wide unrouted tile: the height whose items, dealt in rounds to the CUs, end first, an item's time being
// that of its 32-row blocks and about 3.6 blocks' more (dense sibling, 2048 tokens: a superblock of the contraction
// takes 2.3 us and 0.64 us per block; down 385 us at 192 rows, one round, and 616 at 160, two).
// (A part of a contraction is an item like another: `row_tiles` counts it.)
static int unrouted_tile_rows(const xabe_moe_kernels* k, size_t tokens, size_t row_tiles) {
  int best = 32;
  double best_cost = 1e30;
  for (int h = 32; h <= kWideRows; h += 32) {
    const size_t items = (tokens + h - 1) / h * row_tiles, rounds = (items + k->num_cus - 1) / k->num_cus;
    const double cost = (double)rounds * (h / 32 + 3.6);
    if (cost < best_cost) best_cost = cost, best = h;
  }
  return best;
}

bool mfma_tile_plan(const xabe_moe_kernels* k, const xabe_moe_buffers* b, int* bm, int* capacity) {
  if (!b->tile_list || b->n_tile_list < 8 || !k->tensor_cores || k->exact_regime) return false;
  const size_t tokens = pass_tokens(k, b);
  *bm = routed_tile_rows(k->g, tokens);
  if (pc_form(k, tokens)) *bm = kPM;  // (the specialised launches: 128-row tiles)
  *capacity = (int)((b->n_tile_list - 4) / 4);
  return true;
}

// LDS of the kernels is dynamic, above the static limit, which is raised per function once, when a kernels handle is
// created (mfma_configure): nothing on the launch path but the launch.
template <int NM, bool ROUTED, int MI, int WAVES>
static int configure_one() {
  XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_mfma_rows<kQ6K, NM, ROUTED, MI, WAVES>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)mfma_rows_lds<kQ6K, MI, WAVES>()));
  XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_mfma_rows<kQ8_0, NM, ROUTED, MI, WAVES>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)mfma_rows_lds<kQ8_0, MI, WAVES>()));
  return XABE_OK;
}
template <int QUANT, int MI, int WAVES>
static int configure_parts() {
  XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_mfma_parts<QUANT, MI, WAVES>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)mfma_rows_lds<QUANT, MI, WAVES>()));
  return XABE_OK;
}
template <int NM>
static int configure_pc() {
  const void* fns[2] = {reinterpret_cast<const void*>(k_mfma_pc<kQ6K, NM>), reinterpret_cast<const void*>(k_mfma_pc<kQ8_0, NM>)};
  for (const void* f : fns)
    XABE_HIP_TRY(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)mfma_pc_lds_bytes()));
  return XABE_OK;
}
template <int NM>
static int launch_pc(const xabe_moe_kernels* k, int quant, const MfmaArgs& a, size_t max_items, hipStream_t s) {
  const unsigned grid = (unsigned)std::max<size_t>(1, std::min<size_t>(max_items, (size_t)k->num_cus));  // one workgroup per CU
  constexpr size_t smem = mfma_pc_lds_bytes();
  if (quant == XABE_QUANT_Q6K) hipLaunchKernelGGL((k_mfma_pc<kQ6K, NM>), dim3(grid), dim3(1024), smem, s, a);
  else hipLaunchKernelGGL((k_mfma_pc<kQ8_0, NM>), dim3(grid), dim3(1024), smem, s, a);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

template <int QUANT, int SQUANT, int NM>
constexpr size_t with_shared_lds() { return std::max(mfma_rows_lds<QUANT, 2, 4>(), mfma_rows_lds<SQUANT, 2, 4>()); }
template <int QUANT, int SQUANT>
static int configure_with_shared() {
  XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_mfma_with_shared<QUANT, SQUANT, 2>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)with_shared_lds<QUANT, SQUANT, 2>()));
  XABE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_mfma_with_shared<QUANT, SQUANT, 1>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)with_shared_lds<QUANT, SQUANT, 1>()));
  return XABE_OK;
}

static int mfma_set_limits() {
  XABE_TRY((configure_with_shared<kQ6K, kQ6K>()));
  XABE_TRY((configure_with_shared<kQ6K, kQ8_0>()));
  XABE_TRY((configure_with_shared<kQ8_0, kQ6K>()));
  XABE_TRY((configure_with_shared<kQ8_0, kQ8_0>()));
  XABE_TRY((configure_pc<2>()));
  XABE_TRY((configure_pc<1>()));
  XABE_TRY((configure_one<1, false, 6, 8>()));
  XABE_TRY((configure_one<2, false, 6, 8>()));
  XABE_TRY((configure_one<1, true, 6, 8>()));
  XABE_TRY((configure_one<2, true, 6, 8>()));
  XABE_TRY((configure_one<1, false, 2, 4>()));
  XABE_TRY((configure_one<2, false, 2, 4>()));
  XABE_TRY((configure_one<1, true, 2, 4>()));
  XABE_TRY((configure_one<2, true, 2, 4>()));
  XABE_TRY((configure_parts<kQ6K, 6, 8>()));
  XABE_TRY((configure_parts<kQ8_0, 6, 8>()));
  XABE_TRY((configure_parts<kQ6K, 2, 4>()));
  XABE_TRY((configure_parts<kQ8_0, 2, 4>()));
  return XABE_OK;
}

// at handle creation, for the current device
int mfma_configure() {
  static DeviceOnce once;
  int dev = 0;
  XABE_HIP_TRY(hipGetDevice(&dev));
  return once.run(dev, mfma_set_limits);
}

template <int NM, bool ROUTED, int MI, int WAVES>
static int launch_rows(const xabe_moe_kernels* k, int quant, MfmaArgs a, size_t max_mtiles, hipStream_t s, bool twice = false) {
  const size_t max_items = max_mtiles * (size_t)(a.n_rows / (WAVES * kWRows / NM));
  a.resident = k->num_cus * kWgsPerCu<MI, WAVES>;
  const size_t most = (size_t)a.resident * (twice ? 2 : 1);
  const unsigned grid = (unsigned)std::max<size_t>(1, std::min(max_items, most));
  if (quant == XABE_QUANT_Q6K)
    hipLaunchKernelGGL((k_mfma_rows<kQ6K, NM, ROUTED, MI, WAVES>), dim3(grid), dim3(64 * WAVES), (mfma_rows_lds<kQ6K, MI, WAVES>()), s, a);
  else
    hipLaunchKernelGGL((k_mfma_rows<kQ8_0, NM, ROUTED, MI, WAVES>), dim3(grid), dim3(64 * WAVES), (mfma_rows_lds<kQ8_0, MI, WAVES>()), s, a);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

template <int NM>
static int launch_with_shared(const xabe_moe_kernels* k, int quant, int shared_quant, MfmaArgs a, const MfmaArgs& sh, size_t max_mtiles,
                              size_t shared_mtiles, hipStream_t s, bool twice) {
  const size_t max_items = (max_mtiles + shared_mtiles) * (size_t)(a.n_rows / (4 * kWRows / NM));
  a.resident = k->num_cus * kWgsPerCu<2, 4>;
  const unsigned grid = (unsigned)std::max<size_t>(1, std::min(max_items, (size_t)a.resident * (twice ? 2 : 1)));
  auto launch = [&](auto q, auto sq) {
    constexpr int Q = decltype(q)::value, SQ = decltype(sq)::value;
    hipLaunchKernelGGL((k_mfma_with_shared<Q, SQ, NM>), dim3(grid), dim3(256), (with_shared_lds<Q, SQ, NM>()), s, a, sh);
  };
  auto with = [&](auto q) {
    if (shared_quant == XABE_QUANT_Q6K) launch(q, std::integral_constant<int, kQ6K>{});
    else launch(q, std::integral_constant<int, kQ8_0>{});
  };
  if (quant == XABE_QUANT_Q6K) with(std::integral_constant<int, kQ6K>{});
  else with(std::integral_constant<int, kQ8_0>{});
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

template <int MI, int WAVES>
static int launch_parts(const xabe_moe_kernels* k, int quant, const MfmaArgs& a, size_t mtiles, hipStream_t s) {
  const size_t items = mtiles * (size_t)(a.n_rows / (WAVES * kWRows)) * a.parts;
  const unsigned grid = (unsigned)std::max<size_t>(1, std::min<size_t>(items, (size_t)k->num_cus * kWgsPerCu<MI, WAVES>));
  if (quant == XABE_QUANT_Q6K)
    hipLaunchKernelGGL((k_mfma_parts<kQ6K, MI, WAVES>), dim3(grid), dim3(64 * WAVES), (mfma_rows_lds<kQ6K, MI, WAVES>()), s, a);
  else
    hipLaunchKernelGGL((k_mfma_parts<kQ8_0, MI, WAVES>), dim3(grid), dim3(64 * WAVES), (mfma_rows_lds<kQ8_0, MI, WAVES>()), s, a);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

static int to_f16(const xabe_moe_kernels* k, hipStream_t s, const xabe_moe_buffers* b, const float* x) {
  hipLaunchKernelGGL(k_to_f16_rows, dim3((unsigned)k->g.max_tokens), dim3(256), 0, s, x, b->valid_tokens, (int)k->g.hidden,
                     reinterpret_cast<_Float16*>(b->x_h));
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

int mfma_convert_activations(const xabe_moe_kernels* k, hipStream_t s, xabe_moe_buffers* b, const float* x) {
  return to_f16(k, s, b, x);
}

int mfma_grouped_forward_partial(const xabe_moe_kernels* k, hipStream_t s, xabe_moe_buffers* b, xabe_quant_tensor gate,
                                 xabe_quant_tensor up, xabe_quant_tensor down, const float* x, const MfmaShared* shared) {
  const xabe_moe_geometry& g = k->g;
  if (!b->x_h_ready) XABE_TRY(to_f16(k, s, b, x));
  int bm = 0, cap = 0;
  if (!mfma_tile_plan(k, b, &bm, &cap))
    return set_error(XABE_ERR_INVALID_ARGUMENT, "grouped_forward: these buffers hold no token-tile list");
  // the dispatch build has usually left the list, cut for this height:
  // trusted only when nothing can have rewritten them since: inside the capture that holds the build, or eagerly
  // after an eager build on buffers no graph has ever recorded a build on
  const unsigned long long capture = stream_capture_id(s);
  const bool trusted = b->tiles_bm == bm && capture != kCaptureUnknown &&
                       b->tiles_capture == capture && (capture != 0 || !b->tiles_graph_owned);
  if (!trusted) {
    hipLaunchKernelGGL(k_build_tiles, dim3(1), dim3(256), 0, s, b->expert_counts, (int)g.num_experts, (int)g.block_size, cap,
                       bm, b->tile_list);
    XABE_HIP_TRY(hipGetLastError());
  }
  MfmaArgs a;
  memset(&a, 0, sizeof(a));
  a.valid_tokens = b->valid_tokens;
  a.sorted_token_ids = b->sorted_token_ids;
  a.topk_weights = b->topk_weights;
  a.tile_list = b->tile_list;
  a.top_k = (int)g.experts_per_token;
  const size_t max_mtiles = (size_t)cap;
  // gate/up + SwiGLU -> inter_h[slot][I]
  a.w0 = static_cast<const uint8_t*>(gate.bytes);
  a.w1 = static_cast<const uint8_t*>(up.bytes);
  a.expert_bytes = g.intermediate * stack_row_bytes(gate.quant, g.hidden);
  a.w_bytes = gate.len;
  a.a = reinterpret_cast<const _Float16*>(b->x_h);
  a.out = b->inter_h;
  a.K = (int)g.hidden;
  a.n_rows = (int)g.intermediate;
  const bool pc = pc_form(k, pass_tokens(k, b));
  MfmaArgs sh = a;
  size_t shared_tiles = 0;
  if (shared) {  // (mfma_takes_shared)
    sh.top_k = 1;
    sh.tile_rows = kNarrowRows;
    sh.w0 = static_cast<const uint8_t*>(shared->gate.bytes);
    sh.w1 = static_cast<const uint8_t*>(shared->up.bytes);
    sh.expert_bytes = 0;
    sh.w_bytes = shared->gate.len;
    sh.out = b->shared_inter_h;
    shared_tiles = (g.max_tokens + kNarrowRows - 1) / kNarrowRows;
    XABE_TRY((launch_with_shared<2>(k, gate.quant, shared->gate.quant, a, sh, max_mtiles, shared_tiles, s, gate_up_twice(g, pass_tokens(k, b)))));
  } else if (pc) XABE_TRY((launch_pc<2>(k, gate.quant, a, max_mtiles * (g.intermediate / (kPR / 2)), s)));
  else if (bm == kNarrowRows) XABE_TRY((launch_rows<2, true, 2, 4>(k, gate.quant, a, max_mtiles, s, gate_up_twice(g, pass_tokens(k, b)))));
  else XABE_TRY((launch_rows<2, true, 6, 8>(k, gate.quant, a, max_mtiles, s)));
  // down -> partial[flat][H], scaled by the routing weight
  a.w0 = static_cast<const uint8_t*>(down.bytes);
  a.w1 = nullptr;
  a.expert_bytes = g.hidden * stack_row_bytes(down.quant, g.intermediate);
  a.w_bytes = down.len;
  a.a = reinterpret_cast<const _Float16*>(b->inter_h);
  a.out = b->partial;
  a.K = (int)g.intermediate;
  a.n_rows = (int)g.hidden;
  if (shared) {
    sh.w0 = static_cast<const uint8_t*>(shared->down.bytes);
    sh.w1 = nullptr;
    sh.w_bytes = shared->down.len;
    sh.a = reinterpret_cast<const _Float16*>(b->shared_inter_h);
    sh.out = shared->out;
    sh.K = a.K;
    sh.n_rows = a.n_rows;
    XABE_TRY((launch_with_shared<1>(k, down.quant, shared->down.quant, a, sh, max_mtiles, shared_tiles, s, false)));
  } else if (pc) XABE_TRY((launch_pc<1>(k, down.quant, a, max_mtiles * (g.hidden / kPR), s)));
  else if (bm == kNarrowRows) XABE_TRY((launch_rows<1, true, 2, 4>(k, down.quant, a, max_mtiles, s)));
  else XABE_TRY((launch_rows<1, true, 6, 8>(k, down.quant, a, max_mtiles, s)));
  return XABE_OK;
}

// Parts of an unrouted down contraction.  Its row tiles are few where the contraction is long (5120 rows: 40 narrow tiles, 20
// wide), and a tile walks its whole contraction alone: 64 tokens took 147 us on 40 workgroups.  Up to 1024 tokens the
// contraction is in four parts (or as many as divide it), whose sums are added in order by one more launch; by the
// buffers' size and the geometry alone, so that a token's row is the same bits in every pass and in every pass of buffers up to
// that size.  (Not in those of larger ones, where few live tokens walk one chain, too.)  Wider passes have tiles enough, and four
// planes of sums would cost them more than they gain (2048 tokens of the dense sibling: as many rounds of items, and 170 MB each
// way).  The planes lie in the fp32 intermediate rows, which the matrix-core regime does not use.
constexpr size_t kPartsMaxTokens = 1024;
static int down_parts(const xabe_moe_geometry& g) {
  if (g.max_tokens > kPartsMaxTokens) return 1;
  const size_t nsb = g.intermediate / 256;
  for (int parts = 4; parts > 1; --parts)
    if (nsb % parts == 0 && nsb / parts >= 8 && (size_t)(parts - 1) * g.hidden <= g.intermediate) return parts;
  return 1;
}

// Whether the shared expert's items go along with the routed ones (k_mfma_with_shared): where both take narrow tiles, the shared
// down projection is whole, and shared_along's rule on sizes says so.
static_assert(kNarrowUpRows == 4 * kWRows / 2 && kNarrowDownRows == 4 * kWRows, "the items that shared_along counts");
bool mfma_takes_shared(const xabe_moe_kernels* k, const xabe_moe_buffers* b) {
  const xabe_moe_geometry& g = k->g;
  const size_t tokens = pass_tokens(k, b);
  if (!shared_along(tokens, g.max_tokens, g.experts_per_token, g.num_experts, g.hidden, g.intermediate, (size_t)k->num_cus * kWgsPerCu<2, 4>)) return false;
  int bm = 0, cap = 0;
  if (!mfma_tile_plan(k, b, &bm, &cap) || bm != kNarrowRows || pc_form(k, tokens)) return false;
  return down_parts(g) == 1 && !unrouted_up_wide(k, tokens) && !unrouted_down_wide(k, tokens, 1);
}

// The parts' sums of a live row in order, and the residual where there is one.  Bound by memory (hidden is a multiple of 256).
__global__ void __launch_bounds__(256) k_add_parts(const float* __restrict__ planes, size_t plane, int parts, const int* __restrict__ valid_tokens,
                                                   int hidden, const float* __restrict__ residual, float* __restrict__ out, float* __restrict__ l_out) {
  const int t = blockIdx.x, j = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (t >= *valid_tokens || j >= hidden) return;
  const size_t i = (size_t)t * hidden + j;
  const bool whole = ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(residual) | reinterpret_cast<uintptr_t>(l_out)) & 15) == 0;
  float v[4], x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (whole) {
    const float4 f = *reinterpret_cast<const float4*>(out + i);
    v[0] = f.x, v[1] = f.y, v[2] = f.z, v[3] = f.w;
    if (l_out) {
      const float4 r = *reinterpret_cast<const float4*>(residual + i);
      x[0] = r.x, x[1] = r.y, x[2] = r.z, x[3] = r.w;
    }
  } else {  // (rows that start on any float)
    for (int c = 0; c < 4; ++c) v[c] = out[i + c], x[c] = l_out ? residual[i + c] : 0.0f;
  }
  float4 p[3];
#pragma unroll
  for (int n = 0; n < 3; ++n) p[n] = *reinterpret_cast<const float4*>(planes + (size_t)min(n, parts - 2) * plane + i);
#pragma unroll
  for (int n = 0; n < 3; ++n)
    if (n + 1 < parts) v[0] += p[n].x, v[1] += p[n].y, v[2] += p[n].z, v[3] += p[n].w;
  if (whole) {
    *reinterpret_cast<float4*>(out + i) = make_float4(v[0], v[1], v[2], v[3]);
    if (l_out) *reinterpret_cast<float4*>(l_out + i) = make_float4(v[0] + x[0], v[1] + x[1], v[2] + x[2], v[3] + x[3]);
  } else {
    for (int c = 0; c < 4; ++c) {
      out[i + c] = v[c];
      if (l_out) l_out[i + c] = v[c] + x[c];
    }
  }
}

int mfma_shared_expert(const xabe_moe_kernels* k, hipStream_t s, xabe_moe_buffers* b, xabe_quant_tensor gate,
                       xabe_quant_tensor up, xabe_quant_tensor down, const float* x, float* out, const float* residual, float* l_out,
                       bool* added) {
  const xabe_moe_geometry& g = k->g;
  if (!b->x_h_ready) XABE_TRY(to_f16(k, s, b, x));
  MfmaArgs a;
  memset(&a, 0, sizeof(a));
  a.valid_tokens = b->valid_tokens;
  a.top_k = 1;
  a.w0 = static_cast<const uint8_t*>(gate.bytes);
  a.w1 = static_cast<const uint8_t*>(up.bytes);
  a.a = reinterpret_cast<const _Float16*>(b->x_h);
  a.out = b->shared_inter_h;
  a.K = (int)g.hidden;
  a.n_rows = (int)g.intermediate;
  a.w_bytes = gate.len;
  const size_t tokens = pass_tokens(k, b);
  bool wide = unrouted_up_wide(k, tokens);
  a.tile_rows = wide ? unrouted_tile_rows(k, tokens, g.intermediate / 128) : kNarrowRows;
  size_t tiles = (g.max_tokens + a.tile_rows - 1) / a.tile_rows;
  if (wide) XABE_TRY((launch_rows<2, false, 6, 8>(k, gate.quant, a, tiles, s)));
  else XABE_TRY((launch_rows<2, false, 2, 4>(k, gate.quant, a, tiles, s)));
  a.w0 = static_cast<const uint8_t*>(down.bytes);
  a.w1 = nullptr;
  a.w_bytes = down.len;
  a.a = reinterpret_cast<const _Float16*>(b->shared_inter_h);
  a.out = out;
  a.K = (int)g.intermediate;
  a.n_rows = (int)g.hidden;
  a.parts = down_parts(g);
  a.planes = b->shared_inter;
  a.plane = g.max_tokens * g.hidden;
  wide = unrouted_down_wide(k, tokens, a.parts);
  a.tile_rows = wide ? unrouted_tile_rows(k, tokens, g.hidden / 256 * a.parts) : kNarrowRows;
  tiles = (g.max_tokens + a.tile_rows - 1) / a.tile_rows;
  *added = a.parts > 1;
  if (a.parts == 1) {
    if (wide) return launch_rows<1, false, 6, 8>(k, down.quant, a, tiles, s);
    return launch_rows<1, false, 2, 4>(k, down.quant, a, tiles, s);
  }
  if (wide) XABE_TRY((launch_parts<6, 8>(k, down.quant, a, tiles, s)));
  else XABE_TRY((launch_parts<2, 4>(k, down.quant, a, tiles, s)));
  hipLaunchKernelGGL(k_add_parts, dim3((unsigned)g.max_tokens, (unsigned)((g.hidden + 1023) / 1024)), dim3(256), 0, s, a.planes, a.plane,
                     a.parts, b->valid_tokens, (int)g.hidden, residual, out, l_out);
  XABE_HIP_TRY(hipGetLastError());
  return XABE_OK;
}

}  // namespace xabe
