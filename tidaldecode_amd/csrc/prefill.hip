// Causal attention of the n_q newest tokens of a sequence over its paged KV cache (prefill) for
// gfx950 (MI355X), on the matrix cores.  Replaces BatchPrefillWithPagedKVCache of the reference
// (kernels/include/prefill/prefill.cuh:674-870, bound in tidal/ops/csrc/batch_prefill.cu:27-117).
//
// What bounds it.  A long prompt is a contraction (4 n^2 / 2 flops per head dimension and head), so the
// matrix cores; but per 64 keys and 32 query rows the softmax costs a wave nearly as much as the two
// products (some 130 instructions of exp2, fma and pack, exp2 at a quarter of the rate, against 1024 cycles of
// MFMA), so the two have to run at the same time: 1567 cycles pass per wave and tile, the matrix cores being
// busy for 65 % of them.  A short prompt or a further turn on a long cache has few query rows and is bound by how many
// CUs have work at all.  Hence:
//   - The query rows of all heads of a KV head are packed into one list of rows (token * group + head),
//     cut into workgroup tiles of up to 256: grouped heads share every staged key, and 16 new tokens of four
//     heads fill 64 rows instead of four quarter-empty tiles.
//   - The keys of a row tile are cut into pieces when the tiles alone leave CUs idle (plan_prefill);
//     prefill_merge_kernel adds the pieces up.
//   - Eight waves of 32 rows, two per SIMD in opposite phases: one multiplies while the other forms
//     weights (see "the steps" in the kernel).  S^T = K Q^T and O^T = V^T P^T with 32x32x16 MFMA: the
//     query row is the lane in both results, so P stays in registers and the row maximum and sum cross
//     one pair of lanes.
//   - Key tiles go from memory to LDS without passing through registers, into rings of four (K) and five
//     (V) tiles; a piece is asked for three to four tiles before it is needed.
// LDS layout: gfx950 serves 256 bytes a cycle, and lanes {0-3, 12-15, 20-27} of a 16-byte read together
// (measured), so those 16 lanes must hit 16 different bank groups.  head_dim 128: four rows form a block
// of 1024 + 16 bytes and piece p of row r lies at p ^ 4 (r % 4); head_dim 64: rows of 128 bytes, pieces
// of K at p ^ ((r / 2) % 8), of V (read transposed, eight bytes a lane) at p ^ 4 ((r / 2) % 2).
// Measured in turn on one card (bf16, pages of 16, us, before with one 128- or 256-row tile per query head and
// 16x16x32 MFMA -> now): prompt of 32768 x 32 heads 8633 -> 7592 (1159 TFLOP/s; a 16384^3 library GEMM reached
// 1332 in the same run, and cards differ by 7 %), 8192 x 32 over 8 KV heads 588 -> 495, 1000 x 32 36.6 -> 24.0,
// 300 x 32 14.1 -> 9.8 (staged kernel, two key groups: bound by the latency of five steps and cold code); 500 new tokens on 32768
// cached ones, 32 heads 991 -> 285, over 8 KV heads 993 -> 252; 16 tokens, 8 KV heads 792 -> 33.
// Rows past the end of the sequence are clamped (never out of the pool) and masked.

#include <type_traits>

#include "common.cuh"
#include "../../include/tidal_hip.h"

namespace tidal {


// LDS read with transpose (gfx950): within every 16 lanes, lane 4a + b receives element b of the
// four 8-byte pieces addressed by lanes a, a + 4, a + 8, a + 12.
typedef short i16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 lds_read_tr16(const uint16_t* at) {
  const i16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) i16x4*)(at));
  return __builtin_bit_cast(u32x2, v);
}

// 16 bytes per lane from memory (scalar base + lane offset, or a lane address) to LDS bytes
// lds + 16 lane.  As asm: the compiler would wait for the load before every later LDS read.
// It inserts no wait states inside the asm, so they stand there: one between m0 and the load, and five
// between a scalar register that a vector instruction (v_readlane) wrote and the load that reads it.
// (m0 is a register the compiler allocates to no variable, which it warns about; it does set m0 for
// instructions of its own, and the list tells it that the value is gone.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_lds(uint32_t lds, uint64_t base, uint32_t offset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(lds), "v"(offset), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void load_lds(uint32_t lds, uint64_t at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(lds), "v"(at) : "memory", "m0");
}
#pragma clang diagnostic pop

// A lane's share of a tile's row sum (32 weights).  A weight of 1 is exact in 16 bits and a larger one is
// rounded, so a low limit keeps a row's largest weights exact.  At 64 the scores of normalised queries and
// keys exceed it in a row's first tile only (32768 tokens x 32 heads: no difference in time to 16384), and
// against 64 bits the error of queries four times as large is 1.8e-3 - 2.1e-3 in bf16, where a limit of 16384
// gave 2.0e-3 - 2.3e-3.
constexpr float kTopWeight = 64.f;

constexpr int kSgMfma = 0x8, kSgRead = 0x100;  // instruction classes of sched_group_barrier

constexpr float kRowFloor = -1.0e20f;  // below every score, far above a masked one (kNegBig)

// n / d for 0 <= n < 2^31 (round-up division by a constant: magic = ceil(2^(31 + down) / d), down =
// ceil(log2 d)).  The compiler's own division is some 20 dependent instructions, and every wave began with
// eight: prompts of 16 to 300 tokens, 32 heads, 6.7 -> 6.5 to 11.4 -> 11.2 us, 16 heads of 256 5.5 -> 5.1 to
// 17.0 -> 16.4.
struct Divisor {
  uint32_t magic, down;
};
static Divisor divisor(int d) {
  Divisor f = {0, 0};
  while (((int64_t)1 << f.down) < d) ++f.down;
  f.magic = (uint32_t)((((uint64_t)1 << (31 + f.down)) + (uint64_t)d - 1) / (uint64_t)d);
  return f;
}
__device__ __forceinline__ int operator/(int n, const Divisor& f) {
  return (int)(__umulhi(2u * (uint32_t)n, f.magic) >> f.down);
}

struct PrefillParams {
  const uint16_t* kv;
  int64_t page_stride, v_offset;  // elements
  int32_t entry_stride, head_stride, page_size;
  uint32_t entry_stride_b;                 // bytes
  Divisor by_page, by_group, by_kv, by_tiles, by_head;  // page_size, q_per_kv, n_kv, n_tiles, n_tiles * n_splits
  uint32_t max_page;
  const int32_t* page_table;
  int32_t n_pages, kv_len;
  const uint16_t* q;
  uint16_t* o;
  int32_t n_q, num_qo_heads, q_per_kv;
  float scale_log2;
  int32_t causal;
  // The work of a KV head: n_rows = n_q * q_per_kv query rows (row = token * q_per_kv + head of the
  // group), n_tiles workgroup tiles of bm of them, each cut into n_splits pieces of `chunk` keys.
  int32_t n_kv, n_rows, bm, n_tiles, n_splits, chunk, head_major;
  bool staged;     // prefill_attn_staged_kernel
  int32_t key_groups;  // of it: 1 or 2
  float lag;           // of it: log2 of the largest weight a row may have before its reference point moves
  float* part_o;   // [n_splits][n_kv * n_rows][D]: un-normalised partial results (n_splits > 1)
  float* part_ml;  // [n_splits][n_kv * n_rows][2]: running maximum (base 2) and denominator
};

// keys that the rows of a tile see together: up to the position of its last query row
__device__ __forceinline__ int tile_kv_end(const PrefillParams& p, int qtile) {
  int last_row = (qtile + 1) * p.bm - 1;
  last_row = last_row < p.n_rows ? last_row : p.n_rows - 1;
  return p.causal ? p.kv_len - p.n_q + last_row / p.by_group + 1 : p.kv_len;
}

// Where a workgroup's piece of the work lies.
struct PrefillPiece {
  int kvh, split, q0;      // KV head, piece of the keys, first query row
  int k_begin, k_end;      // keys of the piece
  bool whole;              // the tile has this piece alone: the result goes to o
};
__device__ __forceinline__ bool prefill_piece(const PrefillParams& p, PrefillPiece& w) {
  // Workgroups go to the eight XCDs round-robin by linear id, and each XCD has its own L2.  Many
  // tiles (head_major): all tiles of a KV head go to one XCD, one head after the other, so that its L2
  // streams one head's K/V.  Few tiles: the heads alternate and all of them start with their longest
  // tile, so that no long tile starts last.  (Placement only decides what the L2 holds and when a
  // workgroup starts; results do not depend on it.)
  const int lin = blockIdx.x;
  int rem;
  if (p.head_major) {
    const int slot = lin >> 3, idx = slot / p.by_head;  // which of this XCD's heads
    w.kvh = idx * 8 + (lin & 7);
    rem = slot - idx * p.n_tiles * p.n_splits;
  } else {
    rem = lin / p.by_kv;
    w.kvh = lin - rem * p.n_kv;
  }
  // The first pieces of all tiles before the second ones: full-length pieces come first and the shortest
  // last.  (Tile by tile, a short tile's only piece starts last and is as long as any: 16 heads of 256,
  // pieces of half the keys, 1400 tokens 63 -> 55 us, 2000 119 -> 81; 28 / 4 heads of 64, 2000 50 -> 38.)
  w.split = rem / p.by_tiles;
  const int qtile = p.n_tiles - 1 - (rem - w.split * p.n_tiles);
  w.q0 = qtile * p.bm;
  const int end = tile_kv_end(p, qtile);
  w.k_begin = __builtin_amdgcn_readfirstlane(w.split * p.chunk);
  w.k_end = end - w.k_begin > p.chunk ? w.k_begin + p.chunk : end;
  w.whole = end <= p.chunk;
  return w.k_begin < end;  // false: this tile has fewer pieces
}

// head_dim 64 and 128: eight waves, 32 query rows each, key tiles of 64 tokens.
// OCT: pages hold a multiple of eight tokens, so eight aligned tokens share a page: one page lookup per
// wave and tile, made 64 tiles at a time.  Other page sizes look up a page per row (8192 x 28 heads
// over 4: 477 us at pages of 1 and 476 at 4 against 441 at 16).
template <typename T, int D, bool OCT>
__global__ __launch_bounds__(512, 2) void prefill_attn_kernel(const PrefillParams p) {
  constexpr int BN = 64, NS = D / 16, DB = D / 32;
  // LDS: rings of RK key tiles and RV value tiles (values are read half a step later than keys)
  constexpr int RK = 4, RV = 5, NL = D / 64;         // NL: loads per lane, tile and matrix
  constexpr int BLK = D == 128 ? 1040 : 1024;        // bytes from one load's block to the next
  constexpr int TILE_B = BN / (512 / D) * BLK;       // a block holds 512 / D rows
  __shared__ __attribute__((aligned(16))) char smem[(RK + RV) * TILE_B];

  // the wave index is made scalar: the activity tests below must be real branches, because matrix
  // instructions do not honour the EXEC mask of a masked-off region
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, h = lane >> 5;
  const int late = wave >> 2;  // 0: the first of the two waves of a SIMD, 1: the second, a phase behind

  PrefillPiece w;
  if (!prefill_piece(p, w)) return;  // uniform
  const int q_off = p.kv_len - p.n_q;     // position of query token 0
  const int row0 = w.q0 + wave * 32;      // first query row of the wave
  const int row_end = w.q0 + p.bm < p.n_rows ? w.q0 + p.bm : p.n_rows;  // behind the last of the workgroup

  // ---- Q operand: row (row0 + c), pieces [16 s + 8 h, +8) --------------------------------------
  int row = row0 + c;
  row = row < row_end ? row : row_end - 1;
  const int tok = row / p.by_group;
  const int64_t o_at = ((int64_t)tok * p.num_qo_heads + w.kvh * p.q_per_kv + (row - tok * p.q_per_kv)) * D;
  int row_lim = p.kv_len - 1;  // last token this row sees
  if (p.causal && q_off + tok < row_lim) row_lim = q_off + tok;
  u32x4 qb[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) qb[s] = *reinterpret_cast<const u32x4*>(p.q + o_at + 16 * s + 8 * h);
  const int wave_first_pos = q_off + row0 / p.by_group;  // position of the wave's first query row

  // ---- staging: rows go from memory straight into LDS -------------------------------------------
  // A wave brings rows 8 wave .. 8 wave + 7 of a tile, one KB (a block) per load: lane l fills bytes
  // 16 l .. 16 l + 15 of the block and so chooses, by what it fetches, which piece of which row lies
  // there (the swizzle).
  constexpr int RPB = 512 / D, CPR = D / 8;  // rows per block, 16-byte pieces per row
  const int rb = lane / CPR;                 // row of the block that this lane fetches a piece of
  uint32_t piece_k, piece_v;                 // and the byte offset of the piece
  if constexpr (D == 128) {
    piece_k = piece_v = (uint32_t)((lane & 15) ^ (4 * rb)) * 16;
  } else {
    piece_k = (uint32_t)((lane & 7) ^ ((4 * wave + (rb >> 1)) & 7)) * 16;
    piece_v = (uint32_t)((lane & 7) ^ (4 * ((rb >> 1) & 1))) * 16;
  }
  const uint32_t smem_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const uint64_t k_base = (uint64_t)(uintptr_t)(p.kv + (int64_t)w.kvh * p.head_stride);
  const int last_tok = p.kv_len - 1;
  auto page_of = [&](int t) { return t / p.by_page; };
  // OCT: first token of the wave's rows of tile j (tiles past the end repeat the last tokens: the loads need
  // no branch and what they bring is masked)
  auto first_tok = [&](int j) {
    const int t = w.k_begin + j * BN + 8 * wave;
    return t < last_tok ? t : last_tok & ~7;
  };
  // Row addresses are formed for several tiles at once, one per lane.  OCT (the wave's eight rows of a
  // tile share a page): lane l holds the offset of the first row of tile (j & ~63) + l, which is
  // broadcast when that tile is brought; the other rows lie at fixed distances, except in the tiles from
  // `tail_from` on, whose rows end with the sequence.  Otherwise lane l holds the page of row l % 8 of
  // tile (j & ~7) + l / 8, and `ahead` those of the eight tiles after that.
  uint32_t addr_lo = 0, addr_hi = 0;
  int pages = 0, ahead = 0;
  const int tail_from = (last_tok - 7 - w.k_begin - 8 * wave + BN) >> 6;
  uint32_t row_at[NL];
#pragma unroll
  for (int x = 0; x < NL; ++x) row_at[x] = (uint32_t)(RPB * x + rb) * p.entry_stride_b;
  auto page_at = [&](int t) {
    const uint32_t page = (uint32_t)p.page_table[page_of(t)];
    return page > p.max_page ? p.max_page : page;
  };
  // brings tile j to the ring slots at LDS bytes k_to and v_to
  auto bring = [&](int j, uint32_t k_to, uint32_t v_to) __attribute__((always_inline)) {
    k_to += NL * wave * BLK;
    v_to += NL * wave * BLK;
    if constexpr (OCT) {
      if ((j & 63) == 0) {
        const int t = first_tok(j + lane);
        const uint64_t at = k_base + (uint64_t)page_at(t) * (uint64_t)(p.page_stride * 2) +
                            (uint64_t)(uint32_t)(t - page_of(t) * p.page_size) * p.entry_stride_b;
        addr_lo = (uint32_t)at;
        addr_hi = (uint32_t)(at >> 32);
      }
      const uint64_t k_row = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(addr_lo, j & 63) |
                             (uint64_t)(uint32_t)__builtin_amdgcn_readlane(addr_hi, j & 63) << 32;
      const uint64_t v_row = k_row + (uint64_t)p.v_offset * 2;
      uint32_t at[NL];
#pragma unroll
      for (int x = 0; x < NL; ++x) at[x] = row_at[x];
      if (__builtin_expect(j >= tail_from, 0)) {
        const int lim = last_tok - first_tok(j);
#pragma unroll
        for (int x = 0; x < NL; ++x)
          at[x] = (uint32_t)(RPB * x + rb < lim ? RPB * x + rb : lim) * p.entry_stride_b;
      }
#pragma unroll
      for (int x = 0; x < NL; ++x) {
        load_lds(k_to + x * BLK, k_row, at[x] + piece_k);
        load_lds(v_to + x * BLK, v_row, at[x] + piece_v);
      }
    } else {
      auto page_of_lane = [&](int j8) {
        const int t = w.k_begin + (j8 + (lane >> 3)) * BN + 8 * wave + (lane & 7);
        return (int)page_at(t < last_tok ? t : last_tok);
      };
      if ((j & 7) == 0) {
        pages = j == 0 ? page_of_lane(0) : ahead;
        asm volatile("" : "+v"(pages));  // waited for here and not, with everything else, in every step
        ahead = page_of_lane(j + 8);
      }
      const int t0 = w.k_begin + j * BN + 8 * wave;
#pragma unroll
      for (int x = 0; x < NL; ++x) {
        // the token whose page page_of_lane looked up: rows past the end are the last token's
        const int t = t0 + RPB * x + rb < last_tok ? t0 + RPB * x + rb : last_tok;
        const uint32_t page = (uint32_t)__shfl(pages, 8 * (j & 7) + RPB * x + rb, 64);
        const uint64_t row = (uint64_t)page * (uint64_t)(p.page_stride * 2) +
                             (uint64_t)(uint32_t)(t - page_of(t) * p.page_size) * p.entry_stride_b;
        load_lds(k_to + x * BLK, k_base + row + piece_k);
        load_lds(v_to + x * BLK, k_base + (uint64_t)p.v_offset * 2 + row + piece_v);
      }
    }
  };

  // ---- the two matrix products and the softmax between them --------------------------------------
  f32x16 st[2], oacc[DB];
  u32x4 pa[4];
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[b][v] = 0.f;
  float m_run = kNegBig, l_run = 0.f;

  // S^T = K Q^T, two halves of 32 tokens; the first PRE operands were read in the phase before
  constexpr int PRE = 4;
  u32x4 kpre[PRE];
  uint32_t k_lane[4], v_lane[DB];  // byte offsets of this lane's pieces in a tile
  {
    const int r = c & 3, vr = (lane & 15) >> 2, q = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
#pragma unroll
    for (int a = 0; a < 4; ++a)
      k_lane[a] = D == 128 ? (c >> 2) * BLK + r * 256 + 16 * h + 64 * (a ^ r)
                           : c * 128 + ((16 * h + 32 * a) ^ (16 * ((c >> 1) & 7)));
#pragma unroll
    for (int b = 0; b < DB; ++b)
      v_lane[b] = 16 * q + 8 * (lane & 1) +
                  (D == 128 ? h * BLK + vr * 256 + 64 * (b ^ vr) : (4 * h + vr) * 128 + 64 * (b ^ (vr >> 1)));
  }
  // operand x of the scores: 16 dimensions (x / 2) of 32 keys (x % 2)
  auto k_operand = [&](const uint32_t (&at)[4], int x) {
    const int s = x >> 1, t = x & 1;
    const uint32_t off = D == 128 ? at[s >> 1] + 32 * (s & 1) + 8 * BLK * t : at[s & 3] + 4096 * t;
    return *reinterpret_cast<const u32x4*>(smem + off);
  };
  auto prefetch = [&](uint32_t kslot) {
    uint32_t at[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) at[a] = k_lane[a] + kslot;
#pragma unroll
    for (int x = 0; x < PRE; ++x) kpre[x] = k_operand(at, x);
  };
  auto scores = [&](uint32_t kslot) {
    uint32_t at[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) at[a] = k_lane[a] + kslot;
    const f32x16 zero = {};
#pragma unroll
    for (int x = 0; x < 2 * NS; ++x) {
      const u32x4 ka = x < PRE ? kpre[x] : k_operand(at, x);
      st[x & 1] = mfma_32x32x16<T>(ka, qb[x >> 1], x < 2 ? zero : st[x & 1]);
    }
  };
  // O^T += V^T P^T
  auto weigh = [&](uint32_t vslot) {
    uint32_t at[DB];
#pragma unroll
    for (int b = 0; b < DB; ++b) at[b] = v_lane[b] + vslot;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int b = 0; b < DB; ++b) {
        const uint32_t off = at[b] + s * (16 / RPB) * BLK;
        const u32x2 t0 = lds_read_tr16(reinterpret_cast<const uint16_t*>(smem + off));
        const u32x2 t1 = lds_read_tr16(reinterpret_cast<const uint16_t*>(smem + off + 8 / RPB * BLK));
        oacc[b] = mfma_32x32x16<T>(u32x4{t0.x, t0.y, t1.x, t1.y}, pa[s], oacc[b]);
      }
  };
  // Order of a matrix phase: operands are read LEAD matrix instructions ahead of their use (left to
  // itself the compiler reads them one instruction ahead and waits).
  auto order_scores = [&]() {
    __builtin_amdgcn_sched_group_barrier(kSgRead, 2, 0);
#pragma unroll
    for (int x = 0; x < 2 * NS - PRE - 2; ++x) {
      __builtin_amdgcn_sched_group_barrier(kSgMfma, 1, 0);
      __builtin_amdgcn_sched_group_barrier(kSgRead, 1, 0);
    }
  };
  auto order_weigh = [&]() {
    __builtin_amdgcn_sched_group_barrier(kSgRead, 8, 0);
#pragma unroll
    for (int x = 0; x < 4 * DB - 4; ++x) {
      __builtin_amdgcn_sched_group_barrier(kSgMfma, 1, 0);
      __builtin_amdgcn_sched_group_barrier(kSgRead, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(kSgMfma, 4, 0);
  };
  auto order_both = [&]() {
    __builtin_amdgcn_sched_group_barrier(kSgRead, 2, 0);
#pragma unroll
    for (int x = 0; x < 2 * NS - PRE - 2; ++x) {
      __builtin_amdgcn_sched_group_barrier(kSgMfma, 1, 0);
      __builtin_amdgcn_sched_group_barrier(kSgRead, 1, 0);
    }
#pragma unroll
    for (int x = 0; x < PRE + 4 * DB - 2; ++x) {  // the scores' last products, then the weights'
      __builtin_amdgcn_sched_group_barrier(kSgMfma, 1, 0);
      __builtin_amdgcn_sched_group_barrier(kSgRead, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(kSgMfma, 4, 0);
  };
  // first tile in which a row of the wave sees less than all keys
  int mask_from = (p.kv_len - BN - w.k_begin) >> 6;
  if (p.causal) {
    const int m = (wave_first_pos - (BN - 1) - w.k_begin) >> 6;
    mask_from = m < mask_from ? m : mask_from;
  }
  mask_from += 1;
  auto first_key = [&](int i) { return w.k_begin + i * BN; };
  // P = 2^(s scale - m_run), its row sums (of this lane's half of the keys)
  auto weights = [&]() __attribute__((always_inline)) {
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        uint32_t pk[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = fast_exp2(fmaf(st[t][8 * u + 2 * e], p.scale_log2, -m_run));
          const float b = fast_exp2(fmaf(st[t][8 * u + 2 * e + 1], p.scale_log2, -m_run));
          pk[e] = pack2<T>(a, b);
          sum[0] += a;
          sum[1] += b;
        }
        pa[2 * t + u] = u32x4{pk[0], pk[1], pk[2], pk[3]};
      }
    float all = sum[0] + sum[1];
    asm volatile("" : "+v"(all));  // here, not where the next phase would have to keep its summands
    return all;
  };
  // The reference point m_run is the row's maximum of some earlier tile: softmax does not depend on it.
  // So a tile's maximum is formed only when its weights turn out larger than kTopWeight (and in the first
  // tile, where m_run is no score yet); then the accumulators are rescaled and the weights formed again.
  auto softmax = [&](int i) __attribute__((always_inline)) {
    if (__builtin_expect(i >= mask_from, 0)) {
      int lim = row_lim - first_key(i) - 4 * h;
      asm volatile("" : "+v"(lim));  // keeps the 32 differences of the comparisons out of the loop's registers
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          st[t][v] = 32 * t + 8 * (v / 4) + v % 4 <= lim ? st[t][v] : kNegBig;
    }
    float l_tile = weights();
    if (__builtin_expect(__ballot(!(l_tile <= kTopWeight)) != 0, 0)) {
      float mx = kRowFloor;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 16; v += 2) mx = fmaxf(fmaxf(st[t][v], st[t][v + 1]), mx);
      float lo, hi;
      swap_halves32(mx, lo, hi);
      const float m_new = fmaxf(fmaxf(lo, hi) * p.scale_log2, m_run);
      const float alpha = fast_exp2(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) oacc[b][v] *= alpha;
      l_tile = weights();
    }
    l_run += l_tile;
  };

  const int nt = __builtin_amdgcn_readfirstlane((w.k_end - w.k_begin + BN - 1) / BN);
  // tiles that hold keys for the wave's own rows; a wave goes through one even if it has none
  int own = nt;
  if (p.causal) {
    const int last_row = row0 + 31 < row_end ? row0 + 31 : row_end - 1;
    const int mine = (q_off + last_row / p.by_group - w.k_begin) / BN + 1;
    own = mine < nt ? mine : nt;
  }
  if (row0 >= row_end || own < 1) own = 1;
  own = __builtin_amdgcn_readfirstlane(own);
  auto phase_end = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- the steps ----------------------------------------------------------------------------------
  // The two waves of a SIMD take turns, half a step apart: while one forms the scores of its next tile
  // and the weighted values of its last one (matrix phase), the other turns scores into weights (vector
  // phase); a barrier ends every half step.  Both walk the same tiles in LDS:
  //   half step      2i            2i + 1         2i + 2
  //   early wave     matrix i      vector i       matrix i + 1        matrix i: scores i, values i - 1
  //   late wave      vector i - 1  matrix i       vector i
  // A wave asks for its rows of tile i + 3 (late: i + 4) in vector phase i, which is when the last
  // reader has left the ring slots that they go to, and has them by the end of matrix phase i + 2
  // (late: i + 2), before the early waves read the first operands of tile i + 3 at the end of vector
  // phase i + 2.  A wave stops computing after its own last tile (a causal workgroup tile has four to go
  // on its diagonal) and then only brings its share of the rows: 15.2 -> 13.5 us for 300 tokens x 32 heads.
  constexpr uint32_t K_END = RK * TILE_B, V_END = K_END + RV * TILE_B;
  uint32_t kr = 0, vr = V_END - TILE_B;  // ring slots of K(i) and V(i - 1)
  // ring slots of the tile that is asked for next
  uint32_t kw = (3 + late) % RK * TILE_B, vw = K_END + (3 + late) % RV * TILE_B;
  auto next_k = [&](uint32_t slot) { return slot == K_END - TILE_B ? 0u : slot + TILE_B; };
  auto next_v = [&](uint32_t slot) { return slot == V_END - TILE_B ? K_END : slot + TILE_B; };
  auto matrix_done = [&]() {
    __builtin_amdgcn_s_setprio(0);
    // the wave's operands have been read, and all rows it asked for but those of the youngest tile are there
    if constexpr (NL == 2)
      asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)" ::: "memory");
    phase_end();
  };
  auto bring_next = [&](int i) __attribute__((always_inline)) {  // of vector phase i
    bring(i + 3 + late, smem_at + kw, smem_at + vw);
    kw = next_k(kw);
    vw = next_v(vw);
  };
#pragma unroll
  for (int j = 0; j < 3; ++j) bring(j, smem_at + j * TILE_B, smem_at + K_END + j * TILE_B);
  if (late) bring(3, smem_at + 3 * TILE_B, smem_at + K_END + 3 * TILE_B);
  if constexpr (NL == 2)
    asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  else
    asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
  phase_end();
  prefetch(0);
  if (late) phase_end();
  scores(0);
  order_scores();
  matrix_done();
  for (int i = 0; i < own - 1; ++i) {
    kr = next_k(kr);
    vr = next_v(vr);
    bring_next(i);
    prefetch(kr);
    softmax(i);
    phase_end();
    __builtin_amdgcn_s_setprio(1);
    scores(kr);
    weigh(vr);
    order_both();
    matrix_done();
  }
  vr = next_v(vr);
  if (own < nt) bring_next(own - 1);
  softmax(own - 1);
  if (own < nt || !late) phase_end();
  weigh(vr);
  order_weigh();
  if (own < nt) {  // the other waves still need this one's share of the rows
    matrix_done();
    for (int i = own; i < nt - 1; ++i) {
      bring_next(i);
      phase_end();
      matrix_done();
    }
    if (!late) phase_end();
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing is on its way to LDS when the workgroup ends

  // ---- normalise and store (or leave the piece's partial result): a lane holds dimensions
  //      32 b + 8 (v / 4) + 4 h + v % 4 of its row ---------------------------------------------------
  float l0, l1;
  swap_halves32(l_run, l0, l1);
  const float l = l0 + l1;
  if (row0 + c >= row_end) return;
  if (w.whole) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int v = 0; v < 16; v += 4)
        *reinterpret_cast<u32x2*>(p.o + o_at + 32 * b + 2 * v + 4 * h) =
            u32x2{pack2<T>(oacc[b][v] * inv, oacc[b][v + 1] * inv),
                  pack2<T>(oacc[b][v + 2] * inv, oacc[b][v + 3] * inv)};
  } else {
    const int64_t part = ((int64_t)w.split * p.n_kv + w.kvh) * p.n_rows + row0 + c;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int v = 0; v < 16; v += 4)
        *reinterpret_cast<f32x4*>(p.part_o + part * D + 32 * b + 2 * v + 4 * h) =
            f32x4{oacc[b][v], oacc[b][v + 1], oacc[b][v + 2], oacc[b][v + 3]};
    if (h == 0) *reinterpret_cast<f32x2*>(p.part_ml + part * 2) = f32x2{m_run, l};
  }
}

// head_dim 256, whose output alone would take 128 registers of a wave in the kernel above; short caches (see
// plan_prefill); and pools that are not 16-byte aligned, which direct loads to LDS are not specified for: four
// waves of 16 query rows and 16x16x32 MFMA, 32 tokens per key tile.  KG = 2: four more waves with buffers of
// their own take every other key tile of the same rows, and the two halves meet in LDS at the end.
// K/V tiles pass through registers into two LDS buffers per matrix, one barrier per tile; LDS rows are
// padded by 32 bytes, which keeps the 16-byte K reads and the transposed V reads free of bank conflicts.
// A step is a serial chain (scores, weights, values, barrier), so two workgroups share a compute unit: within
// 256 registers (186) instead of 328 with accumulators copied between register files, whole tiles of 16
// heads, bf16, take 45.1 us instead of 47.1 for 1000 tokens, 142 instead of 202 for 2900, 497 instead of
// 751 for 6000.
template <typename T, int D, int KG>
__device__ __forceinline__ void staged_attention(const PrefillParams& p) {
  constexpr int WR = 16;            // query rows per wavefront
  constexpr int NS = D / 32;        // 16-byte pieces of a Q/K row per lane (one MFMA each)
  constexpr int DC = D / 16;        // head dimensions per lane in the P.V product
  constexpr int PITCH = D + 16;     // LDS row pitch in elements: +32 bytes
  constexpr int CPR = D / 8;        // 16-byte chunks per row
  constexpr int BN = 32;            // tokens per key tile
  constexpr int NSUB = BN / 16;     // 16-token sub-tiles per key tile
  constexpr int CPT = CPR / 8;      // staging: chunks per thread, tile and matrix (row = tid / 8,
                                    // chunk = tid % 8 + 8 jc)
  static_assert(D % 64 == 0, "a thread stages whole pieces");
  constexpr int STEP = BN * KG;     // tokens from one tile of a key group to its next
  // two buffers per matrix and key group: tile t + 1 is written while tile t is still being read
  constexpr int TILE = BN * PITCH;
  __shared__ __attribute__((aligned(16))) uint16_t sm[KG][4 * TILE];

  // the wave index is made scalar: the per-tile activity tests below must be real branches, because
  // matrix instructions do not honour the EXEC mask of a masked-off region
  const int tid = threadIdx.x & 255, lane = tid & 63;  // inside the key group
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) & 3);
  const int kg = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8));
  uint16_t* const ks = sm[kg];
  uint16_t* const vs = sm[kg] + 2 * TILE;
  const int r = lane & 15, g = lane >> 4;
  PrefillPiece w;
  if (!prefill_piece(p, w)) return;  // uniform
  const int kvh = w.kvh, split = w.split, q0 = w.q0, k_begin = w.k_begin, kv_end = w.k_end;
  const bool whole = w.whole;
  const int q_off = p.kv_len - p.n_q;  // position of query token 0

  // ---- Q operand: row (q0 + 16 wave + r), pieces [32 s + 8 g, +8) -------------------------------
  int q_row = q0 + wave * WR + r;
  q_row = q_row < p.n_rows ? q_row : p.n_rows - 1;
  const int q_tok = q_row / p.by_group;
  const int qpos = q_off + q_tok;  // position of this lane's query row
  const u32x4* q_src = reinterpret_cast<const u32x4*>(
      p.q + ((int64_t)q_tok * p.num_qo_heads + kvh * p.q_per_kv + (q_row - q_tok * p.q_per_kv)) * D);
  u32x4 qb[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) qb[s] = q_src[4 * s + g];

  f32x4 oacc[DC];
  float m_run = kNegBig, l_run = 0.f;
#pragma unroll
  for (int d = 0; d < DC; ++d) oacc[d] = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- staging: thread -> CPT chunks of K and of V per tile --------------------------------------
  // eight adjacent lanes move 128 contiguous bytes of one row (one cache line in, one conflict-free
  // LDS write out); a thread looks up the page of its row once
  // Two register sets for keys: the loads of tile t + 2 are issued while tile t + 1 still waits in the
  // other set for its turn to be written to LDS, so its rows have two iterations to arrive.  Values have
  // one set and one iteration: a second set would not fit 256 registers, and with more a compute unit
  // holds one workgroup instead of two and accumulators are moved between register files in every step.
  u32x4 kreg_a[CPT], kreg_b[CPT], vreg[CPT];
  const int srow = tid >> 3, sl8 = tid & 7;
  // page ids are looked up one tile ahead of the rows they address, so that a tile's loads never wait
  // for a page-table load issued in the same iteration
  uint32_t pg, pg_v;  // of the next tile of keys, of values
  auto split_tok = [&](int kt, int& pg_i, int& entry) {
    int tok = kt + srow;
    tok = tok < p.kv_len ? tok : p.kv_len - 1;
    pg_i = tok / p.by_page;
    entry = tok - pg_i * p.page_size;
  };
  auto lookup = [&](int kt) {
    int pg_i, entry;
    split_tok(kt, pg_i, entry);
    pg = (uint32_t)p.page_table[pg_i];
  };
  auto fetch = [&](int kt, uint32_t page, int64_t matrix, u32x4 (&reg)[CPT]) {
    int pg_i, entry;
    split_tok(kt, pg_i, entry);
    page = page > p.max_page ? p.max_page : page;
    const uint16_t* src = p.kv + (matrix + (int64_t)page * p.page_stride + (int64_t)entry * p.entry_stride +
                                  (int64_t)kvh * p.head_stride + sl8 * 8);
#pragma unroll
    for (int jc = 0; jc < CPT; ++jc) reg[jc] = *reinterpret_cast<const u32x4*>(src + jc * 64);
  };
  auto fetch_v = [&](int kt) { fetch(kt, pg_v, p.v_offset, vreg); };
  auto fetch_k = [&](int kt, u32x4 (&kreg)[CPT]) {  // needs lookup(kt) before it; fetch_v(kt) comes after it
    fetch(kt, pg, 0, kreg);
    pg_v = pg;
    lookup(kt + STEP);
  };
  auto stash = [&](int buf, const u32x4 (&kreg)[CPT]) {
#pragma unroll
    for (int jc = 0; jc < CPT; ++jc) {
      const int at = buf * TILE + srow * PITCH + (sl8 + 8 * jc) * 8;
      *reinterpret_cast<u32x4*>(&ks[at]) = kreg[jc];
      *reinterpret_cast<u32x4*>(&vs[at]) = vreg[jc];
    }
  };

  // positions of the wave's first and last query row (a wave without rows sees no key tile)
  const int wave_row0 = q0 + wave * WR;
  const int wave_first_pos = q_off + wave_row0 / p.by_group;
  const int wave_last_pos = wave_row0 < p.n_rows ? (p.causal ? q_off + (wave_row0 + WR - 1) / p.by_group : p.kv_len) : -1;
  auto compute = [&](int kt, int buf) {
    // A wave whose last query row lies before the key tile sees none of it (causal).  In an active wave a
    // row that lies wholly before the key tile is masked to zero weight below.
    if (kt <= wave_last_pos && (KG == 1 || kt < kv_end)) {
      // ---- S^T = K Q^T ---------------------------------------------------------------------------
      // (the two matrix phases run at raised wave priority: while one wave of a SIMD is in its
      // softmax arithmetic, the other's matrix instructions are issued first and keep the matrix
      // pipeline busy)
      __builtin_amdgcn_s_setprio(2);
      f32x4 st[NSUB];  // raw q.k; the softmax scale is folded into the exponent below
#pragma unroll
      for (int sub = 0; sub < NSUB; ++sub) {
        u32x4 ka[NS];
        const uint16_t* krow = &ks[buf * TILE + (sub * 16 + r) * PITCH + 8 * g];
#pragma unroll
        for (int s = 0; s < NS; ++s) ka[s] = *reinterpret_cast<const u32x4*>(krow + 32 * s);
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NS; ++s) acc = mfma_16x16x32<T>(ka[s], qb[s], acc);
        st[sub] = acc;
      }
      __builtin_amdgcn_s_setprio(0);
      // ---- online softmax of query row r (lanes r, r+16, r+32, r+48 share the row) ---------------
      if ((p.causal && kt + BN - 1 > wave_first_pos) || kt + BN > p.kv_len) {
        // the last token this row sees, counted from the lane's first one of the tile (opaque: the
        // compiler would keep the differences of the comparisons below in registers for the loop)
        int lim = p.kv_len - 1;
        if (p.causal && qpos < lim) lim = qpos;
        lim -= kt + 4 * g;
        asm volatile("" : "+v"(lim));
#pragma unroll
        for (int sub = 0; sub < NSUB; ++sub)
#pragma unroll
          for (int i = 0; i < 4; ++i) st[sub][i] = sub * 16 + i <= lim ? st[sub][i] : kNegBig;
      }
      float t_max = kNegBig;
#pragma unroll
      for (int sub = 0; sub < NSUB; ++sub)
#pragma unroll
        for (int i = 0; i < 4; ++i) t_max = fmaxf(t_max, st[sub][i]);
      t_max = rows_max(t_max);
      // m_run is kept in the scaled base-2 domain.  A masked entry (kNegBig) gives exp2(-huge) = 0 by
      // itself, also in a tile that masks the whole row (a later piece of the keys may begin with
      // one): the reference point never falls to where kNegBig lies.
      // Softmax does not depend on the reference point, but a weight of 1 is exact in 16 bits and a larger one
      // is rounded.  So the reference lags a row's maximum by no more than 2^lag (p.lag), and the accumulator's
      // rescale stays rare.  With key groups a step is half as long: one row's move moves all rows of the wave.
      const float m_tile = fmaxf(t_max, kRowFloor) * p.scale_log2;
      const bool moves = KG == 1 ? m_tile > m_run + (D == 256 ? 8.f : p.lag) : __ballot(m_tile > m_run + p.lag) != 0;
      const float m_new = moves ? fmaxf(m_tile, m_run) : m_run;
      const float alpha = fast_exp2(m_run - m_new);
      m_run = m_new;
      uint32_t pa[NSUB][2];
      float psum = 0.f;
#pragma unroll
      for (int sub = 0; sub < NSUB; ++sub) {
        float pr[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          pr[i] = fast_exp2(fmaf(st[sub][i], p.scale_log2, -m_new));
          psum += pr[i];
        }
        pa[sub][0] = pack2<T>(pr[0], pr[1]);
        pa[sub][1] = pack2<T>(pr[2], pr[3]);
      }
      l_run = fmaf(l_run, alpha, psum);
      // rescale: accumulator row 4g + i is query row 4g + i, whose factor sits in lane 4g + i
      if (__ballot(alpha != 1.f)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float f = __shfl(alpha, 4 * g + i, 64);
#pragma unroll
          for (int d = 0; d < DC; ++d) oacc[d][i] *= f;
        }
      }
      __builtin_amdgcn_s_setprio(2);
      // ---- O += P V, 32 tokens (two sub-tiles) per matrix instruction ------------------------------
      // B operand of head dimensions [16 a, 16 a + 16): lane (r, g) needs dimension 16 a + r of the
      // tokens 4g..4g+3 of both sub-tiles.  ds_read_b64_tr_b16 transposes a 4 token x 16 dimension
      // block inside every 16 lanes: lane r points at the 8-byte piece r % 4 of token row r / 4
      // and receives dimension r of the four rows.
      const uint16_t* vlane = &vs[buf * TILE + (4 * g + (r >> 2)) * PITCH + 4 * (r & 3)];
      const u32x4 pp = {pa[0][0], pa[0][1], pa[1][0], pa[1][1]};
#pragma unroll
      for (int a = 0; a < DC; ++a) {
        const u32x2 t0 = lds_read_tr16(vlane + 16 * a);
        const u32x2 t1 = lds_read_tr16(vlane + 16 * PITCH + 16 * a);
        oacc[a] = mfma_16x16x32<T>(pp, u32x4{t0.x, t0.y, t1.x, t1.y}, oacc[a]);
      }
      __builtin_amdgcn_s_setprio(0);
    }
  };

  // first tile into buffer 0, keys of the second into register set a.  Key group kg takes the tiles kg,
  // kg + KG, ...; the groups keep step (the barriers are shared), so a group may be handed a tile past the
  // end: its rows are clamped, and compute leaves it alone.
  const int k_first = k_begin + kg * BN;
  lookup(k_first);
  fetch_k(k_first, kreg_a);
  fetch_v(k_first);
  stash(0, kreg_a);
  if (k_begin + STEP < kv_end) fetch_k(k_first + STEP, kreg_a);
  // One barrier per tile: it makes tile kt visible in its buffer, and it tells that every wave has
  // finished reading the other buffer, which the end of the step overwrites with the group's next tile.
  for (int k0 = k_begin; k0 < kv_end; k0 += 2 * STEP) {  // of key group 0
    const int kt = k0 + kg * BN;
    __syncthreads();
    if (k0 + STEP < kv_end) fetch_v(kt + STEP);
    if (k0 + 2 * STEP < kv_end) fetch_k(kt + 2 * STEP, kreg_b);
    compute(kt, 0);
    if (k0 + STEP >= kv_end) break;
    stash(1, kreg_a);
    __syncthreads();
    if (k0 + 2 * STEP < kv_end) fetch_v(kt + 2 * STEP);
    if (k0 + 3 * STEP < kv_end) fetch_k(kt + 3 * STEP, kreg_a);
    compute(kt + STEP, 1);
    if (k0 + 2 * STEP < kv_end) stash(0, kreg_b);
  }

  // ---- the key groups' results of a row meet in LDS: wave w of group 0 adds those of the waves w ------
  // (a group in which a row sees no key has denominator 0 and is left out, whatever its values are)
  const float l = rows_sum(l_run);
  float m_row[4], l_row[4];  // of rows 4 g + i
  if constexpr (KG > 1) {
    static_assert((KG - 1) * 4 * 16 * D * 4 <= KG * 4 * TILE * 2, "the partial results fit the tiles' LDS");
    __shared__ float sm_ml[KG][4][16][2];
    f32x4* const part = reinterpret_cast<f32x4*>(&sm[0][0]);
    __syncthreads();  // the last tiles have been read
    if (g == 0) {
      sm_ml[kg][wave][r][0] = m_run;
      sm_ml[kg][wave][r][1] = l;
    }
    if (kg > 0) {
#pragma unroll
      for (int a = 0; a < DC; ++a) part[(((kg - 1) * 4 + wave) * DC + a) * 64 + lane] = oacc[a];
    }
    __syncthreads();
    if (kg > 0) return;
    float f[KG][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float m[KG], l_of[KG], top = kNegBig;
#pragma unroll
      for (int j = 0; j < KG; ++j) {
        m[j] = sm_ml[j][wave][4 * g + i][0];
        l_of[j] = sm_ml[j][wave][4 * g + i][1];
        if (l_of[j] != 0.f) top = fmaxf(top, m[j]);
      }
      l_row[i] = 0.f;
      m_row[i] = top;
#pragma unroll
      for (int j = 0; j < KG; ++j) {
        f[j][i] = l_of[j] != 0.f ? fast_exp2(m[j] - top) : 0.f;
        l_row[i] = fmaf(l_of[j], f[j][i], l_row[i]);
      }
    }
#pragma unroll
    for (int a = 0; a < DC; ++a) {
#pragma unroll
      for (int i = 0; i < 4; ++i) oacc[a][i] = f[0][i] != 0.f ? oacc[a][i] * f[0][i] : 0.f;
#pragma unroll
      for (int j = 1; j < KG; ++j) {
        const f32x4 v = part[(((j - 1) * 4 + wave) * DC + a) * 64 + lane];
#pragma unroll
        for (int i = 0; i < 4; ++i) oacc[a][i] = f[j][i] != 0.f ? fmaf(v[i], f[j][i], oacc[a][i]) : oacc[a][i];
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      m_row[i] = __shfl(m_run, 4 * g + i, 64);
      l_row[i] = __shfl(l, 4 * g + i, 64);
    }
  }

  // ---- normalise and store (or leave the piece's partial result): lane holds rows 4g + i,
  //      dimensions 16 a + r ------------------------------------------------------------------------
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float li = l_row[i];
    const int row = wave_row0 + 4 * g + i;
    if (whole) {
      const float inv = li > 0.f ? 1.f / li : 0.f;
      if (row < p.n_rows) {
        const int tok = row / p.by_group;
        uint16_t* dst = p.o + ((int64_t)tok * p.num_qo_heads + kvh * p.q_per_kv + (row - tok * p.q_per_kv)) * D + r;
#pragma unroll
        for (int a = 0; a < DC; ++a) dst[16 * a] = from_float<T>(oacc[a][i] * inv);
      }
    } else {
      const float mi = m_row[i];
      if (row < p.n_rows) {
        const int64_t part = ((int64_t)split * p.n_kv + kvh) * p.n_rows + row;
        float* dst = p.part_o + part * D + r;
#pragma unroll
        for (int a = 0; a < DC; ++a) dst[16 * a] = oacc[a][i];
        if (r == 0) {
          p.part_ml[part * 2] = mi;
          p.part_ml[part * 2 + 1] = li;
        }
      }
    }
  }
}

template <typename T, int D>
__global__ __launch_bounds__(256, 2) void prefill_attn_staged_kernel(const PrefillParams p) {
  staged_attention<T, D, 1>(p);
}
template <typename T, int D>
__global__ __launch_bounds__(512, 2) void prefill_two_groups_kernel(const PrefillParams p) {
  staged_attention<T, D, 2>(p);
}

// Adds up the pieces of every row whose keys were split: D / 4 adjacent threads own a row, four
// dimensions each.  The piece that holds token 0 is seen by every row; a piece in which a row sees no key
// has denominator 0 and its partial result is not used (a wave that sees none of a piece walks its first tile
// with weights 0, and 0 * V is NaN where a value behind the row is infinite or NaN).
template <typename T, int D>
__global__ __launch_bounds__(256) void prefill_merge_kernel(const PrefillParams p) {
  constexpr int TPR = D / 4;
  const int64_t at = (int64_t)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
  if (at >= (int64_t)p.n_kv * p.n_rows) return;
  const int kvh = (int)(at / p.n_rows), row = (int)(at - (int64_t)kvh * p.n_rows);
  const int kv_end = tile_kv_end(p, row / p.bm);
  const int n_parts = 1 + (kv_end - 1) / p.chunk;
  if (n_parts <= 1) return;  // the attention kernel wrote the result
  const int c = threadIdx.x % TPR;
  const int64_t stride = (int64_t)p.n_kv * p.n_rows;
  float M = kNegBig, L = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < n_parts; s0 += 4) {  // four pieces in flight
    f32x4 v[4];
    float m[4], l[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t part = (int64_t)(s0 + u < n_parts ? s0 + u : n_parts - 1) * stride + at;
      v[u] = *reinterpret_cast<const f32x4*>(p.part_o + part * D + 4 * c);
      const f32x2 ml = *reinterpret_cast<const f32x2*>(p.part_ml + part * 2);
      m[u] = s0 + u < n_parts ? ml.x : 2.f * kNegBig;
      l[u] = s0 + u < n_parts ? ml.y : 0.f;
      if (l[u] == 0.f) v[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const float m_new = fmaxf(fmaxf(fmaxf(m[0], m[1]), fmaxf(m[2], m[3])), M);
    const float alpha = fast_exp2(M - m_new);
    M = m_new;
    L *= alpha;
    acc *= alpha;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float f = s0 + u < n_parts ? fast_exp2(m[u] - m_new) : 0.f;
      L = fmaf(l[u], f, L);
#pragma unroll
      for (int d = 0; d < 4; ++d) acc[d] = fmaf(v[u][d], f, acc[d]);
    }
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  const int tok = row / p.by_group;
  uint16_t* dst = p.o + ((int64_t)tok * p.num_qo_heads + kvh * p.q_per_kv + (row - tok * p.q_per_kv)) * D + 4 * c;
  *reinterpret_cast<u32x2*>(dst) = u32x2{pack2<T>(acc[0] * inv, acc[1] * inv), pack2<T>(acc[2] * inv, acc[3] * inv)};
}

// Rows per workgroup tile and pieces per tile.  A workgroup walks its keys one tile after the other, so a
// few query rows on a long cache (a further turn of a conversation) leave most of the chip idle however
// many keys there are, and so do a short prompt and a prompt of few heads.  Pieces shorten the walk for the
// price of a merge; smaller row tiles (waves without rows compute nothing) give more workgroups, each with a
// SIMD per wave, and so a shorter step.  The estimate, in steps of a full workgroup (at head_dim 128 64 keys and
// 1.2 us, at 256 32 keys and 1.3 us): the chip runs `slots` workgroups at a time (one of eight waves per CU,
// two of four); a workgroup of 256, 128 or 64 rows costs 1, 0.87 or 0.83 per key tile and 6.5 or 4.5 to start
// (page table, queries, first tiles, cold code, diagonal), all measured at head_dim 128; causal tiles start
// longest first, which leaves a tail of about a quarter of the longest; pieces cost the merge launch (two) and
// their fp32 round trip through memory.
// Measured with pages of 16, us for tiles of 256 / 128 / 64 rows, whole: prompts of 32 heads over 8 KV heads of
// 128, 150 tokens 11.9 / 9.8 / 9.3, 300 14.8 / 12.7 / 11.4, 640 22.7 / 18.5 / 17.4, 1000 30 / 25 / 28, 2000
// 54 / 50 / 83, 2900 81 / 96 / 157; of 64, 300 10.6 / 9.5 / 9.0, 1000 21 / 18 / 21, 2000 38 / 35 / 60, 2900
// 54 / 68 / 112.  Pieces against whole tiles of 256: 500 rows of 32 heads of 128 on 32768 keys 272 against 670.
// Against the best of the tile sizes and eight piece counts, the choice took 1.03 times as long at 64 and at 128
// dimensions (51 and 34 shapes of 16 to 6000 rows, no keys to 32768 before them) and 1.01 at 256 (68 shapes),
// at worst 1.19, 1.12 and 1.12.
static double prefill_cost(const PrefillParams& p, double tile, int64_t tiles, int64_t jobs, int64_t c) {
  const int64_t slots = (int64_t)td_num_cus() * (p.staged ? 2 : 1);
  const double start = p.bm == 256 ? 6.5 : 4.5;
  const double mean = tile * (double)tiles / jobs + start, longest = tile * c + start;
  const double share = mean * jobs / slots + 0.25 * longest, rounds = (double)((jobs + slots - 1) / slots) * mean;
  const double cost = share < rounds ? share : rounds;
  return cost > longest ? cost : longest;
}

// sum of (a i + b) / m over 0 <= i < n, in as many steps as Euclid's algorithm takes for a and m: whole
// multiples of m come out of a and b, and what is left counts the lattice points under a line of slope below
// one, which is the same sum with the axes exchanged (Graham, Knuth, Patashnik, Concrete Mathematics, 3.5)
static int64_t floor_sum(int64_t n, int64_t m, int64_t a, int64_t b) {
  int64_t sum = 0;
  while (true) {
    sum += n * (n - 1) / 2 * (a / m) + n * (b / m);
    a %= m;
    b %= m;
    const int64_t top = a * n + b;
    if (top < m) return sum;
    n = top / m;
    b = top % m;
    const int64_t slope = a;
    a = m;
    m = slope;
  }
}

// sum of ceil(key tiles / c) over a KV head's row tiles: its key tiles (c = 1), its pieces of c key tiles
static int64_t key_pieces(const PrefillParams& p, int kv_len, int bn, int64_t c) {
  if (!p.causal) return p.n_tiles * ((((int64_t)kv_len + bn - 1) / bn + c - 1) / c);
  // a tile's last row r sees the keys up to kv_len - n_q + r / group, so that it has
  // (r + group (kv_len - n_q + bn)) / (group bn) key tiles; r = (i + 1) bm - 1 in all row tiles but the last
  const int64_t g = p.q_per_kv, m = g * bn * c, b = g * (kv_len - p.n_q + bn) + g * bn * (c - 1);
  return floor_sum(p.n_tiles - 1, m, p.bm, b + p.bm - 1) + (p.n_rows - 1 + b) / m;
}

template <typename T>
static int launch_prefill(const PrefillParams& p, int head_dim, bool oct, hipStream_t st) {
  const dim3 grid(p.n_tiles * p.n_kv * p.n_splits), block(p.staged ? 256 * p.key_groups : 512);
  if (head_dim == 256)
    hipLaunchKernelGGL((prefill_attn_staged_kernel<T, 256>), grid, block, 0, st, p);
  else if (head_dim == 128 && p.staged && p.key_groups == 2)
    hipLaunchKernelGGL((prefill_two_groups_kernel<T, 128>), grid, block, 0, st, p);
  else if (head_dim == 64 && p.staged && p.key_groups == 2)
    hipLaunchKernelGGL((prefill_two_groups_kernel<T, 64>), grid, block, 0, st, p);
  else if (head_dim == 128 && p.staged)
    hipLaunchKernelGGL((prefill_attn_staged_kernel<T, 128>), grid, block, 0, st, p);
  else if (head_dim == 64 && p.staged)
    hipLaunchKernelGGL((prefill_attn_staged_kernel<T, 64>), grid, block, 0, st, p);
  else if (head_dim == 128 && oct)
    hipLaunchKernelGGL((prefill_attn_kernel<T, 128, true>), grid, block, 0, st, p);
  else if (head_dim == 128)
    hipLaunchKernelGGL((prefill_attn_kernel<T, 128, false>), grid, block, 0, st, p);
  else if (head_dim == 64 && oct)
    hipLaunchKernelGGL((prefill_attn_kernel<T, 64, true>), grid, block, 0, st, p);
  else if (head_dim == 64)
    hipLaunchKernelGGL((prefill_attn_kernel<T, 64, false>), grid, block, 0, st, p);
  else
    return fail(TD_ERR_UNSUPPORTED,
                "BatchPrefillWithPagedKVCache failed to dispatch with head_dim %d (supported: 64, 128, 256)",
                head_dim);
  if (p.n_splits > 1) {
    const int rows_per_block = 256 / (head_dim / 4);
    const dim3 mgrid((unsigned)(((int64_t)p.n_kv * p.n_rows + rows_per_block - 1) / rows_per_block));
    if (head_dim == 128)
      hipLaunchKernelGGL((prefill_merge_kernel<T, 128>), mgrid, dim3(256), 0, st, p);
    else if (head_dim == 64)
      hipLaunchKernelGGL((prefill_merge_kernel<T, 64>), mgrid, dim3(256), 0, st, p);
    else
      hipLaunchKernelGGL((prefill_merge_kernel<T, 256>), mgrid, dim3(256), 0, st, p);
  }
  return TD_OK;
}

}  // namespace tidal

using namespace tidal;

static int check_prefill(const td_paged_kv* kv, int32_t n_pages, int32_t kv_len, int32_t n_q,
                         int32_t num_qo_heads) {
  TD_REQUIRE(kv->page_size >= 1 && kv->num_kv_heads >= 1 && kv->max_pages >= 1,
             "td_prefill_attn: bad pool geometry");
  TD_REQUIRE(num_qo_heads >= kv->num_kv_heads && num_qo_heads % kv->num_kv_heads == 0,
             "td_prefill_attn: num_qo_heads %d is not a multiple of num_kv_heads %d", num_qo_heads,
             kv->num_kv_heads);
  // 32-bit positions and rows, of which the kernels look up to 80 key tiles and a row tile past the end
  TD_REQUIRE(n_q >= 0 && kv_len >= n_q && kv_len <= INT32_MAX - (1 << 14), "td_prefill_attn: n_q %d, kv_len %d",
             n_q, kv_len);
  TD_REQUIRE((int64_t)n_pages * kv->page_size >= kv_len,
             "td_prefill_attn: %d pages of %d entries do not hold %d tokens", n_pages,
             kv->page_size, kv_len);
  TD_REQUIRE(kv->layout == TD_NHD || kv->layout == TD_HND, "td_prefill_attn: layout %d", kv->layout);
  TD_REQUIRE((int64_t)n_q * (num_qo_heads / kv->num_kv_heads) <= INT32_MAX - (1 << 9),
             "td_prefill_attn: %d queries of %d heads", n_q, num_qo_heads);
  return TD_OK;
}

// Pieces are not cut where their partial results would take more memory than this: 40 heads of 128, 3000
// tokens on 131072, would get 476 MB for six pieces.  Fewer pieces cost it 7.01 -> 7.20 ms (whole tiles of
// the earlier kernel 8.57), 32 heads of 256, 3188 on 98304 16.9 -> 19.1 (26.7).
constexpr int64_t kMaxScratch = (int64_t)256 << 20;

static int64_t prefill_ws_bytes(const PrefillParams& p, int head_dim) {
  return p.n_splits > 1 ? (int64_t)p.n_splits * p.n_kv * p.n_rows * (head_dim + 2) * 4 : 0;
}

// Shape of the launch for a call that passed check_prefill: of the staged kernel or of the eight-wave kernel,
// with pieces whose partial results take at most `limit` bytes.
static void plan_shape(const td_paged_kv* kv, int32_t kv_len, int32_t n_q, int32_t num_qo_heads, int32_t causal,
                       bool staged, int64_t limit, PrefillParams& p) {
  const int H = kv->num_kv_heads, D = kv->head_dim;
  p.n_kv = H;
  p.q_per_kv = num_qo_heads / H;
  p.n_rows = n_q * p.q_per_kv;
  p.n_q = n_q;
  p.causal = causal;
  p.staged = staged;
  p.key_groups = 1;
  p.lag = 8.f;
  const int bn = p.staged ? 32 : 64, max_tiles = (kv_len + bn - 1) / bn;
  const int64_t cus = td_num_cus();
  double best = 0.0;
  PrefillParams c = p;
  for (c.bm = p.staged ? 64 : 256; c.bm >= 64; c.bm /= 2) {
    c.n_tiles = (c.n_rows + c.bm - 1) / c.bm;
    const double tile = p.staged || c.bm == 256 ? 1.0 : c.bm == 128 ? 0.87 : 0.83;
    const int64_t tiles = H * key_pieces(c, kv_len, bn, 1);
    for (int s = 1; s <= 64; s = s < 8 ? s + 1 : (s < 16 ? s + 2 : s * 2)) {
      const int chunk = (max_tiles + s - 1) / s;
      if (s > 1 && (limit <= 0 || chunk < 4 || (int64_t)c.n_tiles * H >= 8 * cus)) break;
      c.chunk = chunk * bn;
      c.n_splits = 1 + (kv_len - 1) / c.chunk;
      if (prefill_ws_bytes(c, D) > limit) break;
      const double pieces = s > 1 ? 2.0 + (double)H * c.n_rows * D * 4e-6 * s / 4.0 : 0.0;
      // no cost is below that of the longest piece alone
      if (s > 1 && tile * chunk + pieces >= best) continue;
      const int64_t jobs = H * (s > 1 ? key_pieces(c, kv_len, bn, chunk) : c.n_tiles);
      const double cost = prefill_cost(c, tile, tiles, jobs, chunk) + pieces;
      if (best == 0.0 || cost < best) {
        best = cost;
        p.bm = c.bm;
        p.n_tiles = c.n_tiles;
        p.chunk = c.chunk;
        p.n_splits = c.n_splits;
      }
    }
  }
  // one head after the other on its XCD once there are enough tiles for the last head to end evenly
  p.head_major = H % 8 == 0 && (int64_t)p.n_tiles * p.n_splits * H > 4 * (int64_t)td_num_cus();
}

// The plan that scratch is asked for: the staged kernel where the eight-wave one cannot run or has nothing to
// overlap (up to one key tile).
static void plan_prefill(const td_paged_kv* kv, int32_t kv_len, int32_t n_q, int32_t num_qo_heads, int32_t causal,
                         bool may_split, PrefillParams& p) {
  const bool staged = kv->head_dim == 256 || kv_len <= 64 || ((uintptr_t)kv->data & 15) != 0;
  plan_shape(kv, kv_len, n_q, num_qo_heads, causal, staged, may_split ? kMaxScratch : 0, p);
}

// Short caches go to the staged kernel all the same, with no more scratch than was asked for: a step of either
// kernel is a serial chain of about 1 us, the eight-wave kernel's rings and phases cost more to start than two
// buffers, and two key groups halve the staged kernel's steps for 1 us of joining.  us, bf16, 32 / 8 heads of
// 128 (32 / 32 within 0.4), eight waves | staged | staged with two key groups: 16 tokens 6.5 | 4.0 | 5.6, 96
// 7.3 | 5.8 | 6.6, 128 7.3 | 6.7 | 6.4, 200 8.8 | 8.9 | 8.1, 300 10.5 | 11.5 | 9.8, 500 13.5 | 16.4 | 13.3; of
// 64, 500 10.1 | - | 10.0.  A few rows on a cache of up to 1600 tokens, in pieces, eight waves | two key groups
// with as much scratch: 16 on 484 11.4 | 10.9, 40 on 460 11.9 | 11.3, 16 on 1484 12.5 | 11.9; 16 of 40 / 40
// heads on 2000 15.1 | 15.5; twice as many row tiles gain nothing.
// The reference points lag so little that no call is less exact than on the eight-wave kernel, whose first tile
// shows a row twice as many keys.  Error against 64 bits in bf16, 1e-3, eight waves | here with a lag of 2^8 | now,
// for queries of a normalised model and of four times the size: 96 tokens 1.88 | 1.91 | 1.87 and 1.72 | 1.87 | 1.70,
// 300 1.98 | 1.96 | 1.94 and 1.81 | 1.92 | 1.70, 16 on 1500 2.28 | 2.26 | 2.19 and 1.78 | 1.87 | 1.67.  That costs
// 0.1 - 0.4 us; a lag of 0 in the two groups as much again, and 500 tokens would gain nothing.
static void plan_short(const td_paged_kv* kv, int32_t kv_len, int32_t n_q, int32_t num_qo_heads, int32_t causal,
                       int64_t scratch, PrefillParams& p) {
  if (p.staged || kv_len > 1600) return;
  const int64_t cus = td_num_cus(), tiles64 = (int64_t)p.n_kv * ((p.n_rows + 63) / 64);
  if (kv_len <= 96) {
    plan_shape(kv, kv_len, n_q, num_qo_heads, causal, true, 0, p);
    p.lag = 0.f;
  } else if (p.n_splits > 1 && kv_len > 256 ? tiles64 <= cus * 3 / 16 : kv_len <= 512 && tiles64 <= 2 * cus) {
    plan_shape(kv, kv_len, n_q, num_qo_heads, causal, true, kv_len > 256 ? scratch : 0, p);
    p.key_groups = 2;
    p.lag = 2.f;
  }
}

extern "C" int64_t td_prefill_workspace_bytes(const td_paged_kv* kv, int32_t kv_len, int32_t n_q,
                                              int32_t num_qo_heads, int32_t causal) {
  if (!kv || n_q <= 0 || check_prefill(kv, kv->page_size >= 1 ? kv_len / kv->page_size + 1 : 0, kv_len, n_q,
                                       num_qo_heads) != TD_OK)
    return 0;  // the call itself reports what is wrong
  PrefillParams p;
  plan_prefill(kv, kv_len, n_q, num_qo_heads, causal, true, p);
  return prefill_ws_bytes(p, kv->head_dim);
}

extern "C" int td_prefill_attn_split(const td_paged_kv* kv, const int32_t* page_table, int32_t n_pages,
                                     int32_t kv_len, const void* q, void* o, int32_t n_q,
                                     int32_t num_qo_heads, float sm_scale, int32_t causal,
                                     void* workspace, int64_t workspace_bytes, void* stream) {
  TD_REQUIRE(kv && kv->data && page_table && q && o, "td_prefill_attn: NULL argument");
  const int crc = check_prefill(kv, n_pages, kv_len, n_q, num_qo_heads);
  if (crc != TD_OK) return crc;
  if (n_q == 0) return TD_OK;
  const int P = kv->page_size, H = kv->num_kv_heads, D = kv->head_dim;
  PrefillParams p;
  plan_prefill(kv, kv_len, n_q, num_qo_heads, causal, true, p);
  if (workspace == nullptr || workspace_bytes < prefill_ws_bytes(p, D))
    plan_prefill(kv, kv_len, n_q, num_qo_heads, causal, false, p);
  TD_REQUIRE(p.n_splits == 1 || ((uintptr_t)workspace & 15) == 0,
             "td_prefill_attn: the workspace must be 16-byte aligned");
  plan_short(kv, kv_len, n_q, num_qo_heads, causal, prefill_ws_bytes(p, D), p);
  p.part_o = reinterpret_cast<float*>(workspace);
  p.part_ml = p.part_o ? p.part_o + (int64_t)p.n_splits * p.n_kv * p.n_rows * D : nullptr;
  p.kv = reinterpret_cast<const uint16_t*>(kv->data);
  p.page_stride = (int64_t)2 * P * H * D;
  p.v_offset = (int64_t)P * H * D;
  p.entry_stride = kv->layout == TD_NHD ? H * D : D;
  p.head_stride = kv->layout == TD_NHD ? D : P * D;
  p.page_size = P;
  p.entry_stride_b = (uint32_t)(p.entry_stride * 2);
  const bool oct = P % 8 == 0;
  p.by_page = divisor(P);
  p.by_group = divisor(p.q_per_kv);
  p.by_kv = divisor(H);
  p.by_tiles = divisor(p.n_tiles);
  p.by_head = divisor(p.n_tiles * p.n_splits);
  p.max_page = (uint32_t)(kv->max_pages - 1);
  p.page_table = page_table;
  p.n_pages = n_pages;
  p.kv_len = kv_len;
  p.q = reinterpret_cast<const uint16_t*>(q);
  p.o = reinterpret_cast<uint16_t*>(o);
  p.num_qo_heads = num_qo_heads;
  p.scale_log2 = sm_scale * 1.4426950408889634f;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  int rc;
  if (kv->dtype == TD_F16)
    rc = launch_prefill<F16>(p, D, oct, st);
  else if (kv->dtype == TD_BF16)
    rc = launch_prefill<BF16>(p, D, oct, st);
  else
    return fail(TD_ERR_UNSUPPORTED, "BatchPrefillWithPagedKVCache failed to dispatch with dtype %d",
                kv->dtype);
  if (rc != TD_OK) return rc;
  TD_HIP_CHECK(hipGetLastError());
  return TD_OK;
}

extern "C" int td_prefill_attn(const td_paged_kv* kv, const int32_t* page_table, int32_t n_pages,
                               int32_t kv_len, const void* q, void* o, int32_t n_q,
                               int32_t num_qo_heads, float sm_scale, int32_t causal, void* stream) {
  return td_prefill_attn_split(kv, page_table, n_pages, kv_len, q, o, n_q, num_qo_heads, sm_scale, causal,
                               nullptr, 0, stream);
}
