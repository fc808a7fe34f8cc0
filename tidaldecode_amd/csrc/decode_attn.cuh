// Decode attention over a paged KV pool for gfx950 (MI355X): one new query token per sequence
// attends to a listed subset of the cache (sparse layers), or to the whole cache while emitting
// per-token logits (token-selection layers).
//
// Mapping.  A K or V row of one head is head_dim two-byte elements; LPR = head_dim/8 adjacent
// lanes hold it, 16 bytes (one global_load_dwordx4) per lane, so a 64-wide wavefront carries
// HPW = 64/LPR "head rows" at once and never reduces across more than one DPP row for
// head_dim 128.  A workgroup owns one group of HPW head rows and one chunk of the token list;
// its waves take interleaved tiles of U tokens, each wave keeping a private online-softmax
// state in base 2.  Wave states are merged through LDS, workgroup results through a fp32
// partial buffer that the last-arriving workgroup of a head group reduces (ticket counter), or
// that a second small kernel reduces when the plan asks for it.
//
// With grouped-query attention and an index list shared by the query heads of a KV head
// (QPG > 1) each lane group loads the KV row once and scores it against QPG query heads.
// QPG is 2, 4 or 8; other group sizes are padded up (3 -> 4, 5..7 -> 8) or cut into head rows of
// 8 (groups above 8), the padding heads scoring with q = 0 and never being written.
//
// Semantics follow kernels/include/decode/decode_attn.cuh:432-658 of the reference
// (BatchDecodeWithPagedKVCacheKernel) including the forced last page
// (decode_page.cuh:320-346) and the logits output (decode_attn.cuh:107-109).

#pragma once

#include <type_traits>

#include "common.cuh"

namespace tidal {

struct DecodeParams {
  const void* q;
  void* o;
  const void* kv;
  int64_t page_stride;   // elements from page p to page p+1  (2 * P * H_kv * D)
  int64_t v_offset;      // elements from a K row to its V row (P * H_kv * D)
  int32_t entry_stride;  // elements between consecutive tokens of a page
  int32_t head_stride;   // elements between consecutive KV heads of a token
  int32_t page_size;
  int32_t page_shift;  // log2(page_size) or -1
  uint32_t max_slot;   // max_pages * page_size - 1
  int32_t lean;        // 1: power-of-two pages and a pool below 4 GiB (32-bit byte offsets)
  uint32_t page_stride_b, entry_stride_b;  // byte strides for the lean path
  uint32_t max_page;   // max_pages - 1
  int32_t page_mode;   // 1: list entries are pages, 0: token slots
  int32_t num_qo_heads;
  int32_t n_hrows;   // head rows: num_qo_heads (QPG == 1) or num_kv_heads * subs (QPG > 1)
  int32_t q_per_kv;  // query heads per KV head
  int32_t vheads;    // head slots of the split workspace: n_hrows * QPG (QPG may be padded: a group
                     // of 3 runs as 4, 5-7 as 8; the padding heads have q = 0 and are never stored)
  int32_t subs;      // head rows per KV head on the shared-row kernels: groups above 8 are cut
                     // into rows of 8 query heads (the last one padded)
  int32_t num_kv_heads;
  // (What a launch needs first lies together from here to `scale_log2`, with no word between that it does not: scalar
  // loads come in blocks of up to eight words, and a register that a block fills for nothing is given out again,
  // behind a wait for the block.  With two such words the short lists without a new token waited twice, 0.2 us.)
  // index list
  const int32_t* idx;
  int32_t idx_row_stride;  // 0 for a shared row
  int32_t idx_cols;        // elements a row holds (the caller's row stride; 0: unknown): reads stop there
  int32_t idx_per_kv;      // 1: rows are per KV head while QPG == 1
  int32_t n_list_host;
  const int32_t* indptr;
  const int32_t* count_arr;  // per-sequence entry counts of a padded table (else indptr differences)
  const int32_t* last_len_arr;
  const int32_t* last_idx_arr;
  int32_t last_len;
  int32_t last_idx;
  // split
  int32_t chunk_tokens;
  uint32_t chunk_magic;  // 2^32 / chunk_tokens, rounded up: exact for the short-list kernel's up to 2^16 tokens
  uint32_t kv_magic;    // 2^24 / q_per_kv, rounded up
  int32_t max_splits;
  int32_t fused_merge;
  float scale_log2;  // sm_scale * log2(e)
  // outputs
  void* scores;
  int32_t scores_f32;
  int64_t score_stride;
  float* lse;
  float* ws_o;      // [batch * H_q * max_splits, D]
  float* ws_ml;     // [batch * H_q * max_splits, 2]
  int32_t* ws_cnt;  // [batch * head rows] ticket counters, ticket_stride words apart
  int32_t ticket_stride;
  int32_t batch, slots;  // balanced launches: sequences, and workgroups per head row
  int32_t list_shift;    // short-list kernel: log2 of the tokens a list entry stands for
  // the token being decoded (FRESH kernels): un-rotated k, v, its rotary cos/sin and its slot
  const void* fresh_k;
  const void* fresh_v;
  const float* fresh_cos;
  const float* fresh_sin;
  const int32_t* fresh_slot;
};

template <bool LEAN>
__device__ __forceinline__ void divmod_page(const DecodeParams& p, uint32_t x, uint32_t& page,
                                            uint32_t& entry) {
  if (LEAN || p.page_shift >= 0) {
    page = x >> p.page_shift;
    entry = x & ((1u << p.page_shift) - 1u);
  } else {
    page = x / (uint32_t)p.page_size;
    entry = x - page * (uint32_t)p.page_size;
  }
}

// Per-sequence view of the token list.
struct SeqList {
  const int32_t* row;  // this lane group's index row, already offset to the sequence
  int32_t n_list;      // listed entries (pages or slots)
  int32_t n_items;     // tokens attended
  int32_t last_len;
  int32_t last_idx;
};

// 8-byte device-coherent accesses for the split partials: they are written by one workgroup and
// read by another that may sit on a different XCD (own L2), so they go to memory (sc1) instead
// of relying on an L2-wide write-back fence.
__device__ __forceinline__ void store_coherent(float* dst, float a, float b) {
  const uint64_t v = (uint64_t)__builtin_bit_cast(uint32_t, a) |
                     ((uint64_t)__builtin_bit_cast(uint32_t, b) << 32);
  __hip_atomic_store(reinterpret_cast<uint64_t*>(dst), v, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void load_coherent(const float* src, float& a, float& b) {
  const uint64_t v = __hip_atomic_load(reinterpret_cast<const uint64_t*>(src), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  a = __builtin_bit_cast(float, (uint32_t)v);
  b = __builtin_bit_cast(float, (uint32_t)(v >> 32));
}

// Reduce the n_splits partial results of the QPG query heads of one head row and write o (and
// lse).  Runs in one workgroup of NT threads: NT / (QPG * D / 2) "slots" of threads each own a
// float2 column and a subset of the splits; slots are combined through LDS.
// part_first: the partial of head slot 0 and split 0; part_heads: partials from one head slot to the next.
template <typename T, int D, int QPG, int NT>
__device__ __forceinline__ void merge_splits(const DecodeParams& p, int b, int64_t part_first, int part_heads,
                                             int rq0, int gsz, int n_splits) {
  constexpr int COLS = QPG * D / 2;
  constexpr int SLOTS = NT / COLS;
  constexpr int PRE = SLOTS >= 8 ? 4 : (SLOTS >= 4 ? 8 : 16);  // partial loads in flight per thread
  static_assert(SLOTS >= 1, "workgroup too small for the merge");
  __shared__ float mg_m[QPG][64], mg_l[QPG][64];
  __shared__ float mg_part[SLOTS][COLS][2];
  const int tid = threadIdx.x;
  const int c = tid % COLS, slot = tid / COLS;
  const int j = c / (D / 2), d2 = c % (D / 2);
  const int64_t part0 = part_first + (int64_t)j * part_heads;

  // (m, l) of every split and head: one pair per thread; the load is unconditional (clamped
  // thread index) so that it is in flight together with the partial loads below
  float ml_m, ml_l;
  const bool has_ml = tid < n_splits * QPG;
  {
    const int tc = has_ml ? tid : 0;
    const int jj = tc / n_splits, ss = tc % n_splits;
    load_coherent(p.ws_ml + (part_first + (int64_t)jj * part_heads + ss) * 2, ml_m, ml_l);
  }
  // Loads are unconditional (index clamped, contribution zeroed) so that a batch of PRE of them
  // is in flight per thread; a branch around a load makes the compiler wait for each one.
  float pa[PRE], pb[PRE];
  auto issue = [&](int base) {
#pragma unroll
    for (int u = 0; u < PRE; ++u) {
      int sidx = base + u * SLOTS;
      sidx = sidx < n_splits ? sidx : n_splits - 1;
      load_coherent(p.ws_o + (part0 + sidx) * D + d2 * 2, pa[u], pb[u]);
    }
  };
  if (slot < SLOTS) issue(slot);
  if (has_ml) {
    mg_m[tid / n_splits][tid % n_splits] = ml_m;
    mg_l[tid / n_splits][tid % n_splits] = ml_l;
  }
  __syncthreads();
  float M = kNegBig;
  for (int sidx = 0; sidx < n_splits; ++sidx) M = fmaxf(M, mg_m[j][sidx]);
  float ra = 0.f, rb = 0.f;
  if (slot < SLOTS) {
    for (int base = slot; base < n_splits; base += PRE * SLOTS) {
      if (base != slot) issue(base);
#pragma unroll
      for (int u = 0; u < PRE; ++u) {
        const int sidx = base + u * SLOTS;
        const int sc = sidx < n_splits ? sidx : n_splits - 1;
        const bool live = sidx < n_splits;
        const float f = fast_exp2(mg_m[j][sc] - M);
        ra = fmaf(live ? pa[u] : 0.f, f, ra);
        rb = fmaf(live ? pb[u] : 0.f, f, rb);
      }
    }
    mg_part[slot][c][0] = ra;
    mg_part[slot][c][1] = rb;
  }
  __syncthreads();
  if (tid < COLS && j < gsz) {
    float L = 0.f;
    for (int sidx = 0; sidx < n_splits; ++sidx)
      L = fmaf(mg_l[j][sidx], fast_exp2(mg_m[j][sidx] - M), L);
    float oa = 0.f, ob = 0.f;
#pragma unroll
    for (int sl = 0; sl < SLOTS; ++sl) {
      oa += mg_part[sl][c][0];
      ob += mg_part[sl][c][1];
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    const int qh = rq0 + j;
    reinterpret_cast<uint32_t*>(p.o)[((int64_t)b * p.num_qo_heads + qh) * (D / 2) + d2] =
        pack2<T>(oa * inv, ob * inv);
    if (p.lse && d2 == 0)
      p.lse[(int64_t)b * p.num_qo_heads + qh] = L > 0.f ? (M + fast_log2(L)) * kLn2 : -INFINITY;
  }
}

// Which query heads a head row of a shared-row kernel (QPG > 1) stands for: its KV head, its first
// query head and how many of its QPG head slots are real.
template <int QPG>
__device__ __forceinline__ void head_row_geom(const DecodeParams& p, int hrow, int& kv_head, int& rq0,
                                              int& gsz) {
  if constexpr (QPG > 1) {
    kv_head = hrow / p.subs;
    const int sub = hrow - kv_head * p.subs;
    rq0 = kv_head * p.q_per_kv + sub * QPG;
    const int left = p.q_per_kv - sub * QPG;
    gsz = left < QPG ? left : QPG;
  } else {
    kv_head = hrow / p.q_per_kv;
    rq0 = hrow;
    gsz = 1;
  }
}

// Columns of a sequence's list segment that a kernel may read: the host's bound, cut to the segment
// [list_beg, list_end) when the call has an indptr and to what is left of the row (row_cols columns;
// 0: a row of unknown length).  Device-resident counts are clamped to it.
__device__ __forceinline__ int list_capacity(int n_list_host, bool has_indptr, int list_beg,
                                             int list_end, int row_cols) {
  int cap = n_list_host;
  if (has_indptr) cap = list_end - list_beg < cap ? list_end - list_beg : cap;
  if (row_cols > 0) cap = row_cols - list_beg < cap ? row_cols - list_beg : cap;
  return cap < 0 ? 0 : cap;
}

__device__ __forceinline__ int seq_items(const DecodeParams& p, int b, SeqList& s, int& list_beg) {
  list_beg = 0;
  int list_end = 0;
  if (p.indptr) {
    list_beg = p.indptr[b];
    list_end = p.indptr[b + 1];
    s.n_list = p.count_arr ? p.count_arr[b] : list_end - list_beg;
  } else {
    s.n_list = p.n_list_host;
  }
  const int cap = list_capacity(p.n_list_host, p.indptr != nullptr, list_beg, list_end, p.idx_cols);
  s.n_list = s.n_list < 0 ? 0 : (s.n_list > cap ? cap : s.n_list);
  s.last_len = p.last_len_arr ? p.last_len_arr[b] : p.last_len;
  s.last_idx = p.last_idx_arr ? p.last_idx_arr[b] : p.last_idx;
  // device-resident lengths are not trusted: a fill beyond the page, or more splits than the
  // grid holds, would leave tickets that no workgroup ever takes
  s.last_len = s.last_len < 0 ? 0 : (s.last_len > p.page_size ? p.page_size : s.last_len);
  s.n_items = (p.page_mode ? s.n_list * p.page_size : s.n_list) + s.last_len;
  int n_splits = (s.n_items + p.chunk_tokens - 1) / p.chunk_tokens;
  n_splits = n_splits > p.max_splits ? p.max_splits : n_splits;
  return n_splits < 1 ? 1 : n_splits;
}

// The matrix cores take the weights of shared rows in the KV type, as a sum of parts.
// kRounded: a rounded value and the rounded remainder, 16 bits of a weight in bf16 and 22 in fp16.
// kWhole: three truncated parts, which hold all 24 bits, so that nothing is lost against products in fp32.  Every part
// of a weight above 0 is above 0 (fp16: of 2^-39 and more): an infinite value times a remainder of 0, or of the other
// sign, would give NaN.  fp16 weights are taken times kWeightScale, or those below 2^-25 would vanish beside a
// denominator that counts them.  Head_dim 64 takes kWhole, and short lists in fp16 do: their values met fp32 weights or
// a single part before they came to the matrix cores in two.  The third part costs a launch 2 % (its arithmetic; the four
// sums by turns instead of part after part change nothing), one of 300 tokens, which is a chain of latencies, 6: one
// layer, rounded | whole, us: 16/8 heads x 64, bf16, logits out, 300 tokens 5.50 | 5.88, 2000 7.28 | 7.50; 28/4 x 64 300
// 5.87 | 6.07, 60000 24.9 | 25.3; 32/8 x 64, fp16, 60000 37.1 | 37.5; 32/8 heads x 128, fp16, lists of 4096 8.2 | 8.4.
enum WeightParts { kRounded = 2, kWhole = 3 };
template <typename T, WeightParts PARTS>
constexpr float kWeightScale = PARTS == kWhole && std::is_same<T, F16>::value ? 32768.f : 1.f;

template <typename T, WeightParts PARTS>
__device__ __forceinline__ void split_weights(float w0, float w1, uint32_t (&part)[PARTS]) {
  float r0, r1;
  if constexpr (PARTS == kRounded) {
    part[0] = pack2<T>(w0, w1);
    unpack2<T>(part[0], r0, r1);
    part[1] = pack2<T>(w0 - r0, w1 - r1);
  } else {
    constexpr float kLeast = std::is_same<T, F16>::value ? 0x1p-24f : 0x1p-120f;  // what a part holds at least
    w0 *= kWeightScale<T, PARTS>;
    w1 *= kWeightScale<T, PARTS>;
    const float least0 = fminf(w0, kLeast), least1 = fminf(w1, kLeast);
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      part[x] = pack2_toward_zero<T>(w0, w1);
      unpack2<T>(part[x], r0, r1);
      w0 = fmaxf(w0 - r0, least0);
      w1 = fmaxf(w1 - r1, least1);
    }
  }
}

// o += P V for four rows of values per lane: pr are the weights of one head (column c16; head_dim 64: of the tokens of
// both halves of the 16-lane row), acc[e] dimension e of the lane (head_dim 128: li * 8 + e; 64: li * 8 + 4 (c16 / 8)
// + e) of the heads 4 g4 + 0 .. 3, times kWeightScale.
template <typename T, int D, WeightParts PARTS, int NH = 128 / D, int NACC = D / 16>
__device__ __forceinline__ void weigh_rows(const float (&pr)[NH][4], const u32x4 (&v)[4], f32x4 (&acc)[NACC]) {
  constexpr uint32_t kLow = 0x05040100u, kHigh = 0x07060302u;  // v_perm: the low or the high halves of two dwords
  uint32_t part[NH][2][PARTS];
#pragma unroll
  for (int h = 0; h < NH; ++h)
#pragma unroll
    for (int w = 0; w < 2; ++w) split_weights<T, PARTS>(pr[h][2 * w], pr[h][2 * w + 1], part[h][w]);
  if constexpr (D == 128) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint32_t lo0 = __builtin_amdgcn_perm(v[1][w], v[0][w], kLow), lo1 = __builtin_amdgcn_perm(v[3][w], v[2][w], kLow);
      const uint32_t hi0 = __builtin_amdgcn_perm(v[1][w], v[0][w], kHigh), hi1 = __builtin_amdgcn_perm(v[3][w], v[2][w], kHigh);
#pragma unroll
      for (int x = 0; x < PARTS; ++x) {
        acc[2 * w] = mfma_16x16x16<T>(part[0][0][x], part[0][1][x], lo0, lo1, acc[2 * w]);
        acc[2 * w + 1] = mfma_16x16x16<T>(part[0][0][x], part[0][1][x], hi0, hi1, acc[2 * w + 1]);
      }
    }
  } else {
    // Rows of eight lanes: the two halves of a 16-lane row hold different tokens.  They exchange half of their
    // dimensions, after which a lane has four dimensions of the eight tokens of both.
    uint32_t t[2][4][2];  // half, row, two dimensions each
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        t[0][u][w] = (uint32_t)__builtin_amdgcn_update_dpp((int)v[u][w], (int)v[u][2 + w], 0x128, 0xf, 0xc, false);
        t[1][u][w] = (uint32_t)__builtin_amdgcn_update_dpp((int)v[u][2 + w], (int)v[u][w], 0x128, 0xf, 0x3, false);
      }
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const uint32_t sel = half ? kHigh : kLow;
        const u32x4 vv = {__builtin_amdgcn_perm(t[0][1][w], t[0][0][w], sel), __builtin_amdgcn_perm(t[0][3][w], t[0][2][w], sel),
                          __builtin_amdgcn_perm(t[1][1][w], t[1][0][w], sel), __builtin_amdgcn_perm(t[1][3][w], t[1][2][w], sel)};
#pragma unroll
        for (int x = 0; x < PARTS; ++x)
          acc[2 * w + half] = mfma_16x16x32<T>(u32x4{part[0][0][x], part[0][1][x], part[NH - 1][0][x], part[NH - 1][1][x]}, vv,
                                               acc[2 * w + half]);
      }
  }
}

// One of the n splits of a sequence; PLANNED: n is what the plan's chunk size gives, and the partials are
// where the plan has them, else part_first is the first partial of the sequence in those of a head slot.
struct Share {
  int split, n_splits, part_first;
};

template <typename T, int D, int QPG, int U, int NW, bool PAGE_MODE, bool EMIT, bool LEAN, bool FRESH, bool PLANNED>
__device__ __forceinline__ void attend_share(const DecodeParams& p, const int hrow, const int b, const Share& share) {
  static_assert(!FRESH || LEAN, "the fused decode step exists for the lean addressing only");
  constexpr int LPR = D / 8;     // lanes per K/V row
  constexpr int TPI = 64 / LPR;  // tokens one wave instruction covers
  constexpr int TILE = U * TPI;  // tokens per wave tile
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  // scalar on purpose: control flow that depends on the wave index must be a real branch, because
  // matrix instructions do not honour the EXEC mask of a masked-off region
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane / LPR;   // lane group = token slot inside the instruction
  const int li = lane % LPR;  // 16-byte column of the row
  const int split = share.split;
  const int qh0 = hrow * QPG;  // first head slot of this head row in the split workspace
  int kv_head, rq0, gsz;       // KV head, first query head, query heads that really exist in the row
  head_row_geom<QPG>(p, hrow, kv_head, rq0, gsz);

  SeqList s;
  int list_beg;
  const int planned = seq_items(p, b, s, list_beg);
  const int n_splits = PLANNED ? planned : share.n_splits;
  if (split >= n_splits) return;  // uniform for the whole workgroup
  const int64_t part_first = PLANNED ? ((int64_t)b * p.vheads + qh0) * p.max_splits
                                     : (int64_t)qh0 * p.slots + share.part_first;
  const int part_heads = PLANNED ? p.max_splits : p.slots;
  const int idx_row = (QPG > 1 || p.idx_per_kv) ? kv_head : hrow;
  s.row = p.idx + (int64_t)idx_row * p.idx_row_stride + list_beg;

  // The splits of a head row interleave: split s takes the workgroup-wide tiles s, s + n_splits,
  // s + 2 n_splits, ... so that all workgroups sweep the sequence together as one moving window
  // (DRAM row locality of a streaming read) instead of as n_splits distant streams.
  const int c1 = s.n_items;

  // MMA: shared rows (QPG > 1) of head_dim 64 and 128, weighted values on the matrix cores.
  constexpr bool MMA = QPG > 1 && LPR <= 16;
  static_assert(!MMA || U == 4, "shared-row tiles: four rows per lane group");
  // The scores: rows of 16 lanes with 2 or 4 heads stay on dot products (see `reduce`).
  constexpr bool MMA_SCORES = MMA && (QPG == 8 || LPR == 8);
  constexpr int NS = MMA ? D / 32 : 1;     // matrix instructions of a score
  constexpr int NB = MMA ? TILE / 16 : 1;  // blocks of 16 tokens in a tile
  const int g4 = lane >> 4, c16 = lane & 15;

  // query, packed in the KV dtype.  MMA_SCORES: column c16 of the operand is head c16 % QPG, elements
  // [32 s + 8 g4, +8); otherwise QPG heads x 8 elements per lane.
  uint32_t qp[MMA_SCORES ? 1 : QPG][4];
  u32x4 qm[NS];
  {
    const u32x4* qptr = reinterpret_cast<const u32x4*>(p.q) + ((int64_t)b * p.num_qo_heads + rq0) * LPR;
    if constexpr (MMA_SCORES) {
      const int j = c16 % QPG;
#pragma unroll
      for (int x = 0; x < NS; ++x) {
        const u32x4 v = qptr[(j < gsz ? j : gsz - 1) * LPR + 4 * x + g4];  // unconditional load, clamped row
        qm[x] = j < gsz ? v : u32x4{0u, 0u, 0u, 0u};                       // padding heads score with q = 0
      }
    } else {
#pragma unroll
      for (int j = 0; j < QPG; ++j) {
        const u32x4 v = qptr[(j < gsz ? j : gsz - 1) * LPR + li];
        const bool real = j < gsz;
        qp[j][0] = real ? v.x : 0u;
        qp[j][1] = real ? v.y : 0u;
        qp[j][2] = real ? v.z : 0u;
        qp[j][3] = real ? v.w : 0u;
      }
    }
  }

  // Decode-step fusion: q arrives un-rotated and is rotated in registers; the new token's k is
  // rotated here as well, written to its cache slot by one workgroup per KV head, and used from
  // registers wherever the list refers to that slot (the cache write races with nobody: no lane
  // consumes what it loaded from that slot).
  uint32_t knew[4] = {0, 0, 0, 0}, vnew[4] = {0, 0, 0, 0};
  uint32_t new_page = 0xffffffffu, new_entry = 0;
  float rcs[8], rsn[8];  // cos and signed sin of this lane's 8 dimensions
  if constexpr (FRESH) {
    constexpr int HALF = LPR / 2;  // lanes holding the first half of the head dimension
    const uint32_t ns = (uint32_t)p.fresh_slot[b];
    new_page = ns >> p.page_shift;
    new_entry = ns & ((1u << p.page_shift) - 1u);
    const f32x4* cp = reinterpret_cast<const f32x4*>(p.fresh_cos + (int64_t)b * (D / 2) + (li % HALF) * 8);
    const f32x4* sp = reinterpret_cast<const f32x4*>(p.fresh_sin + (int64_t)b * (D / 2) + (li % HALF) * 8);
    const f32x4 c0 = cp[0], c1v = cp[1], s0 = sp[0], s1 = sp[1];
    rcs[0] = c0.x; rcs[1] = c0.y; rcs[2] = c0.z; rcs[3] = c0.w;
    rcs[4] = c1v.x; rcs[5] = c1v.y; rcs[6] = c1v.z; rcs[7] = c1v.w;
    const float sgn = li < HALF ? -1.f : 1.f;  // y_lo = x_lo c - x_hi s,  y_hi = x_hi c + x_lo s
    rsn[0] = sgn * s0.x; rsn[1] = sgn * s0.y; rsn[2] = sgn * s0.z; rsn[3] = sgn * s0.w;
    rsn[4] = sgn * s1.x; rsn[5] = sgn * s1.y; rsn[6] = sgn * s1.z; rsn[7] = sgn * s1.w;
    const int64_t fresh_off =
        ((int64_t)b * (p.num_qo_heads / p.q_per_kv) + kv_head) * LPR + li;
    const u32x4 kn = reinterpret_cast<const u32x4*>(p.fresh_k)[fresh_off];
    const u32x4 vn = reinterpret_cast<const u32x4*>(p.fresh_v)[fresh_off];
    knew[0] = kn.x; knew[1] = kn.y; knew[2] = kn.z; knew[3] = kn.w;
    vnew[0] = vn.x; vnew[1] = vn.y; vnew[2] = vn.z; vnew[3] = vn.w;
  }
  // Rotation of q and of the new key, and the cache write; called once the first K/V tile of
  // the wave is in flight so that these few loads and shuffles hide behind it.
  // rotate-half RoPE of 8 elements per lane; the partner dimension (+- D/2) sits LPR/2 lanes away
  auto rotate = [&](uint32_t(&w)[4]) {
    float x[8], y[8];
#pragma unroll
    for (int c = 0; c < 4; ++c) unpack2<T>(w[c], x[2 * c], x[2 * c + 1]);
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      float partner;
      if constexpr (LPR == 16)
        partner = dpp_move<0x128>(x[d]);  // row_ror:8 == lane ^ 8 inside the 16-lane row
      else if constexpr (LPR == 8)
        partner = lane_xor16<4>(x[d]);
      else
        partner = __shfl_xor(x[d], LPR / 2, 64);
      y[d] = x[d] * rcs[d] + partner * rsn[d];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) w[c] = pack2<T>(y[2 * c], y[2 * c + 1]);
  };
  // (Rotating the new key lazily, only where the list meets the new slot, keeps cos/sin alive
  // through the main loop and costs more registers than it saves instructions.)
  auto finish_fresh = [&]() {
    if constexpr (FRESH) {
      if constexpr (MMA_SCORES) {
        // element d of the operand piece s has its partner, d +- D/2, at the same place of piece s +- NS/2
        const float* cs = p.fresh_cos + (int64_t)b * (D / 2) + 8 * g4;
        const float* sn = p.fresh_sin + (int64_t)b * (D / 2) + 8 * g4;
#pragma unroll
        for (int x = 0; x < NS / 2; ++x)
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const f32x2 c2 = *reinterpret_cast<const f32x2*>(cs + 32 * x + 2 * w);
            const f32x2 s2 = *reinterpret_cast<const f32x2*>(sn + 32 * x + 2 * w);
            float a0, a1, b0, b1;
            unpack2<T>(qm[x][w], a0, a1);
            unpack2<T>(qm[x + NS / 2][w], b0, b1);
            qm[x][w] = pack2<T>(a0 * c2.x + b0 * -s2.x, a1 * c2.y + b1 * -s2.y);
            qm[x + NS / 2][w] = pack2<T>(b0 * c2.x + a0 * s2.x, b1 * c2.y + a1 * s2.y);
          }
      } else {
#pragma unroll
        for (int j = 0; j < QPG; ++j) rotate(qp[j]);
      }
      rotate(knew);
      const bool writer_row = rq0 == kv_head * p.q_per_kv;  // the KV head's first head row
      if (split == 0 && wave == 0 && g == 0 && writer_row) {
        const uint32_t page_c = new_page > p.max_page ? p.max_page : new_page;
        char* dst = reinterpret_cast<char*>(const_cast<void*>(p.kv)) + page_c * p.page_stride_b +
                    new_entry * p.entry_stride_b + (uint32_t)(kv_head * p.head_stride + li * 8) * 2u;
        u32x4 ko = {knew[0], knew[1], knew[2], knew[3]};
        u32x4 vo = {vnew[0], vnew[1], vnew[2], vnew[3]};
        *reinterpret_cast<u32x4*>(dst) = ko;
        *reinterpret_cast<u32x4*>(dst + p.v_offset * 2) = vo;
      }
    }
  };

  // Shared-row state: a lane works on ONE query head, c16 % QPG; the running maximum mh of a head is kept
  // equal in all lanes of the wave, lh is the lane's share of the denominator, and accm[dd][i] is
  // o[head (4 g4 + i) % QPG] of dimension dd of the lane (see weigh_rows).
  constexpr int NACC = MMA ? D / 16 : 1;
  constexpr WeightParts kParts = D == 64 ? kWhole : kRounded;
  float mh = kNegBig, lh = 0.f;
  f32x4 accm[NACC];
#pragma unroll
  for (int d = 0; d < NACC; ++d) accm[d] = f32x4{0.f, 0.f, 0.f, 0.f};

  constexpr int NV = MMA ? 1 : QPG;  // heads on the vector ALU
  float m[NV], l[NV], acc[NV][8];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    m[j] = kNegBig;
    l[j] = 0.f;
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[j][d] = 0.f;
  }

  const int kv_head_off = kv_head * p.head_stride + li * 8;
  const uint16_t* kv16 = reinterpret_cast<const uint16_t*>(p.kv);

  // ---- software pipeline over this wave's tiles ------------------------------------------------
  // program order per iteration: list entries of tile t+2, K/V rows of tile t+1, arithmetic of
  // tile t.  Waiting for older list entries never waits for younger K/V loads, so two tiles of
  // K/V stay in flight per wave.
  u32x4 kA[U], vA[U], kB[U], vB[U];
  int32_t rawA[U], rawB[U];
  uint32_t hitA = 0, hitB = 0;

  // Address generation is branch-free: an item past the end of the chunk is redirected to the
  // chunk's last item (a valid address; its contribution is masked out in the arithmetic) and
  // list reads are clamped into the list.  With power-of-two pages and a pool below 4 GiB
  // (LEAN) the offsets are 32-bit byte offsets from a uniform base and pages are shifts.
  const char* kbase = reinterpret_cast<const char*>(p.kv);
  const char* vbase = kbase + p.v_offset * 2;
  const uint32_t head_byte_off = (uint32_t)kv_head_off * 2u;
  const bool has_list = s.n_list > 0;

  auto fetch_list = [&](int base, int32_t(&raw)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int i = base + u * TPI + g;
      i = i < c1 ? i : c1 - 1;
      uint32_t pos = (uint32_t)i;
      if constexpr (PAGE_MODE) {
        uint32_t e;
        divmod_page<LEAN>(p, (uint32_t)i, pos, e);
      }
      pos = (int32_t)pos < s.n_list ? pos : (uint32_t)(s.n_list - 1);
      raw[u] = has_list ? *reinterpret_cast<const int32_t*>(
                              reinterpret_cast<const char*>(s.row) + (pos << 2))
                        : 0;
    }
  };
  auto issue = [&](int base, const int32_t(&raw)[U], u32x4(&kb)[U], u32x4(&vb)[U], uint32_t& hit) {
    uint32_t page[U], entry[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int i = base + u * TPI + g;
      i = i < c1 ? i : c1 - 1;
      if constexpr (PAGE_MODE) {
        uint32_t pg;
        divmod_page<LEAN>(p, (uint32_t)i, pg, entry[u]);
        page[u] = (int32_t)pg < s.n_list ? (uint32_t)raw[u] : (uint32_t)s.last_idx;
      } else {
        uint32_t slot = i < s.n_list ? (uint32_t)raw[u]
                                     : (uint32_t)s.last_idx * (uint32_t)p.page_size +
                                           (uint32_t)(i - s.n_list);
        slot = slot > p.max_slot ? p.max_slot : slot;
        divmod_page<LEAN>(p, slot, page[u], entry[u]);
      }
      page[u] = page[u] > p.max_page ? p.max_page : page[u];
    }
    hit = 0;
    if constexpr (FRESH) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        hit |= (page[u] == new_page && entry[u] == new_entry) ? (1u << u) : 0u;
    }
    if constexpr (LEAN) {
      uint32_t offs[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        offs[u] = page[u] * p.page_stride_b + entry[u] * p.entry_stride_b + head_byte_off;
        kb[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kbase + offs[u]));
      }
      // V after all K: the q.k arithmetic of a tile starts while its V rows are still in flight.
      // K/V rows are read once per launch: non-temporal loads keep them from displacing the lists,
      // q and the split partials in L2 / Infinity Cache (measured: +15 % on the streaming layer).
#pragma unroll
      for (int u = 0; u < U; ++u)
        vb[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vbase + offs[u]));
    } else {
      int64_t offs[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        offs[u] = (int64_t)page[u] * p.page_stride + (int64_t)entry[u] * p.entry_stride + kv_head_off;
        kb[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kv16 + offs[u]));
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        vb[u] = __builtin_nontemporal_load(
            reinterpret_cast<const u32x4*>(kv16 + offs[u] + p.v_offset));
    }
  };
  // ---- logits (EMIT) ------------------------------------------------------------------------------
  // Vector stores and loads share one in-order completion counter, so a store issued per tile
  // holds back the wait for every younger K/V or list load until its write is acknowledged.  The
  // logits are therefore collected in a per-wave LDS strip and written EMIT_TILES tiles at a
  // time: the stores enter the memory queue once per batch (once per launch for most shapes).
  // The later the better: what the writes cost is their HBM traffic in the middle of the read
  // stream (8 sequences x 32 heads x 32K tokens: 33.5 MB of logits beside 4.3 GB of K/V add 87 us to
  // 665; the same stores aimed at one 16 KB window add 5; write-through, non-temporal or
  // contiguous stores change nothing), and a workgroup that writes once, at its end, writes when
  // the others of its round do.  The shared-row kernels have the LDS for that (one workgroup per
  // compute unit): 12 KB per wave hold the 4 x 3328 logits of a 100K-token plan (32/8 heads at
  // 100K tokens: 86 -> 80.6 us with 12 KB per wave instead of 4; 8 x 32K: 214 -> 204).
  constexpr int EMIT_FLOATS = EMIT ? (NW == 16 ? 512 : (QPG > 1 ? 3072 : 1024)) : 1;  // per wave
  constexpr int EMIT_TILES = EMIT ? EMIT_FLOATS / (QPG * TILE) : 1;
  static_assert(EMIT_TILES >= 1, "logit strip too small for one tile");
  __shared__ float emit_buf[EMIT ? NW * EMIT_FLOATS : 1];
  // Wave states at the end of the launch; before that, in the shared-row kernels, the wave's key tile on its
  // way to operand layout (a wave only ever uses its own part before the barrier).
  constexpr int STATE_F = QPG * D > NB * 16 * D / 2 || !MMA ? QPG * D : NB * 16 * D / 2;  // floats per wave
  __shared__ __attribute__((aligned(16))) float sm_state[NW][STATE_F];
  int emit_n = 0;       // tiles waiting in the strip
  int emit_first = 0;   // first token of the oldest waiting tile
  const int STEP = n_splits * NW * TILE;  // tokens between two tiles of this wave
  auto emit_flush = [&]() {
    if constexpr (EMIT) {
      // The strip was written by other lanes of this wave than the ones that now read it.  LDS
      // accesses of one wave complete in issue order, so the reads below see those writes; the
      // explicit wait and the wave barrier say so to the reader and pin the order for the
      // compiler as well (one wait per flush, that is per 16-64 tiles).
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_wave_barrier();
      // a store instruction covers 64 / TILE tiles of one head: lane -> (tile, token)
      constexpr int TPS = 64 / TILE >= 1 ? 64 / TILE : 1;  // tiles per store (TILE <= 64)
      const int lt = lane / TILE, ltok = lane % TILE;
      for (int n0 = 0; n0 < emit_n; n0 += TPS) {
        const int n = n0 + lt;
        const int i = emit_first + n * STEP + ltok;
#pragma unroll
        for (int j = 0; j < QPG; ++j) {
          if (n < emit_n && i < c1 && j < gsz) {
            const float nat = emit_buf[((wave * EMIT_TILES + n) * QPG + j) * TILE + ltok];
            const int64_t at = ((int64_t)b * p.num_qo_heads + rq0 + j) * p.score_stride + i;
            if (p.scores_f32)
              reinterpret_cast<float*>(p.scores)[at] = nat;
            else
              reinterpret_cast<uint16_t*>(p.scores)[at] = from_float<T>(nat);
          }
        }
      }
      emit_n = 0;
    }
  };
  auto emit_push = [&](int base) {  // the tile that starts at token `base` is in the strip
    if (emit_n == 0) emit_first = base;
    if (++emit_n == EMIT_TILES) emit_flush();
  };

  auto reduce = [&](u32x4(&kb)[U], u32x4(&vb)[U], int base, uint32_t hit) {
    if constexpr (FRESH) {
      if (__ballot(hit != 0)) {  // rare: some lane group of this wave meets the new token
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if ((hit >> u) & 1u) {
            kb[u].x = knew[0]; kb[u].y = knew[1]; kb[u].z = knew[2]; kb[u].w = knew[3];
            vb[u].x = vnew[0]; vb[u].y = vnew[1]; vb[u].z = vnew[2]; vb[u].w = vnew[3];
          }
        }
      }
    }
    if constexpr (MMA) {
      float xe[NB][4], sv[NB][4];
      if constexpr (MMA_SCORES) {
      // ---- S = K Q^T -------------------------------------------------------------------------------
      // A lane group loads whole rows of K, the matrix operand wants 16 rows side by side: the tile goes
      // through the wave's own LDS (LDS accesses of one wave complete in order).  Row r of block x is token
      // TPI (r % 4) + NB (r / 4) + x of the tile, so that a lane's four scores of a block are the tokens whose
      // values its group holds.  Piece c of row r lies at c ^ r (head_dim 64: c ^ (r / 2)): sixteen rows, read
      // at one piece, fall on different banks.  Dot products, which this replaces, take 4 QPG instructions per
      // row and lane and a reduction over the row; eight heads of 128 were bound by them, and so were rows of
      // eight lanes, whose values were weighted on the vector ALU as well.  bf16, logits out, three layers
      // (two of them full, lists of 1024 per KV head), us, before -> now: 28/4 heads x 128 at 60000 tokens 145 -> 115;
      // x 64 139 -> 93; 32/8 heads x 64 at 16000 76.6 -> 61.3.  Two and four heads of
      // 128 are bound by the loads and lose 1 - 3 % to the detour; a third tile of loads in flight costs them 9 %
      // and eight heads 17 % at 60000 tokens.
      auto place = [](int r, int c) { return r * (D * 2) + 16 * (c ^ (LPR == 16 ? r : (r >> 1) & 7)); };
      char* const kt = reinterpret_cast<char*>(sm_state[wave]);
      {
        const int x = LPR == 16 ? 0 : g & 1, r0 = 4 * (LPR == 16 ? g : g >> 1);
#pragma unroll
        for (int u = 0; u < U; ++u)
          *reinterpret_cast<u32x4*>(kt + 16 * x * (D * 2) + place(r0 + u, li)) = kb[u];
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int x = 0; x < NB; ++x) {
        f32x4 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int y = 0; y < NS; ++y)
          st = mfma_16x16x32<T>(
              *reinterpret_cast<const u32x4*>(kt + 16 * x * (D * 2) + place(c16, 4 * y + g4)), qm[y], st);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          xe[x][u] = st[u] * p.scale_log2;
          sv[x][u] = base + u * TPI + NB * g4 + x < c1 ? xe[x][u] : kNegBig;
        }
      }
      asm volatile("" ::: "memory");
      } else {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          float a[QPG];
#pragma unroll
          for (int j = 0; j < QPG; ++j) {
            a[j] = dot2<T>(qp[j][0], kb[u].x, 0.f);
            a[j] = dot2<T>(qp[j][1], kb[u].y, a[j]);
            a[j] = dot2<T>(qp[j][2], kb[u].z, a[j]);
            a[j] = dot2<T>(qp[j][3], kb[u].w, a[j]);
          }
          xe[0][u] = reduce_scatter16<QPG>(a, li) * p.scale_log2;  // head li % QPG
          sv[0][u] = base + u * TPI + g < c1 ? xe[0][u] : kNegBig;
        }
      }
      if constexpr (EMIT) {
        // The 16 / QPG columns that stand for the same head hold the same sums, so no value has to move
        // between lanes: copy c = c16 / QPG keeps the scores c, c + COPIES, ... of the lane's.  The logits
        // wait in the wave's LDS strip, laid out [tile][head][token], and leave in batches (see emit_flush).
        constexpr int COPIES = 16 / QPG;
        const int head = c16 % QPG, c = c16 / QPG;
        float* strip = emit_buf + (wave * EMIT_TILES + emit_n) * (QPG * TILE);
#pragma unroll
        for (int n0 = 0; n0 < 4 * NB; n0 += COPIES) {
          float e = xe[n0 / 4][n0 % 4];
#pragma unroll
          for (int x = 1; x < COPIES; ++x)
            if (n0 + x < 4 * NB) e = (c == x) ? xe[(n0 + x) / 4][(n0 + x) % 4] : e;
          const int n = n0 + c;
          if (n < 4 * NB) strip[head * TILE + n % 4 * TPI + NB * g4 + n / 4] = e * kLn2;
        }
        emit_push(base);
      }
      float mt = kNegBig;
#pragma unroll
      for (int x = 0; x < NB; ++x) mt = fmaxf(mt, fmaxf(fmaxf(sv[x][0], sv[x][1]), fmaxf(sv[x][2], sv[x][3])));
      mt = rows_max(mt);  // the tile's maximum over all four lane groups
      const float m_new = fmaxf(mh, mt);
      const float alpha = fast_exp2(mh - m_new);
      mh = m_new;
      float pr[NB][4], sum = 0.f;
#pragma unroll
      for (int x = 0; x < NB; ++x) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          pr[x][u] = (base + u * TPI + NB * g4 + x < c1) ? fast_exp2(sv[x][u] - m_new) : 0.f;
        sum += (pr[x][0] + pr[x][1]) + (pr[x][2] + pr[x][3]);
      }
      // The probabilities enter the matrix product in the KV type; the denominator, which also
      // gives the log-sum-exp, stays in fp32.  bf16 keeps 8 bits of a weight (fp16 11): against an
      // exact denominator that is an error of 2^-9 |v| (2^-12 |v|) in o, which with few selected
      // tokens and |v| of 3-4 reached the tolerance together with the rounding of o itself.  The
      // weights are therefore split into parts (weigh_rows).
      lh = fmaf(lh, alpha, sum);
      // rescale the accumulators: row 4g + i belongs to head (4g + i) % QPG; the factors are
      // wave-uniform per head (lane x < QPG holds head x), so they travel through SGPRs
      float ah[QPG];
      bool any = false;
#pragma unroll
      for (int x = 0; x < QPG; ++x) {
        ah[x] = __builtin_bit_cast(
            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, alpha), x));
        any |= ah[x] != 1.f;
      }
      if (any) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float f;
          if constexpr (QPG == 8) {
            float low = ah[i], high = ah[4 + i];
            asm volatile("" : "+v"(low), "+v"(high));  // a choice of registers (else an array in scratch memory)
            f = (g4 & 1) ? high : low;
          } else {
            f = ah[i % QPG];
          }
#pragma unroll
          for (int d = 0; d < NACC; ++d) accm[d][i] *= f;
        }
      }
      weigh_rows<T, D, kParts>(pr, vb, accm);
      return;
    } else {
    float sc[QPG][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + u * TPI + g;
      const bool valid = i < c1;
#pragma unroll
      for (int j = 0; j < QPG; ++j) {
        float a = dot2<T>(qp[j][0], kb[u].x, 0.f);
        a = dot2<T>(qp[j][1], kb[u].y, a);
        a = dot2<T>(qp[j][2], kb[u].z, a);
        a = dot2<T>(qp[j][3], kb[u].w, a);
        a = group_sum<LPR>(a) * p.scale_log2;
        sc[j][u] = valid ? a : kNegBig;
      }
    }
    if constexpr (EMIT) {
      // every lane of a lane group holds the group's U logits, so lane li < U of group g keeps
      // row li (token base + li TPI + g) and nothing moves between lanes; the logits wait in the
      // wave's LDS strip and leave in batches (see emit_flush)
      static_assert(U <= LPR, "one lane of the group per row of the tile");
#pragma unroll
      for (int j = 0; j < QPG; ++j) {  // strip layout [tile][head][token]
        float e = sc[j][0];
#pragma unroll
        for (int u = 1; u < U; ++u) e = (li == u) ? sc[j][u] : e;
        if (li < U)
          emit_buf[((wave * EMIT_TILES + emit_n) * QPG + j) * TILE + li * TPI + g] = e * kLn2;
      }
      emit_push(base);
    }
#pragma unroll
    for (int j = 0; j < QPG; ++j) {
      float mt = sc[j][0];
#pragma unroll
      for (int u = 1; u < U; ++u) mt = fmaxf(mt, sc[j][u]);
      const float m_new = fmaxf(m[j], mt);
      const float alpha = fast_exp2(m[j] - m_new);
      m[j] = m_new;
      float pr[U];
      float ps = 0.f;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        pr[u] = (base + u * TPI + g < c1) ? fast_exp2(sc[j][u] - m_new) : 0.f;
        ps += pr[u];
      }
      l[j] = l[j] * alpha + ps;
#pragma unroll
      for (int d = 0; d < 8; ++d) acc[j][d] *= alpha;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float v0, v1, v2, v3, v4, v5, v6, v7;
        unpack2<T>(vb[u].x, v0, v1);
        unpack2<T>(vb[u].y, v2, v3);
        unpack2<T>(vb[u].z, v4, v5);
        unpack2<T>(vb[u].w, v6, v7);
        acc[j][0] = fmaf(pr[u], v0, acc[j][0]);
        acc[j][1] = fmaf(pr[u], v1, acc[j][1]);
        acc[j][2] = fmaf(pr[u], v2, acc[j][2]);
        acc[j][3] = fmaf(pr[u], v3, acc[j][3]);
        acc[j][4] = fmaf(pr[u], v4, acc[j][4]);
        acc[j][5] = fmaf(pr[u], v5, acc[j][5]);
        acc[j][6] = fmaf(pr[u], v6, acc[j][6]);
        acc[j][7] = fmaf(pr[u], v7, acc[j][7]);
      }
    }
    }
  };

  int t = (split * NW + wave) * TILE;  // first token of this wave's current tile
  if (t < c1) {
    fetch_list(t, rawA);
    if (t + STEP < c1) fetch_list(t + STEP, rawB);
    issue(t, rawA, kA, vA, hitA);
    finish_fresh();
    while (true) {
      // A: K/V of tile t in flight; rawB: list entries of tile t+STEP in flight
      const int tn = t + STEP;
      const int tnn = tn + STEP;
      if (tnn < c1) fetch_list(tnn, rawA);
      if (tn < c1) issue(tn, rawB, kB, vB, hitB);
      reduce(kA, vA, t, hitA);
      if (tn >= c1) break;
      const int tnnn = tnn + STEP;
      if (tnnn < c1) fetch_list(tnnn, rawB);
      if (tnn < c1) issue(tnn, rawA, kA, vA, hitA);
      reduce(kB, vB, tn, hitB);
      if (tnn >= c1) break;
      t = tnn;
    }
  } else {
    finish_fresh();  // a wave without tokens still takes part in the shuffles and the write
  }
  emit_flush();

  // ---- combine the TPI token slots of the wave (butterfly over lane groups) ---------------------
  if constexpr (MMA) {  // the matrix product already summed the groups; only lh is per group
    lh += __shfl_xor(lh, 16, 64);
    lh += __shfl_xor(lh, 32, 64);
  }
#pragma unroll
  for (int j = 0; j < (MMA ? 0 : NV); ++j) {
    float mw = m[j];
#pragma unroll
    for (int off = LPR; off < 64; off <<= 1) mw = fmaxf(mw, __shfl_xor(mw, off, 64));
    const float f = fast_exp2(m[j] - mw);
    m[j] = mw;
    l[j] *= f;
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[j][d] *= f;
#pragma unroll
    for (int off = LPR; off < 64; off <<= 1) {
      l[j] += __shfl_xor(l[j], off, 64);
#pragma unroll
      for (int d = 0; d < 8; ++d) acc[j][d] += __shfl_xor(acc[j][d], off, 64);
    }
  }

  // ---- merge the NW wave states of the workgroup through LDS ------------------------------------
  // every wave publishes its QPG states, one barrier, then wave j reduces query head j
  // (QPG <= NW; heads beyond the waves are handled by the waves again in a second trip)
  auto state = [&](int j, int w, int d, int at) -> float& { return sm_state[w][(j * 8 + d) * LPR + at]; };
  __shared__ float sm_ml[QPG][NW][2];
  __shared__ int sm_ticket;
  if constexpr (MMA) {
#pragma unroll
    for (int j = 0; j < QPG; ++j) {  // head j is row j of the accumulator tile: group j / 4, i = j % 4
      if (g4 == j / 4) {
#pragma unroll
        for (int d = 0; d < NACC; ++d) state(j, wave, LPR == 16 ? d : 4 * (c16 >> 3) + d, li) = accm[d][j % 4] * (1.f / kWeightScale<T, kParts>);
      }
    }
    if (lane < QPG) {
      sm_ml[lane][wave][0] = mh;
      sm_ml[lane][wave][1] = lh;
    }
  } else if (lane < LPR) {
#pragma unroll
    for (int j = 0; j < QPG; ++j) {
#pragma unroll
      for (int d = 0; d < 8; ++d) state(j, wave, d, lane) = acc[j][d];
      if (lane == 0) {
        sm_ml[j][wave][0] = m[j];
        sm_ml[j][wave][1] = l[j];
      }
    }
  }
  __syncthreads();
  for (int j = wave; j < QPG; j += NW) {
    if (lane < LPR) {
      float M = kNegBig;
#pragma unroll
      for (int w = 0; w < NW; ++w) M = fmaxf(M, sm_ml[j][w][0]);
      float L = 0.f, r[8];
#pragma unroll
      for (int d = 0; d < 8; ++d) r[d] = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float f = fast_exp2(sm_ml[j][w][0] - M);
        L = fmaf(sm_ml[j][w][1], f, L);
#pragma unroll
        for (int d = 0; d < 8; ++d) r[d] = fmaf(state(j, w, d, lane), f, r[d]);
      }
      const int qh = rq0 + j;
      if (n_splits == 1) {
        if (j >= gsz) continue;  // a padding head: nothing to write
        const float inv = L > 0.f ? 1.f / L : 0.f;
        u32x4 out;
        out.x = pack2<T>(r[0] * inv, r[1] * inv);
        out.y = pack2<T>(r[2] * inv, r[3] * inv);
        out.z = pack2<T>(r[4] * inv, r[5] * inv);
        out.w = pack2<T>(r[6] * inv, r[7] * inv);
        reinterpret_cast<u32x4*>(p.o)[((int64_t)b * p.num_qo_heads + qh) * LPR + lane] = out;
        if (p.lse && lane == 0)
          p.lse[(int64_t)b * p.num_qo_heads + qh] = L > 0.f ? (M + fast_log2(L)) * kLn2 : -INFINITY;
      } else {
        const int64_t part = part_first + (int64_t)j * part_heads + split;
        float* dst = p.ws_o + part * D + lane * 8;
        store_coherent(dst + 0, r[0], r[1]);
        store_coherent(dst + 2, r[2], r[3]);
        store_coherent(dst + 4, r[4], r[5]);
        store_coherent(dst + 6, r[6], r[7]);
        if (lane == 0) store_coherent(p.ws_ml + part * 2, M, L);
      }
    }
  }

  if (n_splits == 1 || !p.fused_merge) return;

  // ---- the last workgroup of this (sequence, head row) to arrive reduces the partials ----------
  // Ordering.  The partials were stored with device-scope write-through stores (store_coherent,
  // sc1): such a store is acknowledged -- vmcnt decremented -- only once it has reached memory, the
  // point where all XCDs meet.  Every wave waits for its own stores, the barrier collects the
  // waves, and only then does one thread take the ticket, a device-scope atomic performed at
  // memory.  The workgroup that draws the last ticket therefore knows that every other partial of
  // the head row was acknowledged before its writer's ticket was issued, and it reads them with
  // device-scope loads (load_coherent, sc1) that a cache level private to one XCD cannot serve
  // from a stale line.  What would break this: a plain store or load on ws_o / ws_ml (a test greps
  // for that), the compiler moving the ticket above the wait (hence asm volatile with a memory
  // clobber), or dropping the barrier between the waves' waits and the ticket.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int32_t* ticket = p.ws_cnt + ((int64_t)b * p.n_hrows + hrow) * p.ticket_stride;
  if (tid == 0)
    sm_ticket = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (sm_ticket != n_splits - 1) return;
  merge_splits<T, D, QPG, NW * 64>(p, b, part_first, part_heads, rq0, gsz, n_splits);
  if (tid == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Splits are the slowest grid dimension: a sequence shorter than the planned maximum leaves its
// last splits without work, and those workgroups then reach the dispatcher after all the others
// instead of between them (where each one that ends at once hands its place to a workgroup that
// should have gone to an empty compute unit).
template <typename T, int D, int QPG, int U, int NW, bool PAGE_MODE, bool EMIT, bool LEAN, bool FRESH>
__global__ __launch_bounds__(NW * 64) void decode_attn_kernel(const DecodeParams p) {
  attend_share<T, D, QPG, U, NW, PAGE_MODE, EMIT, LEAN, FRESH, true>(p, blockIdx.x, blockIdx.y,
                                                                     Share{(int)blockIdx.z, 0, 0});
}

// A ragged batch on the shared-row kernels, of which a compute unit holds one: the workgroups of whole
// rounds (p.slots per head row) are dealt to the sequences by their lengths, read on the device, so that
// the longest piece is as short as that number allows.  With chunks planned from the longest sequence the
// launch lasts as long as the largest remainder of one, and a batch of short sequences leaves most of the
// chip idle.  One MI355X, bf16, logits out, even chunks -> dealt (us): 16 sequences of 500 .. 8192 tokens,
// 32/8 heads x 128, 77 -> 69.7 (4.7 TB/s); 8 of 8000 .. 60000, 295 -> 261; 4 of 2000, 36.7 -> 15.8; 12 of
// 400 .. 9000, 28/4 heads, 59.7 -> 51; few head rows: 8/1 heads, 16 of 2000 .. 32768, 55 -> 47, 40 of 300 .. 4000,
// 4/1 heads, 26.1 -> 17.1, 16/2 heads, 8 of 8000 .. 65536, 98 -> 88.  The lengths and the search cost 1 us and more
// with many sequences, which is what equal lengths lose (16 x 8192: 95.1 -> 96.2; 8/1 heads, 16 x 32768: 69.7 ->
// 71.0); balancing_pays keeps short ones away.  Runs of equal length laid over the ends of the sequences balance better
// still but pay the start and the merge of every further sequence, 5 us: 72 for the first batch, 110 for
// 16 x 8192.
constexpr int kBalancedMaxBatch = 64;  // one lane per sequence
constexpr int kMergedPieces = 64;      // pieces of a sequence that merge_splits takes

template <typename T, int D, int QPG, int U, int NW, bool EMIT, bool LEAN, bool FRESH>
__global__ __launch_bounds__(NW * 64) void decode_attn_balanced_kernel(const DecodeParams p) {
  constexpr int WTILE = NW * U * (64 / (D / 8));  // tokens of a workgroup-wide tile
  const int lane = threadIdx.x & 63, slot = blockIdx.y;
  SeqList mine;
  int beg;
  seq_items(p, lane < p.batch ? lane : p.batch - 1, mine, beg);
  int tiles = (mine.n_items + WTILE - 1) / WTILE;
  tiles = lane < p.batch ? (tiles < 1 ? 1 : tiles) : 0;
  // the shortest piece, in tiles, for which all sequences together have no more pieces than slots: lane l
  // tries the l-th of 64 lengths between the mean (or what cuts the longest sequence into as many pieces as
  // are merged) and the longest sequence, which always fits
  const int sum = (int)__builtin_amdgcn_readlane(wave_prefix_sum_dpp((uint32_t)tiles, lane), 63);
  const int most = wave_max_i32(tiles);
  const int mean = (sum + p.slots - 1) / p.slots, fewest = (most + kMergedPieces - 1) / kMergedPieces;
  const int least = mean > fewest ? mean : fewest;  // <= most: slots >= batch
  const int piece = least + (most - least) * lane / 63;
  // pieces of a sequence: its tiles over the piece, rounded up.  In floats, exact here (fewer than 2^24 tiles):
  // the quotient is taken a little large, so that its whole part is the floor or one more, and the remainder
  // says whether another piece follows
  const float length = (float)piece, inv = (1.f + 0x1p-21f) / length, tiles_f = (float)tiles;
  float pieces = 0.f;
  for (int b = 0; b < p.batch; b += 4) {  // (lanes past the last sequence hold none)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float n = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, tiles_f), b + i));
      const float q = __builtin_truncf(n * inv);
      pieces += q + (fmaf(-q, length, n) > 0.f ? 1.f : 0.f);
    }
  }
  const uint64_t fits = __ballot(pieces <= (float)p.slots);
  const int chosen = __builtin_amdgcn_readlane(piece, __builtin_ctzll(fits | (1ull << 63)));
  const int n_splits = lane < p.batch ? (tiles + chosen - 1) / chosen : 0;
  const int upto = (int)wave_prefix_sum_dpp((uint32_t)n_splits, lane);  // pieces of the sequences up to this lane's
  const int b = __popcll(__ballot(lane < p.batch && upto <= slot));
  if (b >= p.batch) return;
  const int n = __builtin_amdgcn_readlane(n_splits, b), first = __builtin_amdgcn_readlane(upto, b) - n;
  attend_share<T, D, QPG, U, NW, true, EMIT, LEAN, FRESH, false>(p, blockIdx.x, b, Share{slot - first, n, first});
}

// Second-kernel merge (plan.fused_merge == 0): one workgroup per (head row, sequence).
template <typename T, int D, int QPG, int NT>
__global__ __launch_bounds__(NT) void merge_partials_kernel(const DecodeParams p) {
  const int hrow = blockIdx.x;
  const int b = blockIdx.y;
  SeqList s;
  int list_beg;
  const int n_splits = seq_items(p, b, s, list_beg);
  if (n_splits <= 1) return;  // the attention kernel already wrote the final result
  int kv_head, rq0, gsz;
  head_row_geom<QPG>(p, hrow, kv_head, rq0, gsz);
  merge_splits<T, D, QPG, NT>(p, b, ((int64_t)b * p.vheads + hrow * QPG) * p.max_splits, p.max_splits, rq0, gsz,
                              n_splits);
}

// ---------------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------------

// Instantiated shapes (tile_rows = K/V load instructions per wave tile):
//   one query head per head row: head_dim 64/128/256, 8 waves x {2, 4} rows or 16 waves x 4 rows;
//   2, 4 or 8 query heads per head row (KV rows shared inside a GQA group): head_dim 64 and 128
//   (256: 2 or 4), 8 waves x 4 rows; weighted values on the matrix cores (256: on the vector ALU), and scores too
//   for 8 heads and for head_dim 64.
static bool shape_supported(int head_dim, int qpg, int nw, int rows = 4) {
  if (qpg == 1)
    return (head_dim == 64 || head_dim == 128 || head_dim == 256) &&
           ((nw == 8 && (rows == 2 || rows == 4)) || (nw == 16 && rows == 4));
  if (nw != 8 || rows != 4) return false;
  if (head_dim == 256) return qpg == 2 || qpg == 4;  // the split merge holds qpg * head_dim <= 1024
  return (head_dim == 64 || head_dim == 128) && (qpg == 2 || qpg == 4 || qpg == 8);
}

// Query heads scored per loaded KV row.  KV rows are shared between the query heads of a GQA
// group only when the group shares its list and a kernel for that shape exists; otherwise every
// query head walks the list on its own (same result, the KV rows are read once per query head).
static int qpg_for(int num_qo_heads, int num_kv_heads, int idx_rows, int head_dim) {
  const int group = num_qo_heads / num_kv_heads;
  if (group <= 1 || idx_rows == num_qo_heads) return 1;
  // groups of 3 run on the 4-head kernel, 5 to 7 on the 8-head kernel, larger ones as several head
  // rows of 8 (of 4 for head_dim 256): the padding heads cost arithmetic, not memory traffic,
  // which is what bounds these kernels
  int padded = group <= 2 ? 2 : (group <= 4 ? 4 : 8);
  if (head_dim == 256 && padded > 4) padded = 4;
  return shape_supported(head_dim, padded, 8) ? padded : 1;
}

template <typename T, int D, int QPG, int NW, int U, bool EMIT>
static void launch_balanced(const DecodeParams& p, dim3 grid, hipStream_t st) {
  const dim3 even(grid.x, p.slots);
  if (p.lean && p.fresh_k)
    hipLaunchKernelGGL((decode_attn_balanced_kernel<T, D, QPG, U, NW, EMIT, true, true>), even, dim3(NW * 64), 0, st, p);
  else if (p.lean)
    hipLaunchKernelGGL((decode_attn_balanced_kernel<T, D, QPG, U, NW, EMIT, true, false>), even, dim3(NW * 64), 0, st, p);
  else
    hipLaunchKernelGGL((decode_attn_balanced_kernel<T, D, QPG, U, NW, EMIT, false, false>), even, dim3(NW * 64), 0, st, p);
}

template <typename T, int D, int QPG, int NW, int U, bool PAGE_MODE, bool EMIT>
static void launch_lean(const DecodeParams& p, dim3 grid, hipStream_t st) {
  if (p.lean && p.fresh_k)
    hipLaunchKernelGGL((decode_attn_kernel<T, D, QPG, U, NW, PAGE_MODE, EMIT, true, true>), grid,
                       dim3(NW * 64), 0, st, p);
  else if (p.lean)
    hipLaunchKernelGGL((decode_attn_kernel<T, D, QPG, U, NW, PAGE_MODE, EMIT, true, false>), grid,
                       dim3(NW * 64), 0, st, p);
  else
    hipLaunchKernelGGL((decode_attn_kernel<T, D, QPG, U, NW, PAGE_MODE, EMIT, false, false>), grid,
                       dim3(NW * 64), 0, st, p);
}

template <typename T, int D, int QPG, int NW, int U>
static void launch_variant(const DecodeParams& p, bool page_mode, bool emit, bool merge_kernel,
                           dim3 grid, hipStream_t st) {
  if constexpr (QPG > 1) {
    if (p.slots > 0) {
      if (emit)
        launch_balanced<T, D, QPG, NW, U, true>(p, grid, st);
      else
        launch_balanced<T, D, QPG, NW, U, false>(p, grid, st);
      return;
    }
  }
  if (page_mode) {
    if (emit)
      launch_lean<T, D, QPG, NW, U, true, true>(p, grid, st);
    else
      launch_lean<T, D, QPG, NW, U, true, false>(p, grid, st);
  } else {
    if (emit)
      launch_lean<T, D, QPG, NW, U, false, true>(p, grid, st);
    else
      launch_lean<T, D, QPG, NW, U, false, false>(p, grid, st);
  }
  if (merge_kernel)
    hipLaunchKernelGGL((merge_partials_kernel<T, D, QPG, 512>), dim3(grid.x, grid.y), dim3(512), 0,
                       st, p);
}

template <typename T>
static int launch_shape(const DecodeParams& p, int head_dim, int qpg, int nw, int rows,
                        bool page_mode, bool emit, bool merge_kernel, dim3 grid, hipStream_t st) {
#define TD_CASE(D_, Q_, N_, U_)                                                    \
  if (head_dim == D_ && qpg == Q_ && nw == N_ && rows == U_) {                     \
    launch_variant<T, D_, Q_, N_, U_>(p, page_mode, emit, merge_kernel, grid, st); \
    return TD_OK;                                                                  \
  }
  TD_CASE(64, 1, 8, 4)
  TD_CASE(64, 1, 8, 2)
  TD_CASE(64, 1, 16, 4)
  TD_CASE(128, 1, 8, 4)
  TD_CASE(128, 1, 8, 2)
  TD_CASE(128, 1, 16, 4)
  TD_CASE(256, 1, 8, 4)
  TD_CASE(256, 1, 8, 2)
  TD_CASE(256, 1, 16, 4)
  TD_CASE(128, 2, 8, 4)
  TD_CASE(128, 4, 8, 4)
  TD_CASE(128, 8, 8, 4)
  TD_CASE(64, 2, 8, 4)
  TD_CASE(64, 4, 8, 4)
  TD_CASE(64, 8, 8, 4)
  TD_CASE(256, 2, 8, 4)
  TD_CASE(256, 4, 8, 4)
#undef TD_CASE
  return fail(TD_ERR_UNSUPPORTED,
              "BatchDecodeWithPagedKVCache failed to dispatch: head_dim %d with %d query heads per "
              "shared KV row and %d waves (supported: head_dim 64/128/256 with per-head lists; "
              "shared lists with 2, 4 or 8 heads per row, 2 or 4 for head_dim 256)",
              head_dim, qpg, nw);
}

// Launches the instantiation for (head_dim, qpg, nw, page_mode, emit); defined once per element
// type in decode_attn_f16.hip / decode_attn_bf16.hip so that the two halves compile in parallel.
int launch_decode_f16(const DecodeParams& p, int head_dim, int qpg, int nw, int rows, bool page_mode,
                      bool emit, bool merge_kernel, dim3 grid, hipStream_t st);
int launch_decode_bf16(const DecodeParams& p, int head_dim, int qpg, int nw, int rows,
                       bool page_mode, bool emit, bool merge_kernel, dim3 grid, hipStream_t st);

}  // namespace tidal
