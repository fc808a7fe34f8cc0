// Sparse-layer decode attention for gfx950 (MI355X): the short-list form of decode_attn_kernel, for head_dim 64 and
// 128, one query head per list walk or up to eight that share one, token-slot or page lists, with or without logits.
// Pools of 4 GiB and more and pages that are no power of two: head_dim 128, token-slot lists, no logits.  Same
// arguments, same split workspace and the same results as decode_attn_kernel;
// what differs is the shape of the work, chosen for launches that move a few tens of MiB and are
// bound by dependent round trips and instruction issue rather than by bandwidth:
//
//   * a wave owns 4 U tokens, 8 U at head_dim 64 (U = 8 or 16 K rows and as many V rows per lane: 64 or 128
//     VGPRs of loads), all of them in flight at once, K rows first so that q.k runs while V arrives;
//   * the list entry of a token is loaded once, by the lane that owns the token; its byte offset
//     reaches the 16 (8) lanes of a row through DPP row broadcasts (one or two instructions per row);
//   * one head: q.k partial sums are reduce-scattered over the lanes of a row, so that after U partial
//     dot products a lane holds the complete logit of ONE token and the softmax arithmetic runs
//     once per token instead of once per lane; the probabilities go back through row broadcasts;
//   * shared rows: both products on the matrix cores, the keys through the wave's own LDS into operand layout;
//   * the maximum is wave-uniform per tile, so the lane groups add up without rescaling;
//   * the workgroup's waves meet once in LDS, then wave j alone publishes the partials of the heads j, j + NW, ..,
//     takes their tickets and, where it is the last of a head, merges the partials (no further barrier).
//
// Semantics follow kernels/include/decode/decode_attn.cuh:432-658 of the reference
// (BatchDecodeWithPagedKVCacheKernel) including the forced last page (decode_page.cuh:320-346).

#pragma once

#include "decode_attn.cuh"

namespace tidal {

// value of lane N of this lane's 16-lane row (DPP row_newbcast)
template <int N>
__device__ __forceinline__ uint32_t row_bcast_u32(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x150 + N, 0xf, 0xf, true);
}
// value of lane N of this lane's group of LPR = 8 or 16 lanes
template <int N, int LPR>
__device__ __forceinline__ uint32_t group_bcast_u32(uint32_t x) {
  if constexpr (LPR == 16) {
    return row_bcast_u32<N>(x);
  } else {
    const int low = (int)row_bcast_u32<N % 8>(x);  // the upper eight lanes take theirs
    return (uint32_t)__builtin_amdgcn_update_dpp(low, (int)x, 0x150 + N % 8 + 8, 0xf, 0xc, false);
  }
}
template <int N, int LPR>
__device__ __forceinline__ float group_bcast_f32(float x) {
  return __builtin_bit_cast(float, group_bcast_u32<N, LPR>(__builtin_bit_cast(uint32_t, x)));
}

// a[u] = this lane's partial sum for row u (U rows, U = 8 or 16) over its 8 dimensions; returns the sum over
// the LPR = 8 or 16 lanes of the row group for row (lane % U).  Each butterfly step
// halves the rows a lane keeps and hands the other half to a partner whose lane index differs in
// the step's bit (any partner of the opposite class does, as long as every lane's contribution is
// counted once: xor 1, xor 2, rotate by 4, rotate by 8).
template <int U, int LPR>
__device__ __forceinline__ float reduce_scatter_rows(float (&a)[U], int li) {
  static_assert(U == 8 || (U == 16 && LPR == 16), "rows per lane group");
  float c1[U / 2], c2[U / 4], c3[U / 8];
  {
    const bool hi = li & 1;
#pragma unroll
    for (int i = 0; i < U / 2; ++i) {
      const float keep = hi ? a[2 * i + 1] : a[2 * i];
      const float send = hi ? a[2 * i] : a[2 * i + 1];
      c1[i] = keep + dpp_move<0xB1>(send);  // quad_perm [1,0,3,2]
    }
  }
  {
    const bool hi = li & 2;
#pragma unroll
    for (int i = 0; i < U / 4; ++i) {
      const float keep = hi ? c1[2 * i + 1] : c1[2 * i];
      const float send = hi ? c1[2 * i] : c1[2 * i + 1];
      c2[i] = keep + dpp_move<0x4E>(send);  // quad_perm [2,3,0,1]
    }
  }
  {
    const bool hi = li & 4;
#pragma unroll
    for (int i = 0; i < U / 8; ++i) {
      const float keep = hi ? c2[2 * i + 1] : c2[2 * i];
      const float send = hi ? c2[2 * i] : c2[2 * i + 1];
      // row_ror:4: the sender sits in the other quad class; rows of eight lanes exchange with lane ^ 4
      c3[i] = keep + (LPR == 16 ? dpp_move<0x124>(send) : lane_xor16<4>(send));
    }
  }
  if constexpr (U == 16) {
    const bool hi = li & 8;
    const float keep = hi ? c3[1] : c3[0];
    const float send = hi ? c3[0] : c3[1];
    return keep + dpp_move<0x128>(send);  // row_ror:8
  } else if constexpr (LPR == 16) {
    return c3[0] + dpp_move<0x128>(c3[0]);  // lanes li and li ^ 8 hold the same row
  } else {
    return c3[0];
  }
}

// maximum / sum over the 16 lanes of a row, result in every lane
__device__ __forceinline__ float row16_max(float x) {
  x = fmaxf(x, dpp_move<0xB1>(x));
  x = fmaxf(x, dpp_move<0x4E>(x));
  x = fmaxf(x, dpp_move<0x141>(x));
  x = fmaxf(x, dpp_move<0x140>(x));
  return x;
}

// exchange between the halves / the odd and even 16-lane rows of a wavefront: (a, b) -> x, y with
//   swap32: x = [a.lower | b.lower], y = [a.upper | b.upper]
//   swap16: x = [a.row0 | b.row0 | a.row2 | b.row2], y = [a.row1 | b.row1 | a.row3 | b.row3]
__device__ __forceinline__ void swap32(float a, float b, float& x, float& y) {
  const u32pair r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a),
                                                     __builtin_bit_cast(uint32_t, b), false, false);
  const uint32_t lo = r.x, hi = r.y;
  x = __builtin_bit_cast(float, lo);
  y = __builtin_bit_cast(float, hi);
}
__device__ __forceinline__ void swap16(float a, float b, float& x, float& y) {
  const u32pair r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a),
                                                     __builtin_bit_cast(uint32_t, b), false, false);
  const uint32_t lo = r.x, hi = r.y;
  x = __builtin_bit_cast(float, lo);
  y = __builtin_bit_cast(float, hi);
}

// Wave-uniform words of device-resident state, fetched through the scalar cache in one round trip
// (the compiler cannot: the kernel also writes memory, so it would use a vector load and a full
// wait for each word).  The words were written by earlier launches; a launch starts with a clean
// scalar cache.
__device__ __forceinline__ void scalar_load2(const int32_t* a0, const int32_t* a1, int32_t& v0,
                                             int32_t& v1) {
  asm volatile(
      "s_load_dword %0, %2, 0x0\n\t"
      "s_load_dword %1, %3, 0x0\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&s"(v0), "=&s"(v1)
      : "s"(a0), "s"(a1)
      : "memory");
}
__device__ __forceinline__ void scalar_load4(const int32_t* a0, const int32_t* a1, const int32_t* a2,
                                             const int32_t* a3, int32_t& v0, int32_t& v1, int32_t& v2,
                                             int32_t& v3) {
  asm volatile(
      "s_load_dword %0, %4, 0x0\n\t"
      "s_load_dword %1, %5, 0x0\n\t"
      "s_load_dword %2, %6, 0x0\n\t"
      "s_load_dword %3, %7, 0x0\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&s"(v0), "=&s"(v1), "=&s"(v2), "=&s"(v3)
      : "s"(a0), "s"(a1), "s"(a2), "s"(a3)
      : "memory");
}

__device__ __forceinline__ const float* bytes_on(const float* base, uint32_t bytes) {
  return reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + bytes);
}

// The tail of a head's computation, run by ONE wave that holds the workgroup's partial result of that head (lane:
// dimensions 2 lane, 2 lane + 1; M, L uniform): publish_head writes the result if the head was not split, else the
// partial; after the ticket merge_head, in the last of the splits to arrive, merges all partials.
template <typename T, int D>
__device__ __forceinline__ void publish_head(const DecodeParams& p, int lane, int n_splits, int64_t part, uint32_t* o32,
                                             float* lse_out, float o0, float o1, float M, float L) {
  const bool live = D == 128 || lane < D / 2;  // lanes that hold dimensions
  if (n_splits == 1) {
    const float inv = L > 0.f ? 1.f / L : 0.f;
    if (live) *o32 = pack2<T>(o0 * inv, o1 * inv);
    if (lse_out && lane == 0) *lse_out = L > 0.f ? (M + fast_log2(L)) * kLn2 : -INFINITY;
    return;
  }
  if (live) store_coherent(p.ws_o + part * D + 2 * lane, o0, o1);
  if (lane == 0) store_coherent(p.ws_ml + part * 2, M, L);
}

// Ordering.  A head's partial was stored by one wave alone, with device-scope write-through stores
// (sc1): such a store is acknowledged -- vmcnt decremented -- only when it has reached memory, the
// point where all XCDs meet, so after the caller's s_waitcnt vmcnt(0) the partial is visible device-wide.
// Only then is the ticket taken; the increment is a device-scope atomic performed at memory,
// so a wave that draws the last ticket knows that every other partial of the head had been
// acknowledged before its own ticket was even issued.  It reads them with device-scope loads
// (sc1), which do not hit lines a non-coherent cache level may still hold from earlier
// launches.  What would break this: a plain (non-sc1) store or load on ws_o / ws_ml, a compiler
// that moved the ticket above the wait (hence asm volatile with a memory clobber), or partials
// stored by several waves without a barrier between their waits and the ticket.
template <typename T, int D>
__device__ __forceinline__ void merge_head(const DecodeParams& p, int lane, int n_splits, int64_t part0, int32_t* ticket,
                                           uint32_t* o32, float* lse_out) {
  const bool live = D == 128 || lane < D / 2;
  float pm = kNegBig, pl = 0.f;  // (m, l) of split `lane`
  {
    const int sidx = lane < n_splits ? lane : n_splits - 1;
    float a, c;
    load_coherent(p.ws_ml + (part0 + sidx) * 2, a, c);
    if (lane < n_splits) { pm = a; pl = c; }
  }
  constexpr int PRE = 16;  // partial loads in flight
  float pa[PRE], pb[PRE];
  // 32-bit byte offsets from one scalar base: the loads go out two instructions apart instead of five
  const uint32_t mine = 8u * (uint32_t)(lane & (D / 2 - 1)), last = (uint32_t)(n_splits - 1) * (D * 4);
  auto issue = [&](int base) {
#pragma unroll
    for (int u = 0; u < PRE; ++u) {
      const uint32_t at = (uint32_t)(base + u) * (D * 4);
      load_coherent(bytes_on(p.ws_o + part0 * D, (at < last ? at : last) + mine), pa[u], pb[u]);
    }
  };
  issue(0);
  const float Mx = rows_max(row16_max(pm));
  const float pf = fast_exp2(pm - Mx);  // scale of split `lane` (0 for lanes past the splits: pl = 0)
  const float Lx = rows_sum(group_sum<16>(pl * pf));
  float ra = 0.f, rb = 0.f;
  for (int base = 0; base < n_splits; base += PRE) {
    if (base) issue(base);
#pragma unroll
    for (int u = 0; u < PRE; ++u) {
      const int sidx = base + u;  // uniform
      if (sidx < n_splits) {
        const float f = __builtin_bit_cast(
            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, pf), sidx));
        ra = fmaf(pa[u], f, ra);
        rb = fmaf(pb[u], f, rb);
      }
    }
  }
  const float inv = Lx > 0.f ? 1.f / Lx : 0.f;
  if (live) *o32 = pack2<T>(ra * inv, rb * inv);
  if (lse_out && lane == 0) *lse_out = Lx > 0.f ? (Mx + fast_log2(Lx)) * kLn2 : -INFINITY;
  if (lane == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// QPG query heads per loaded K/V row: 1 (every head row is a query head with its own walk of a
// list) or the up to 2, 4 or 8 query heads of a KV head that share one list (a head row is a KV head;
// groups of 3, 5, 6 and 7 leave head slots empty).  ANY: page lists, score output (compiled apart: the branches
// cost the plain walk of token slots 1 - 2 %).
template <typename T, int NW, int U, bool FRESH, bool PROBE = false, int QPG = 1, bool WIDE = false, int D = 128, bool ANY = false>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(1, U == 16 ? 2 : 4))) void sparse_attn_kernel(const DecodeParams p) {
  static_assert(QPG == 1 || U == 8, "shared KV rows: 8 rows per lane");
  constexpr int LPR = D / 8;            // lanes per K/V row
  constexpr int TILE = 64 / LPR * U;    // tokens of a wave tile: lane group g holds tokens g U .. g U + U - 1
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane / LPR, li = lane % LPR;
  const int g4 = lane >> 4, c16 = lane & 15;  // 16-lane row and place in it (operands of the matrix products)
  const int hrow = blockIdx.x, b = blockIdx.y, split = blockIdx.z;
  // One batch of scalar loads for every kernel argument the main path uses: the compiler would
  // otherwise fetch them where they are first needed, a dependent round trip each time.
#define TD_TOUCH(x) asm volatile("" ::"s"(x))
  TD_TOUCH(p.q); TD_TOUCH(p.kv); TD_TOUCH(p.v_offset); TD_TOUCH(p.idx); TD_TOUCH(p.indptr);
  TD_TOUCH(p.count_arr); TD_TOUCH(p.last_len_arr); TD_TOUCH(p.last_idx_arr);
  TD_TOUCH(p.idx_row_stride); TD_TOUCH(p.idx_cols); TD_TOUCH(p.n_list_host); TD_TOUCH(p.kv_magic);
  TD_TOUCH(p.chunk_magic); TD_TOUCH(p.max_splits); TD_TOUCH(p.page_shift); TD_TOUCH(p.max_slot);
  TD_TOUCH(p.page_stride_b); TD_TOUCH(p.entry_stride_b); TD_TOUCH(p.head_stride);
  TD_TOUCH(p.ws_cnt); TD_TOUCH(p.o); TD_TOUCH(p.lse); TD_TOUCH(p.vheads);
  TD_TOUCH(p.ticket_stride); TD_TOUCH(p.fused_merge);
  TD_TOUCH(p.last_len); TD_TOUCH(p.last_idx); TD_TOUCH(p.scale_log2); TD_TOUCH(p.num_qo_heads);
  if constexpr (FRESH) {
    TD_TOUCH(p.fresh_k); TD_TOUCH(p.fresh_v); TD_TOUCH(p.fresh_cos); TD_TOUCH(p.fresh_sin);
    TD_TOUCH(p.fresh_slot);
  }
#undef TD_TOUCH
  // hrow / q_per_kv: kv_magic is 2^24 / q_per_kv rounded up, exact for the head rows that tickets exist for
  const int list_shift = ANY ? p.list_shift : 0;
  const int kv_head = QPG > 1 ? hrow : (int)(((uint64_t)(uint32_t)hrow * p.kv_magic) >> 24);
  const int rq0 = QPG > 1 ? hrow * p.q_per_kv : hrow;  // first query head of the head row
  const int gsz = QPG > 1 ? p.q_per_kv : 1;            // its query heads: at most QPG
  const int own = g * U + (li & (U - 1));  // the token of the tile this lane owns

  // ---- everything that depends on the kernel arguments only is requested at once ---------------
  // The list entries of the first tile are read before the length of the list is known.  The
  // position is clamped to what the sequence's segment of the row is known to hold whatever the
  // device-resident count says: at most n_list_host columns (which the host has checked against
  // the row stride for a segment that starts at column 0), no further than the segment's end
  // indptr[b + 1], and never beyond the row itself.
  const int t0 = (split * NW + wave) * TILE;
  const int idx_row = (QPG > 1 || p.idx_per_kv) ? kv_head : hrow;
  int list_beg = 0, list_end = 0;
  if (p.indptr) scalar_load2(p.indptr + b, p.indptr + b + 1, list_beg, list_end);
  const int32_t* row = p.idx + (int64_t)idx_row * p.idx_row_stride + list_beg;
  const int cap = list_capacity(p.n_list_host, p.indptr != nullptr, list_beg, list_end, p.idx_cols);
  auto fetch_entry = [&](int t) -> int32_t {
    int pos = (t + own) >> list_shift;
    pos = pos < cap ? pos : cap - 1;
    return cap > 0 ? row[pos] : 0;
  };
  int32_t ent = fetch_entry(t0);

  // ---- q, and in the fused decode step (FRESH) what the workgroup's first wave prepares ----------
  // FRESH: q arrives un-rotated.  Wave 0 of the workgroup alone loads q, the step's cos / sin and
  // the new token's k and v, rotates q and k once, and leaves rotated q, rotated k and v in LDS for
  // the other waves (which then issue no global load besides their list entry and K/V rows: eight
  // waves per workgroup asking the same few cache lines for cos / sin cost the launch 0.5 us).
  // One head: 8 elements per lane.  Shared rows: operand of the matrix product, column c16 is head
  // c16 % QPG (empty head slots repeat the last head), elements [32 x + 8 g4, +8).
  constexpr int NQ = QPG > 1 ? D / 32 : 1;
  u32x4 qp[NQ];
  auto load_q = [&](auto piece) __attribute__((always_inline)) {  // piece(head, 16-byte piece)
    const int j = c16 % QPG < gsz ? c16 % QPG : gsz - 1;
#pragma unroll
    for (int x = 0; x < NQ; ++x) qp[x] = QPG > 1 ? piece(j, 4 * x + g4) : piece(0, li);
  };
  const bool prep = FRESH && wave == 0;  // scalar
  const u32x4* const q_rows = reinterpret_cast<const u32x4*>(p.q) + ((int64_t)b * p.num_qo_heads + rq0) * LPR;
  if constexpr (!FRESH) load_q([&](int j, int c) { return q_rows[j * LPR + c]; });
  // What wave 0 loads for the fused step.  Defined in that wave only and read in that wave only:
  // giving the other waves a value here would make them wait for their list entry first (the
  // registers are the destination of loads in flight on the other side of the branch).
  constexpr int GR = 64 / LPR, QX = (QPG + GR - 1) / GR;  // lane group g prepares the heads g, g + GR, ...
  u32x4 q_raw[QX], kn_raw, vn_raw;
  f32x4 cos_lo, cos_hi, sin_lo, sin_hi;
  if constexpr (FRESH) {
    if (prep) {
#pragma unroll
      for (int x = 0; x < QX; ++x) q_raw[x] = q_rows[(g + x * GR < gsz ? g + x * GR : gsz - 1) * LPR + li];
      constexpr int HALF = LPR / 2;
      const f32x4* cp = reinterpret_cast<const f32x4*>(p.fresh_cos + (int64_t)b * (D / 2) + (li % HALF) * 8);
      const f32x4* sp = reinterpret_cast<const f32x4*>(p.fresh_sin + (int64_t)b * (D / 2) + (li % HALF) * 8);
      cos_lo = cp[0]; cos_hi = cp[1]; sin_lo = sp[0]; sin_hi = sp[1];
      const int64_t fresh_off = ((int64_t)b * p.num_kv_heads + kv_head) * LPR + li;
      kn_raw = reinterpret_cast<const u32x4*>(p.fresh_k)[fresh_off];
      vn_raw = reinterpret_cast<const u32x4*>(p.fresh_v)[fresh_off];
    }
  }

  // ---- the sequence: listed entries, forced last page, splits ------------------------------------
  // (seq_items of decode_attn.cuh with the division by the chunk size as a product)
  SeqList s;
  s.n_list = p.n_list_host;
  s.last_len = p.last_len;
  s.last_idx = p.last_idx;
  // slot of the token being decoded (FRESH): it travels with the other state words, load and wait
  // inside one asm statement, so that no register allocation can read it before it has landed; the
  // list entry, which the row loads wait for anyway, is in flight over the same round trip
  uint32_t new_slot = 0xffffffffu;
  if (FRESH || p.count_arr || p.last_len_arr || p.last_idx_arr) {
    // absent arrays read a dummy word (q is never NULL) and keep the host value
    const int32_t* dummy = reinterpret_cast<const int32_t*>(p.q);
    int32_t cnt, ll, lx, ns;
    scalar_load4(p.count_arr ? p.count_arr + b : dummy, p.last_len_arr ? p.last_len_arr + b : dummy,
                 p.last_idx_arr ? p.last_idx_arr + b : dummy, FRESH ? p.fresh_slot + b : dummy, cnt, ll,
                 lx, ns);
    if (p.indptr) s.n_list = p.count_arr ? cnt : list_end - list_beg;
    if (p.last_len_arr) s.last_len = ll;
    if (p.last_idx_arr) s.last_idx = lx;
    if constexpr (FRESH) new_slot = (uint32_t)ns;
  } else if (p.indptr) {
    s.n_list = list_end - list_beg;
  }
  // a count beyond what the first fetch was clamped to would pair tokens with the wrong entries
  s.n_list = s.n_list < 0 ? 0 : (s.n_list > cap ? cap : s.n_list);
  s.last_len = s.last_len < 0 ? 0 : (s.last_len > p.page_size ? p.page_size : s.last_len);
  const int n_listed = s.n_list << list_shift;  // tokens: an entry is a slot, or a page of 2^list_shift of them
  const int c1 = n_listed + s.last_len;
  int n_splits = (int)__umulhi((uint32_t)(c1 + p.chunk_tokens - 1), p.chunk_magic);
  n_splits = n_splits > p.max_splits ? p.max_splits : n_splits;
  n_splits = n_splits < 1 ? 1 : n_splits;
  if (split >= n_splits) return;  // uniform for the workgroup
  const uint32_t last_base = (uint32_t)s.last_idx * (uint32_t)p.page_size;

  const char* kbase = reinterpret_cast<const char*>(p.kv);
  const char* vbase = kbase + p.v_offset * 2;
  const uint32_t head_byte_off = (uint32_t)(kv_head * p.head_stride + li * 8) * 2u;
  const uint32_t entry_mask = (1u << (p.page_shift & 31)) - 1u;
  // Byte offset of a token slot's K row of head 0 in the pool.  Lean form: power-of-two pages, a
  // pool below 4 GiB and strides that fit the 24-bit multiplier.  Wide form: any page size (one
  // division per lane and tile) and 64-bit offsets.
  using off_t = typename std::conditional<WIDE, uint64_t, uint32_t>::type;
  auto slot_offset = [&](uint32_t slot) -> off_t {
    if constexpr (WIDE) {
      uint32_t page, entry;
      if (p.page_shift >= 0) {
        page = slot >> p.page_shift;
        entry = slot & entry_mask;
      } else {
        page = slot / (uint32_t)p.page_size;
        entry = slot - page * (uint32_t)p.page_size;
      }
      return (uint64_t)page * (uint64_t)p.page_stride_b + (uint64_t)(entry * p.entry_stride_b);
    } else {
      return __umul24(slot >> p.page_shift, p.page_stride_b) + __umul24(slot & entry_mask, p.entry_stride_b);
    }
  };

  float m_run = kNegBig;  // wave-uniform running maximum (base-2 logits)
  float l_lane = 0.f;     // this lane's share of the denominator
  float acc[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) acc[d] = 0.f;
  // Shared KV rows (QPG > 1): the lane's head is c16 % QPG; its maximum is equal in all lanes of the wave, lh the
  // lane's share of its denominator, and accm[e][r] = o[head (4 g4 + r) % QPG] of the lane's dimension e
  // (head_dim 128: li 8 + e; 64: li 8 + 4 (c16 / 8) + e), already summed over the lane groups.
  float mh = kNegBig, lh = 0.f;
  constexpr int NACC = QPG > 1 ? D / 16 : 1;
  constexpr WeightParts kParts = D == 64 || std::is_same<T, F16>::value ? kWhole : kRounded;
  f32x4 accm[NACC];
#pragma unroll
  for (int d = 0; d < NACC; ++d) accm[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  // a wave's key tile on its way to operand layout; the wave states at the end of the launch
  constexpr int STATE_F = QPG > 1 && TILE * D / 2 > QPG * D ? TILE * D / 2 : QPG * D;  // floats per wave
  __shared__ __attribute__((aligned(16))) float sm_state[NW][STATE_F];
  // fused decode step: rotated q rows, the new token's rotated key and its value, D elements each
  __shared__ __attribute__((aligned(16))) uint32_t sm_fresh[FRESH ? (QPG + 2) * D / 2 : 4];
  uint32_t* const sm_knew = sm_fresh + (FRESH ? QPG * D / 2 : 0);
  uint32_t* const sm_vnew = sm_knew + (FRESH ? D / 2 : 0);

  // ---- one tile of the wave: slot and row offset of the lane's own token, then every K and V row ----
  u32x4 kb[U], vb[U];
  uint32_t slot = 0;   // of this lane's token
  bool valid = false;  // the token exists
  auto issue = [&](int t, int32_t entry_raw) {
    const int i = t + own;
    valid = i < c1;
    // entry_raw was read at min(i, capacity - 1), which is i for every listed token (n_list <= capacity)
    slot = i < n_listed ? ((uint32_t)entry_raw << list_shift) + (uint32_t)(i & ((1 << list_shift) - 1))
                        : last_base + (uint32_t)(i - n_listed);
    slot = slot > p.max_slot ? p.max_slot : slot;
    off_t off_own = slot_offset(slot);
    // lanes past the end of the list repeat the first token of the tile (which exists: t < c1)
    // with weight 0: a row that holds real data, whatever the unused list entries say
    if constexpr (WIDE) {
      const uint32_t lo = (uint32_t)off_own, hi = (uint32_t)(off_own >> 32);
      const uint32_t lo0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)lo);
      const uint32_t hi0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)hi);
      const uint32_t lo_own = valid ? lo : lo0, hi_own = valid ? hi : hi0;
      const char* ka[U];
#define TD_ROW_OFF(N)                                                                              \
  if constexpr (N < U)                                                                             \
    ka[N] = kbase + ((((uint64_t)group_bcast_u32<N, LPR>(hi_own)) << 32) | (uint64_t)group_bcast_u32<N, LPR>(lo_own)) + \
            head_byte_off;
      TD_ROW_OFF(0) TD_ROW_OFF(1) TD_ROW_OFF(2) TD_ROW_OFF(3) TD_ROW_OFF(4) TD_ROW_OFF(5)
      TD_ROW_OFF(6) TD_ROW_OFF(7) TD_ROW_OFF(8) TD_ROW_OFF(9) TD_ROW_OFF(10) TD_ROW_OFF(11)
      TD_ROW_OFF(12) TD_ROW_OFF(13) TD_ROW_OFF(14) TD_ROW_OFF(15)
#undef TD_ROW_OFF
#pragma unroll
      for (int u = 0; u < U; ++u)
        kb[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(ka[u]));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u)
        vb[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(ka[u] + p.v_offset * 2));
    } else {
      // in a statement of its own: inside the conditional the first lane would be the first one
      // WITHOUT a token
      const uint32_t off_first = (uint32_t)__builtin_amdgcn_readfirstlane((int)off_own);
      off_own = valid ? off_own : off_first;
      uint32_t offs[U];
#define TD_ROW_OFF(N) \
  if constexpr (N < U) offs[N] = group_bcast_u32<N, LPR>(off_own) + head_byte_off;
      TD_ROW_OFF(0) TD_ROW_OFF(1) TD_ROW_OFF(2) TD_ROW_OFF(3) TD_ROW_OFF(4) TD_ROW_OFF(5)
      TD_ROW_OFF(6) TD_ROW_OFF(7) TD_ROW_OFF(8) TD_ROW_OFF(9) TD_ROW_OFF(10) TD_ROW_OFF(11)
      TD_ROW_OFF(12) TD_ROW_OFF(13) TD_ROW_OFF(14) TD_ROW_OFF(15)
#undef TD_ROW_OFF
#pragma unroll
      for (int u = 0; u < U; ++u)
        kb[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kbase + offs[u]));
      // (left to itself the compiler takes K and V by turns, and q.k waits for all but the last V row: 32 heads,
      // lists of 3500, a card at low clocks, 464 -> 452 us for 16 layers)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u)
        vb[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vbase + offs[u]));
    }
  };

  // one logit (base 2 in, natural out) of a selection layer
  auto emit = [&](bool mine, int head, int i, float logit2) __attribute__((always_inline)) {
    if (mine && i < c1) {
      const int64_t at = ((int64_t)b * p.num_qo_heads + head) * p.score_stride + i;
      if (p.scores_f32)
        reinterpret_cast<float*>(p.scores)[at] = logit2 * kLn2;
      else
        reinterpret_cast<uint16_t*>(p.scores)[at] = from_float<T>(logit2 * kLn2);
    }
  };

  // ---- arithmetic of the tile (of tokens t ..) whose rows `issue` asked for -------------------------
  const int STEP = n_splits * NW * TILE;
  int t = t0;
  auto compute = [&](bool first_tile) {
    if constexpr (PROBE) {  // measurement: the loads alone, no arithmetic and no merge
      u32x4 fold = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int u = 0; u < U; ++u) fold ^= kb[u] ^ vb[u];
      uint32_t w = fold.x ^ fold.y ^ fold.z ^ fold.w;
      if (w == 0x12345678u) reinterpret_cast<uint32_t*>(p.o)[0] = w;
      return;
    }
    // The token being decoded is used from LDS (where wave 0 left it) wherever the list names its
    // slot: what the pool holds there is being written by another workgroup of this launch.
    if constexpr (FRESH) {
      bool hit = slot == new_slot;
      const uint32_t hit_first = __builtin_amdgcn_readfirstlane(hit ? 1u : 0u);
      hit = valid ? hit : (hit_first != 0);  // lanes without a token hold a copy of the first lane's rows
      if (__ballot(hit)) {
        const u32x4 kn = *reinterpret_cast<const u32x4*>(sm_knew + li * 4);
        const u32x4 vn = *reinterpret_cast<const u32x4*>(sm_vnew + li * 4);
        const uint32_t hm = hit ? 1u : 0u;
#define TD_ROW_FIX(N)                   \
  if constexpr (N < U) {                \
    if (group_bcast_u32<N, LPR>(hm)) {         \
      kb[N] = kn;                       \
      vb[N] = vn;                       \
    }                                   \
  }
        TD_ROW_FIX(0) TD_ROW_FIX(1) TD_ROW_FIX(2) TD_ROW_FIX(3) TD_ROW_FIX(4) TD_ROW_FIX(5)
        TD_ROW_FIX(6) TD_ROW_FIX(7) TD_ROW_FIX(8) TD_ROW_FIX(9) TD_ROW_FIX(10) TD_ROW_FIX(11)
        TD_ROW_FIX(12) TD_ROW_FIX(13) TD_ROW_FIX(14) TD_ROW_FIX(15)
#undef TD_ROW_FIX
      }
    }

    if constexpr (QPG > 1) {
      // S = K Q^T on the matrix cores: the rows pass through the wave's own LDS into operand layout (LDS accesses
      // of one wave complete in order), in blocks of 16 tokens.  Block (c, h) holds the tokens g U + 4 c + i of
      // the lane groups g = NH g4 + h at row 4 g4 + i, which makes a lane's four scores of a block the tokens
      // whose values its group holds: the weights are the operand of the second product as they stand.
      // Piece x of row r lies at x ^ r (head_dim 64: x ^ (r / 2)), so that 16 rows read at one piece fall on
      // different banks.  (Dot products, a reduction over the row for every head and a strip of LDS for the
      // weights before: with the
      // loads ordered as below, lists of 4096 for 32/8 heads x 128 9.9 -> 9.7 us, of 200 6.9 -> 6.1.)
      constexpr int NH = 16 / LPR, NC = U / 4;
      auto place = [](int r, int x) { return r * (D * 2) + 16 * (x ^ (LPR == 16 ? r : (r >> 1) & 7)); };
      char* const kt = reinterpret_cast<char*>(sm_state[wave]);
#pragma unroll
      for (int u = 0; u < U; ++u)
        *reinterpret_cast<u32x4*>(kt + ((u >> 2) * NH + g % NH) * (32 * D) + place(4 * (g / NH) + (u & 3), li)) = kb[u];
      asm volatile("" ::: "memory");
      float sv[NC][NH][4];
      float mt = kNegBig;
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int h = 0; h < NH; ++h) {
          f32x4 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int x = 0; x < NQ; ++x)
            st = mfma_16x16x32<T>(
                *reinterpret_cast<const u32x4*>(kt + (c * NH + h) * (32 * D) + place(c16, 4 * x + g4)), qp[x], st);
#pragma unroll
          for (int i = 0; i < 4; ++i) sv[c][h][i] = st[i] * p.scale_log2;
        }
      asm volatile("" ::: "memory");
      if (ANY && p.scores) {  // copy c16 / QPG of a head writes the tokens copy, copy + COPIES, ... of the lane's
        constexpr int COPIES = 16 / QPG, NV = NC * NH * 4;
        const int copy = c16 / QPG, head = c16 % QPG;
#pragma unroll
        for (int n0 = 0; n0 < NV; n0 += COPIES) {
          float e = sv[n0 / 4 / NH][n0 / 4 % NH][n0 % 4];
#pragma unroll
          for (int x = 1; x < COPIES; ++x)
            if (n0 + x < NV) e = copy == x ? sv[(n0 + x) / 4 / NH][(n0 + x) / 4 % NH][(n0 + x) % 4] : e;
          const int n = n0 + copy;
          emit(n < NV && head < gsz, rq0 + head, t + (NH * g4 + n / 4 % NH) * U + 4 * (n / 4 / NH) + n % 4, e);
        }
      }
      const int left = c1 - t - NH * g4 * U;  // tokens from the lane's first on
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            sv[c][h][i] = h * U + 4 * c + i < left ? sv[c][h][i] : kNegBig;
            mt = fmaxf(mt, sv[c][h][i]);
          }
      const float m_new = fmaxf(mh, rows_max(mt));
      const float alpha = fast_exp2(mh - m_new);
      mh = m_new;
      float sum = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            // (by position, not by value: a NaN logit keeps its weight)
            const float pr = h * U + 4 * c + i < left ? fast_exp2(sv[c][h][i] - m_new) : 0.f;
            sv[c][h][i] = pr;
            sum += pr;
          }
      lh = fmaf(lh, alpha, sum);
      if (!first_tile) {  // later tiles: rescale what the earlier ones left (row r of group g4: head 4 g4 + r)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float f = __shfl(alpha, (4 * g4 + r) % QPG, 64);
#pragma unroll
          for (int e = 0; e < NACC; ++e) accm[e][r] *= f;
        }
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const u32x4(&v4)[4] = *reinterpret_cast<const u32x4(*)[4]>(&vb[4 * c]);
        weigh_rows<T, D, kParts>(sv[c], v4, accm);
      }
      return;
    }
    // q.k: U partial sums per lane, reduce-scattered so that the lane ends with its own token
    float part[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float a = dot2<T>(qp[0].x, kb[u].x, 0.f);
      a = dot2<T>(qp[0].y, kb[u].y, a);
      a = dot2<T>(qp[0].z, kb[u].z, a);
      part[u] = dot2<T>(qp[0].w, kb[u].w, a);
    }
    const float red = reduce_scatter_rows<U, LPR>(part, li) * p.scale_log2;  // every lane takes part: no branch around it
    if (ANY && p.scores) emit(U >= LPR || li < U, rq0, t + own, red);
    const float sv = valid ? red : kNegBig;
    const float m_new = fmaxf(m_run, rows_max(row16_max(sv)));
    const float alpha = fast_exp2(m_run - m_new);
    m_run = m_new;
    const float pr = valid ? fast_exp2(sv - m_new) : 0.f;
    // with fewer rows than lanes in a group the lanes li and li ^ 8 hold the same token: it counts once
    l_lane = l_lane * alpha + ((U >= LPR || li < U) ? pr : 0.f);
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[d] *= alpha;
#define TD_ROW_PV(N)                                        \
  if constexpr (N < U) {                                    \
    const float pu = group_bcast_f32<N, LPR>(pr);                  \
    float v0, v1, v2, v3, v4, v5, v6, v7;                   \
    unpack2<T>(vb[N].x, v0, v1);                            \
    unpack2<T>(vb[N].y, v2, v3);                            \
    unpack2<T>(vb[N].z, v4, v5);                            \
    unpack2<T>(vb[N].w, v6, v7);                            \
    acc[0] = fmaf(pu, v0, acc[0]);                          \
    acc[1] = fmaf(pu, v1, acc[1]);                          \
    acc[2] = fmaf(pu, v2, acc[2]);                          \
    acc[3] = fmaf(pu, v3, acc[3]);                          \
    acc[4] = fmaf(pu, v4, acc[4]);                          \
    acc[5] = fmaf(pu, v5, acc[5]);                          \
    acc[6] = fmaf(pu, v6, acc[6]);                          \
    acc[7] = fmaf(pu, v7, acc[7]);                          \
  }
    TD_ROW_PV(0) TD_ROW_PV(1) TD_ROW_PV(2) TD_ROW_PV(3) TD_ROW_PV(4) TD_ROW_PV(5) TD_ROW_PV(6)
    TD_ROW_PV(7) TD_ROW_PV(8) TD_ROW_PV(9) TD_ROW_PV(10) TD_ROW_PV(11) TD_ROW_PV(12)
    TD_ROW_PV(13) TD_ROW_PV(14) TD_ROW_PV(15)
#undef TD_ROW_PV
  };

  // ---- the wave's tiles: rows of the first one are asked for before anything else happens --------
  const bool live = t < c1;  // wave-uniform
  if (!prep && live) issue(t, ent);

  if constexpr (FRESH) {
    // Wave 0 rotates q and the new key while the other waves' rows are in flight (its own are asked
    // for right after: what it loaded for the rotation has arrived with its list entry, and the
    // registers are free again before its K/V rows need them) and leaves them and the new value in
    // LDS; the cache write of the new token follows after the tiles, from LDS.
    if (prep) {
      const float rcs[8] = {cos_lo.x, cos_lo.y, cos_lo.z, cos_lo.w, cos_hi.x, cos_hi.y, cos_hi.z, cos_hi.w};
      const float sgn = li < LPR / 2 ? -1.f : 1.f;  // y_lo = x_lo c - x_hi s,  y_hi = x_hi c + x_lo s
      const float rsn[8] = {sgn * sin_lo.x, sgn * sin_lo.y, sgn * sin_lo.z, sgn * sin_lo.w,
                            sgn * sin_hi.x, sgn * sin_hi.y, sgn * sin_hi.z, sgn * sin_hi.w};
      // rotate-half RoPE of 8 elements per lane; the partner dimension (+- D/2) sits LPR/2 lanes away
      auto rotate = [&](uint32_t(&w)[4]) {
        float x[8], y[8];
#pragma unroll
        for (int c = 0; c < 4; ++c) unpack2<T>(w[c], x[2 * c], x[2 * c + 1]);
#pragma unroll
        for (int d = 0; d < 8; ++d)
          y[d] = x[d] * rcs[d] + (LPR == 16 ? dpp_move<0x128>(x[d]) : lane_xor16<4>(x[d])) * rsn[d];
#pragma unroll
        for (int c = 0; c < 4; ++c) w[c] = pack2<T>(y[2 * c], y[2 * c + 1]);
      };
      uint32_t knew[4] = {kn_raw.x, kn_raw.y, kn_raw.z, kn_raw.w};
      rotate(knew);
      if (g == 0) {
        *reinterpret_cast<u32x4*>(sm_knew + li * 4) = u32x4{knew[0], knew[1], knew[2], knew[3]};
        *reinterpret_cast<u32x4*>(sm_vnew + li * 4) = vn_raw;
      }
#pragma unroll
      for (int x = 0; x < QX; ++x) {
        uint32_t qj[4] = {q_raw[x].x, q_raw[x].y, q_raw[x].z, q_raw[x].w};
        rotate(qj);
        const int j = g + x * GR;
        if (j < gsz) *reinterpret_cast<u32x4*>(sm_fresh + j * (D / 2) + li * 4) = u32x4{qj[0], qj[1], qj[2], qj[3]};
      }
      if (live) issue(t, ent);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the LDS writes have landed
    }
    // a bare barrier: the fence of __syncthreads would wait for the rows in flight
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // every wave, the first included: registers that no global load of either branch is still
    // writing to, so that the wait the compiler puts in front of this read is for LDS only
    load_q([&](int j, int c) { return *reinterpret_cast<const u32x4*>(sm_fresh + j * (D / 2) + c * 4); });
  }

  // the first tile apart from the loop: its rows were asked for above, and the loop then keeps no
  // K/V registers alive from one pass to the next
  if (live) {
    compute(true);
    for (t += STEP; t < c1; t += STEP) {
      issue(t, fetch_entry(t));
      compute(false);
    }
  }
  if constexpr (FRESH) {
    // One workgroup per KV head writes the new token into the cache, from the copy in LDS and after
    // the tiles: a store in front of them would have the tiles' first register writes wait for it.
    // Nobody in this launch reads that slot from memory.
    if (prep && split == 0 && (QPG > 1 || hrow == kv_head * p.q_per_kv) && g == 0) {
      const uint32_t ns = new_slot > p.max_slot ? p.max_slot : new_slot;
      char* dst = reinterpret_cast<char*>(const_cast<void*>(p.kv)) + slot_offset(ns) + head_byte_off;
      *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(sm_knew + li * 4);
      *reinterpret_cast<u32x4*>(dst + p.v_offset * 2) = *reinterpret_cast<const u32x4*>(sm_vnew + li * 4);
    }
  }

  if constexpr (PROBE) return;
  auto state = [&](int w, int j, int d) -> float* { return &sm_state[w][j * D + d]; };
  __shared__ float sm_ml[NW][QPG][2];
  if constexpr (QPG > 1) {
    // the matrix product already summed the lane groups: the lanes of group g4 hold heads 4 g4 .. 4 g4 + 3
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int head = 4 * g4 + r;
      if (head < QPG) {
#pragma unroll
        for (int e = 0; e < NACC; e += 4)
          *reinterpret_cast<f32x4*>(state(wave, head, li * 8 + (LPR == 16 ? e : 4 * (c16 >> 3)))) =
              f32x4{accm[e][r], accm[e + 1][r], accm[e + 2][r], accm[e + 3][r]} * (1.f / kWeightScale<T, kParts>);
      }
    }
    const float lw = rows_sum(lh);
    if (lane < QPG) {
      sm_ml[wave][lane][0] = mh;
      sm_ml[wave][lane][1] = lw;
    }
  } else {
    // ---- the lane groups of the wave: the maximum is shared, so the sums simply add --------------
    // reduce-scatter over the groups: lane (g, li) ends with dimensions li 8 + g4 2 + {0, 1} (head_dim 128),
    // or, the two halves of a 16-lane row being groups of their own, with the one of them that is c16 / 8
    float r0, r1;
    {
      float x, y, h[4];
#pragma unroll
      for (int i2 = 0; i2 < 4; ++i2) {
        swap32(acc[i2], acc[i2 + 4], x, y);
        h[i2] = x + y;  // lower half: dimension i2, upper half: dimension i2 + 4
      }
      swap16(h[0], h[2], x, y);
      r0 = x + y;
      swap16(h[1], h[3], x, y);
      r1 = x + y;
    }
    const float l_w = rows_sum(group_sum<16>(l_lane));
    if constexpr (LPR == 16) {
      *reinterpret_cast<f32x2*>(state(wave, 0, li * 8 + g4 * 2)) = f32x2{r0, r1};
    } else {
      const bool odd = c16 >= 8;
      *state(wave, 0, li * 8 + g4 * 2 + (c16 >> 3)) = (odd ? r1 : r0) + dpp_move<0x128>(odd ? r0 : r1);
    }
    if (lane == 0) {
      sm_ml[wave][0][0] = m_run;
      sm_ml[wave][0][1] = l_w;
    }
  }
  // ---- the waves of the workgroup meet in LDS; wave j carries on alone with the heads j, j + NW ------
  constexpr int HW = (QPG + NW - 1) / NW;  // heads of a wave
  uint32_t* out[HW];                       // where they go, before the barrier
  float* lse_out[HW];
  int64_t part[HW];
#pragma unroll
  for (int x = 0; x < HW; ++x) {
    const int j = wave + x * NW;
    out[x] = reinterpret_cast<uint32_t*>(p.o) + ((int64_t)b * p.num_qo_heads + rq0 + j) * (D / 2) + lane;
    lse_out[x] = p.lse ? p.lse + (int64_t)b * p.num_qo_heads + rq0 + j : nullptr;
    part[x] = ((int64_t)b * p.vheads + hrow * QPG + j) * p.max_splits;
  }
  int32_t* const tickets = p.ws_cnt + (((int64_t)b * gridDim.x + hrow) * QPG + wave) * p.ticket_stride;
  __syncthreads();
#pragma unroll
  for (int x = 0; x < HW; ++x) {
    const int j = wave + x * NW;
    if (j >= gsz) break;
    float M = kNegBig;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, sm_ml[w][j][0]);
    float L = 0.f, o0 = 0.f, o1 = 0.f;  // this lane: dimensions 2 lane, 2 lane + 1
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = fast_exp2(sm_ml[w][j][0] - M);
      L = fmaf(sm_ml[w][j][1], f, L);
      const f32x2 v = *reinterpret_cast<const f32x2*>(state(w, j, 2 * (lane & (D / 2 - 1))));
      o0 = fmaf(v.x, f, o0);
      o1 = fmaf(v.y, f, o1);
    }
    publish_head<T, D>(p, lane, n_splits, part[x] + split, out[x], lse_out[x], o0, o1, M, L);
  }
  // (without a merge here a second launch, merge_partials_kernel, reduces the partials)
  if (n_splits == 1 || !p.fused_merge || wave >= gsz) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  int tk = 0;  // lane x: the ticket of head wave + x NW (eight heads by four waves: 28/4 heads, lists of 1024 8.7 -> 7.6 us)
  if (lane < HW && wave + lane * NW < gsz)
    tk = __hip_atomic_fetch_add(tickets + (HW > 1 ? lane * NW * p.ticket_stride : 0), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (int x = 0; x < HW; ++x) {
    const int j = wave + x * NW;
    if (j < gsz && __builtin_amdgcn_readlane(tk, x) == n_splits - 1)
      merge_head<T, D>(p, lane, n_splits, part[x], tickets + x * NW * p.ticket_stride, out[x], lse_out[x]);
  }
}

// Shapes of the sparse-layer kernel: waves per workgroup x K (and V) rows per lane; with shared
// KV rows (2, 4 or 8 query heads per list walk) 8 rows per lane.
static bool sparse_shape_supported(int nw, int rows, int qpg = 1) {
  if (qpg == 1) return (nw == 4 || nw == 8) && (rows == 8 || rows == 16);
  return (qpg == 2 || qpg == 4 || qpg == 8) && (nw == 4 || nw == 8) && rows == 8;
}

// `wide`: 64-bit row offsets and pages of any size (8 rows per lane only)
template <typename T>
static int launch_sparse(const DecodeParams& p, int head_dim, int nw, int rows, bool probe, bool wide, dim3 grid,
                         hipStream_t st) {
  const bool any = p.list_shift > 0 || p.scores;
#define TD_SPARSE_CASE(N_, D_, ANY_)                                                                               \
  if (nw == N_ && rows == 8 && head_dim == D_ && any == ANY_ && !wide && !probe && (D_ == 64 || ANY_)) {           \
    if (p.fresh_k)                                                                                                 \
      hipLaunchKernelGGL((sparse_attn_kernel<T, N_, 8, true, false, 1, false, D_, ANY_>), grid, dim3(N_ * 64), 0,  \
                         st, p);                                                                                   \
    else                                                                                                           \
      hipLaunchKernelGGL((sparse_attn_kernel<T, N_, 8, false, false, 1, false, D_, ANY_>), grid, dim3(N_ * 64), 0, \
                         st, p);                                                                                   \
    return TD_OK;                                                                                                  \
  }
  TD_SPARSE_CASE(4, 64, false)
  TD_SPARSE_CASE(8, 64, false)
  TD_SPARSE_CASE(4, 64, true)
  TD_SPARSE_CASE(8, 64, true)
  TD_SPARSE_CASE(4, 128, true)
  TD_SPARSE_CASE(8, 128, true)
#undef TD_SPARSE_CASE
#define TD_SPARSE_CASE(N_, U_)                                                                   \
  if (nw == N_ && rows == U_ && !wide) {                                                         \
    if (probe)                                                                                   \
      hipLaunchKernelGGL((sparse_attn_kernel<T, N_, U_, false, true>), grid, dim3(N_ * 64), 0,   \
                         st, p);                                                                 \
    else if (p.fresh_k)                                                                          \
      hipLaunchKernelGGL((sparse_attn_kernel<T, N_, U_, true>), grid, dim3(N_ * 64), 0, st, p);  \
    else                                                                                         \
      hipLaunchKernelGGL((sparse_attn_kernel<T, N_, U_, false>), grid, dim3(N_ * 64), 0, st, p); \
    return TD_OK;                                                                                \
  }
  TD_SPARSE_CASE(8, 8)
  TD_SPARSE_CASE(4, 8)
  TD_SPARSE_CASE(4, 16)
  TD_SPARSE_CASE(8, 16)
#undef TD_SPARSE_CASE
#define TD_SPARSE_CASE(N_)                                                                          \
  if (nw == N_ && rows == 8 && wide) {                                                              \
    if (probe)                                                                                      \
      hipLaunchKernelGGL((sparse_attn_kernel<T, N_, 8, false, true, 1, true>), grid, dim3(N_ * 64), \
                         0, st, p);                                                                 \
    else if (p.fresh_k)                                                                             \
      hipLaunchKernelGGL((sparse_attn_kernel<T, N_, 8, true, false, 1, true>), grid, dim3(N_ * 64), \
                         0, st, p);                                                                 \
    else                                                                                            \
      hipLaunchKernelGGL((sparse_attn_kernel<T, N_, 8, false, false, 1, true>), grid,               \
                         dim3(N_ * 64), 0, st, p);                                                  \
    return TD_OK;                                                                                   \
  }
  TD_SPARSE_CASE(8)
  TD_SPARSE_CASE(4)
#undef TD_SPARSE_CASE
  return fail(TD_ERR_UNSUPPORTED, "sparse decode attention: no kernel for %d waves x %d rows%s", nw, rows,
              wide ? " with 64-bit offsets" : "");
}

// shared KV rows: QPG query heads per list walk
template <typename T>
static int launch_sparse_shared(const DecodeParams& p, int head_dim, int nw, int qpg, bool wide, dim3 grid,
                                hipStream_t st) {
  const bool any = p.list_shift > 0 || p.scores;
#define TD_SPARSE_CASE(Q_, W_, D_, ANY_)                                                                    \
  if (qpg == Q_ && wide == W_ && head_dim == D_ && any == ANY_) {                                           \
    if (nw == 4 && p.fresh_k)                                                                               \
      hipLaunchKernelGGL((sparse_attn_kernel<T, 4, 8, true, false, Q_, W_, D_, ANY_>), grid, dim3(256), 0,  \
                         st, p);                                                                            \
    else if (nw == 4)                                                                                       \
      hipLaunchKernelGGL((sparse_attn_kernel<T, 4, 8, false, false, Q_, W_, D_, ANY_>), grid, dim3(256), 0, \
                         st, p);                                                                            \
    else if (p.fresh_k)                                                                                     \
      hipLaunchKernelGGL((sparse_attn_kernel<T, 8, 8, true, false, Q_, W_, D_, ANY_>), grid, dim3(512), 0,  \
                         st, p);                                                                            \
    else                                                                                                    \
      hipLaunchKernelGGL((sparse_attn_kernel<T, 8, 8, false, false, Q_, W_, D_, ANY_>), grid, dim3(512), 0, \
                         st, p);                                                                            \
    return TD_OK;                                                                                           \
  }
  TD_SPARSE_CASE(2, false, 128, false)
  TD_SPARSE_CASE(4, false, 128, false)
  TD_SPARSE_CASE(8, false, 128, false)
  TD_SPARSE_CASE(2, true, 128, false)
  TD_SPARSE_CASE(4, true, 128, false)
  TD_SPARSE_CASE(8, true, 128, false)
  TD_SPARSE_CASE(2, false, 64, false)
  TD_SPARSE_CASE(4, false, 64, false)
  TD_SPARSE_CASE(8, false, 64, false)
  TD_SPARSE_CASE(2, false, 128, true)
  TD_SPARSE_CASE(4, false, 128, true)
  TD_SPARSE_CASE(8, false, 128, true)
  TD_SPARSE_CASE(2, false, 64, true)
  TD_SPARSE_CASE(4, false, 64, true)
  TD_SPARSE_CASE(8, false, 64, true)
#undef TD_SPARSE_CASE
  return fail(TD_ERR_UNSUPPORTED,
              "sparse decode attention: no kernel for %d waves with %d query heads per shared row", nw, qpg);
}

// Launches the sparse-layer kernel (and, when the plan asks for it, the second-launch merge);
// defined once per element type (and once more for shared KV rows) in sparse_attn_*.hip.
int launch_sparse_f16(const DecodeParams& p, int head_dim, int nw, int rows, bool probe, bool wide, bool merge_kernel,
                      dim3 grid, hipStream_t st);
int launch_sparse_bf16(const DecodeParams& p, int head_dim, int nw, int rows, bool probe, bool wide, bool merge_kernel,
                       dim3 grid, hipStream_t st);
int launch_sparse_shared_f16(const DecodeParams& p, int head_dim, int nw, int qpg, bool wide, bool merge_kernel, dim3 grid,
                             hipStream_t st);
int launch_sparse_shared_bf16(const DecodeParams& p, int head_dim, int nw, int qpg, bool wide, bool merge_kernel, dim3 grid,
                              hipStream_t st);

}  // namespace tidal
