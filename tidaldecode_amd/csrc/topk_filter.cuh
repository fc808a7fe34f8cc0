// Top-k of a row by one workgroup that touches every element once (included by topk.hip).
//
// What bounds a selection out of 10^4 .. 10^5 scores is not their 40 .. 400 KB but the instructions
// spent per score on the one compute unit that holds the row: an instruction per element costs a
// 1024-thread workgroup 16 cycles, 0.5 us per row of 64K.  So the radix work is done on few elements:
//
//   1. a sample of 4 elements per thread, spread evenly over the row, gives a threshold that the k-th
//      largest element exceeds almost surely (5 standard deviations of the sample's count);
//   2. one pass over the row (loads in flight from the start) keeps the positions of what is not below
//      it, about 1.1 .. 1.4 k elements, in LDS: two instructions per element, some more per survivor;
//   3. the radix select of the k-th largest runs on the survivors (exact: fewer survivors than k start
//      again with a lower threshold; more than the list holds -- rows of few distinct values -- once more
//      with the sample's value at that rank as the threshold, equal scores being counted and not listed;
//      should even what lies above it be too much, the row is left to select_slice);
//   4. the selected positions go into a bitmap in LDS, whose prefix counts give every one its place
//      in position order, whatever order the survivors were listed in.
//
// Rows of up to 4 elements per thread are their own sample: the radix select on it is the result.
//
// Measured on one MI355X (fp32, bound and page table given, launches of a graph, us; in brackets the
// kernel that had these rows before: every workgroup histograms the whole row, its scores in registers
// up to 64K of them, and up to eight workgroups share the emission):
//   32 x 777 -> 256     4.6 (7.3)     256 x 14000 -> 1024  11.1 (15.8)
//   32 x 4096 -> 256    6.7 (8.3)     256 x 63000 -> 1024  23.3 (58.6)
//   512 x 8192 -> 512    9.7 (19.5)   256 x 65537 -> 1024  24.4 (120)
//   32 x 32769 -> 2048  12.6 (15.9)   8 x 102392 -> 4096   19.5 (28.6: three launches that share a row)
// Rows of equal scores, and of two values by halves, through the ties' threshold (before that kernel; a selection
// by one workgroup out of the whole row, whose additions queue up at one address, took 130 and 630 for the second
// and the last): 32 x 4096 -> 256 21.0, 17.2 (20.5, 14.2); 32 x 32769 -> 2048 27.4, 24.8 (98.8, 54.4); 256 x 63000
// -> 1024 45.6, 42.5 (202, 120); 8 x 102392 -> 4096 40.9, 36.3 (211, 123).  Having that way out costs other rows
// 0.1 - 0.3 us.
// What is left is a chain: two trips to memory (sample, survivors' values), two radix levels of about
// 1 us and the bitmap's 0.8; 256 rows of 63000 also read 64 MB at 2.8 TB/s.
// The results are those of every other variant: the k largest, ties to the lower position, in
// position order.
#pragma once

namespace tidal {

constexpr uint32_t kKeyNegInf = 0x007fffffu, kKeyPosInf = 0xff800000u;
constexpr uint32_t kMaxSpan = 0xff800000u;  // no two keys of scores lie further apart
__device__ __forceinline__ float key_to_float(uint32_t key) {
  return __builtin_bit_cast(float, (key & 0x80000000u) ? key & 0x7fffffffu : ~key);
}
__device__ __forceinline__ int bit_count(uint32_t x) { return x ? 32 - __builtin_clz(x) : 0; }

// A row read four elements at a time.  The descriptor starts at the dword that holds element 0, so
// that every load is dword aligned; `shift` elements (16-bit types: 0 or 1) lie in front of the row.
// Vector i holds the elements 4 i - shift .. 4 i + 3 - shift; dwords past the end read as 0.
template <typename T>
struct RowVectors {
  typedef typename std::conditional<std::is_same<T, F32>::value, u32x4, u32x2>::type vec;
  __amdgpu_buffer_rsrc_t rsrc;
  int shift;
  __device__ __forceinline__ RowVectors(const void* row, int len) {
    if constexpr (std::is_same<T, F32>::value) {
      shift = 0;
      rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(row), 0, len * 4, 0x00020000);
    } else {
      const uint64_t at = reinterpret_cast<uint64_t>(row);
      shift = (int)((at >> 1) & 1);
      rsrc = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(at & ~3ull), 0,
                                               ((len + shift) * 2 + 3) & ~3, 0x00020000);
    }
  }
  // vector lane_vec + uniform_vec
  __device__ __forceinline__ vec load(int lane_vec, int uniform_vec) const {
    if constexpr (std::is_same<T, F32>::value)
      return __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane_vec * 16, uniform_vec * 16, 0));
    else
      return __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b64(rsrc, lane_vec * 8, uniform_vec * 8, 0));
  }
  __device__ static __forceinline__ float element(const vec& v, int c) {
    if constexpr (std::is_same<T, F32>::value)
      return __builtin_bit_cast(float, (uint32_t)v[c]);
    else
      return to_float<T>((uint16_t)((uint32_t)v[c >> 1] >> (16 * (c & 1))));
  }
};

// bit i of the result: element i of the 16 in v[0 .. 3] is not below `floor` (a NaN is not below
// anything).  Two instructions per element: the comparison's mask is shifted in as a carry.  Four comparisons
// write four scalar pairs before the first is read: a mask needs two wait states between the vector
// instruction that writes it and the one that takes it as carry, and the compiler inserts none inside asm.
template <typename T>
__device__ __forceinline__ uint32_t reach16(const typename RowVectors<T>::vec* v, float floor) {
  uint32_t mask = 0;
#pragma unroll
  for (int i = 3; i >= 0; --i) {
    uint64_t m0, m1, m2, m3;
    asm("v_cmp_nlt_f32 %4, %8, %9\n\tv_cmp_nlt_f32 %3, %7, %9\n\t"
        "v_cmp_nlt_f32 %2, %6, %9\n\tv_cmp_nlt_f32 %1, %5, %9\n\t"
        "v_addc_co_u32 %0, %4, %0, %0, %4\n\tv_addc_co_u32 %0, %3, %0, %0, %3\n\t"
        "v_addc_co_u32 %0, %2, %0, %0, %2\n\tv_addc_co_u32 %0, %1, %0, %0, %1"
        : "+v"(mask), "=&s"(m0), "=&s"(m1), "=&s"(m2), "=&s"(m3)
        : "v"(RowVectors<T>::element(v[i], 0)), "v"(RowVectors<T>::element(v[i], 1)),
          "v"(RowVectors<T>::element(v[i], 2)), "v"(RowVectors<T>::element(v[i], 3)), "v"(floor));
  }
  return mask;
}

constexpr int kMidLen = 10240;   // longest rows of 512 threads
constexpr int kFilterRank = 64;  // members of the threshold bin that are ranked in the lanes of a wave

template <int NT, int CAP, int MAXLEN>
struct FilterLds {
  typedef typename std::conditional<(MAXLEN <= 65536), uint16_t, uint32_t>::type pos_t;
  uint32_t hist[4 * NT];         // zero between the radix levels
  pos_t pos[CAP];                // survivors
  uint32_t bits[MAXLEN / 32];    // selected positions
  uint16_t before[MAXLEN / 32];  // set bits in front of the word
  uint32_t mem[kFilterRank];
  uint32_t wa[16], wb[16];
  uint32_t sh[4];
  uint32_t n_cand, n_mem;
};

// page of position i for pages of any size: the quotient from a multiplication is at most one short
__device__ __forceinline__ int page_of(const TopkParams& p, int i) {
  int page = (int)__umulhi((uint32_t)i, p.page_magic);
  if (i - page * p.page_size >= p.page_size) ++page;
  return page;
}

// sums of the first `wave` and of all NW entries of arr
template <int NW>
__device__ __forceinline__ void sums_before(const uint32_t* arr, int wave, int lane, uint32_t& before, uint32_t& all) {
  const uint32_t v = row_prefix_sum((lane & 15) < NW ? arr[lane & (NW - 1)] : 0u);
  all = __builtin_amdgcn_readlane(v, NW - 1);
  before = wave ? __builtin_amdgcn_readlane(v, wave - 1) : 0u;
}

// CAP: survivors the list holds; CAP >= MAXLEN: any row fits.
// kMidLen: two workgroups of a compute unit (four waves a SIMD) are worth the 20 bytes that the registers of the
// ties' way spill: 512 fp32 rows of 8193 -> 512 10.4 us, with one workgroup 14.4.
template <typename T, int NT, int VPT, int CAP, int MAXLEN>
__global__ __launch_bounds__(NT, MAXLEN == kMidLen ? 4 : 1) void topk_filter_kernel(const TopkParams p) {
  typedef typename ElemOf<T>::type elem_t;
  typedef typename RowVectors<T>::vec vec;
  typedef FilterLds<NT, CAP, MAXLEN> Lds;
  constexpr int NW = NT / 64, CPT = CAP / NT, CHUNK = 4 * NT * VPT;
  constexpr int kBits = NT == 1024 ? 12 : (NT == 512 ? 11 : 10);  // log2 of the bins
  constexpr bool kFits = MAXLEN <= CAP;                 // the list holds any row: no way out needed
  constexpr bool kTied = !kFits || MAXLEN > 8192;       // many survivors: the ties' threshold
  constexpr uint32_t kMost = kFits ? 4096u : CAP;       // (a list that long is rows of few distinct values)
  constexpr bool kSampled = MAXLEN > 4 * NT;            // rows may be longer than the sample
  constexpr bool kTieRank = !std::is_same<T, F32>::value;
  static_assert(CPT >= 4 && 4 * NT == 1 << kBits && (VPT == 4 || VPT == 8), "shapes");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = blockIdx.x;
  const int len = row_len(p, row), k = row_k(p, len);
  const elem_t* vals = reinterpret_cast<const elem_t*>(p.values) + (int64_t)row * p.values_stride;
  const RowVectors<T> rv(vals, len);
  const int shift = rv.shift;

  __shared__ union {
    Lds f;
    typename std::conditional<kFits, uint32_t, SliceLds>::type slice;
  } lds;
  Lds& L = lds.f;

  // ---- the sample, then the row: everything in flight ------------------------------------------
  const int nvec = (len + shift + 3) >> 2;
  const bool whole = !kSampled || nvec <= NT;  // the sample is the row
  // four threads share 16 consecutive elements: single vectors would pull a 128-byte line each
  const int svec = whole ? tid : (int)((uint32_t)(tid >> 2) * (uint32_t)(nvec >> 2) / (uint32_t)(NT / 4)) * 4 + (tid & 3);
  const vec sample = rv.load(svec, 0);
  vec v[kSampled ? VPT : 4];
  auto load_group = [&](int chunk, int g) {
#pragma unroll
    for (int j = 4 * g; j < 4 * g + 4; ++j) v[j] = rv.load(tid, (chunk * VPT + j) * NT);
  };
  if (!whole) {
#pragma unroll
    for (int g = 0; g < VPT / 4; ++g) load_group(0, g);
  }

  float bound = __builtin_nanf("");
  if (p.row_bound) bound = p.row_bound[row];
  const bool bounded = __builtin_fabsf(bound) < __builtin_inff();
  reinterpret_cast<uint4*>(L.hist)[tid] = make_uint4(0, 0, 0, 0);
  const int n_words = (len + 31) >> 5;
  for (int i = tid; i < n_words; i += NT) L.bits[i] = 0;
  if (tid == 0) L.n_cand = L.n_mem = 0;

  // ---- 1. the sample's distances below a reference: the caller's bound or the sample's maximum ----
  uint32_t sx[4], kmax = 0u;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    sx[c] = KeyTraits<F32>::key(RowVectors<T>::element(sample, c));
    if ((uint32_t)(4 * svec + c - shift) < (uint32_t)len) kmax = sx[c] > kmax ? sx[c] : kmax;
  }
  if (bounded) {
    kmax = KeyTraits<F32>::key(bound);
    // 16-bit scores may have been rounded up past a bound formed in fp32: one bf16 step of room
    if constexpr (!std::is_same<T, F32>::value) kmax += 0x10000u;
  } else {
    kmax = (uint32_t)wave_max_i32((int32_t)(kmax ^ 0x80000000u));
    if (lane == 0) L.wb[wave] = kmax;
    __syncthreads();
    kmax = (uint32_t)wave_max_i32((int32_t)L.wb[lane & (NW - 1)]) ^ 0x80000000u;
  }
  kmax = __builtin_amdgcn_readfirstlane(kmax);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t d = sx[c] < kmax ? kmax - sx[c] : 0u;
    sx[c] = (uint32_t)(4 * svec + c - shift) < (uint32_t)len ? d : kNoElement;
  }
  uint32_t rank = (uint32_t)k;
  if (!whole) {
    const float mu = (float)k * (float)(4 * NT) / (float)len;
    rank = (uint32_t)(mu + 5.f * __builtin_sqrtf(mu) + 5.f);
  }
  __syncthreads();  // hist, bits and the counters are zero

  // ---- radix select: the krem-th smallest of what each() hands out, as the krem-th smallest of the
  // n_in ones in [lo, lo + 2^s): at most kFilterRank, or all equal (s == 0).  The window [lo, lo + last]
  // comes first, what lies beyond it only if fewer than krem lie inside.  False: fewer than krem in all.
  // exact: until s == 0.  crowded: lanes with equal bins add together, for equal scores queue up at one
  // address (from the second level on by itself: a bin of more than kFilterRank members was chosen).
  uint32_t lo, s, krem, n_in;
  auto narrow = [&](uint32_t last, bool crowded, bool exact, auto each) -> bool {
    auto shift_of = [](uint32_t span) {
      const int b = bit_count(span) - kBits;
      return b > 0 ? (uint32_t)b : 0u;
    };
    lo = 0u;
    s = shift_of(last);
    for (;;) {
      last |= (1u << s) - 1u;  // whole bins: what lies in the last one is counted with it, also beyond the window
      if (__builtin_expect(!crowded, 1)) {
        each([&](uint32_t x) {
          const uint32_t d = x - lo;
          if (d <= last) atomicAdd(&L.hist[d >> s], 1u);
        });
      } else {
        each([&](uint32_t x) {
          const uint32_t d = x - lo, bin = d >> s;
          uint64_t left = __ballot(d <= last);
          while (left) {  // worth a turn for eight lanes and more
            const int one = __builtin_ctzll(left);
            const uint64_t same = __ballot(bin == (uint32_t)__builtin_amdgcn_readlane(bin, one)) & left;
            if (__popcll(same) < 8) break;
            if (lane == one) atomicAdd(&L.hist[bin], (uint32_t)__popcll(same));
            left &= ~same;
          }
          if ((left >> lane) & 1u) atomicAdd(&L.hist[bin], 1u);
        });
      }
      __syncthreads();
      uint4* h4 = reinterpret_cast<uint4*>(L.hist) + tid;
      const uint4 a = *h4;
      *h4 = make_uint4(0, 0, 0, 0);
      const uint32_t local = (a.x + a.y) + (a.z + a.w);
      const uint32_t incl = wave_prefix_sum_dpp(local, lane);
      if (lane == 63) L.wa[wave] = incl;
      __syncthreads();
      uint32_t first, total;
      sums_before<NW>(L.wa, wave, lane, first, total);
      first += incl - local;
      if (first < krem && krem <= first + local) {  // one thread of the workgroup, if any
        const uint32_t b1 = first + a.x, b2 = b1 + a.y, b3 = b2 + a.z;
        const int i = (krem > b1 ? 1 : 0) + (krem > b2 ? 1 : 0) + (krem > b3 ? 1 : 0);
        L.sh[0] = (uint32_t)(4 * tid + i);
        L.sh[1] = krem - (i == 0 ? first : (i == 1 ? b1 : (i == 2 ? b2 : b3)));
        L.sh[2] = i == 0 ? a.x : (i == 1 ? a.y : (i == 2 ? a.z : a.w));
      }
      __syncthreads();
      if (krem <= total) {
        lo += __builtin_amdgcn_readfirstlane(L.sh[0]) << s;
        krem = __builtin_amdgcn_readfirstlane(L.sh[1]);
        n_in = __builtin_amdgcn_readfirstlane(L.sh[2]);
        if (s == 0u || (n_in <= (uint32_t)kFilterRank && !exact)) return true;
        crowded = true;
        last = (1u << s) - 1u;
      } else {
        if (last >= kMaxSpan - lo) return false;
        krem -= total;
        lo += last + 1u;
        last = kMaxSpan - lo;
      }
      s = shift_of(last);
    }
  };
  auto each_sample = [&](auto f) {
#pragma unroll
    for (int c = 0; c < 4; ++c) f(sx[c]);
  };
  constexpr uint32_t kFirst = (1u << 29) - 1u;  // 64 binades below the reference first
  // (a wave's own affair: eight lanes that sampled the same score)
  const bool alike = __popcll(__ballot(sx[0] == (uint32_t)__builtin_amdgcn_readfirstlane(sx[0]))) >= 8;

  // What is selected from, n slots: x (kNoElement: empty) and position.  The row itself if it is its
  // own sample, else the survivors.
  uint32_t x[CPT], krem0;
  int32_t pos[CPT];
  int n;
  uint32_t C = 0;
  auto each_slot = [&](auto f) {  // f(slot)
#pragma unroll
    for (int u4 = 0; u4 < CPT; u4 += 4) {
      if (u4 * NT < n) {  // uniform
#pragma unroll
        for (int u = u4; u < u4 + 4; ++u) f(u);
      }
    }
  };
  const int wpt = (n_words + NT - 1) / NT;
  // before[w] = set bits in front of word w (of more than 16 bits hold: 65535); their number
  auto count_words = [&]() -> uint32_t {
    __syncthreads();
    uint32_t local = 0;
    for (int i = 0; i < wpt; ++i) {
      const int w = tid * wpt + i;
      local += w < n_words ? __popc(L.bits[w]) : 0u;
    }
    const uint32_t incl = wave_prefix_sum_dpp(local, lane);
    if (lane == 63) L.wa[wave] = incl;
    __syncthreads();
    uint32_t run, total;
    sums_before<NW>(L.wa, wave, lane, run, total);
    run += incl - local;
    for (int i = 0; i < wpt; ++i) {
      const int w = tid * wpt + i;
      if (w < n_words) {
        L.before[w] = (uint16_t)(run < 65535u ? run : 65535u);
        run += __popc(L.bits[w]);
      }
    }
    __syncthreads();
    return total;
  };
  if (whole) {
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      x[u] = u < 4 ? sx[u & 3] : kNoElement;
      const int at = 4 * svec + (u & 3) - shift;
      pos[u] = at < 0 ? 0 : (at < len ? at : len - 1);
    }
    n = 4 * NT;
    krem = krem0 = (uint32_t)k;
    narrow(kFirst, alike, false, each_sample);
  } else if constexpr (kSampled) {
    // ---- 2. the survivors: what is not below the far edge of the bin that holds rank `rank` ---------
    // above: a second time, what is above the sample's value at that rank
    uint32_t kbase, tie = 0u;
    bool above = false, equal = false;
    for (;;) {
      kbase = 0u;
      krem = rank;
      if (narrow(kFirst, above || alike, above, each_sample)) {
        const uint32_t edge = lo + ((1u << s) - 1u);
        kbase = kmax > edge ? kmax - edge : 0u;
        equal = n_in > (uint32_t)kFilterRank;
      }
      if (__builtin_expect(above, 0)) {
        tie = kbase;
        C = CAP + 1u;
        if (tie < kKeyNegInf || tie >= kKeyPosInf) break;
        ++kbase;
      }
      kbase = kbase < kKeyNegInf ? kKeyNegInf : (kbase > kKeyPosInf ? kKeyPosInf : kbase);
      const float floor_f = key_to_float(kbase);
      for (int chunk = 0; chunk * CHUNK < len + shift; ++chunk) {
#pragma unroll
        for (int g = 0; g < VPT / 4; ++g) {
          const int first = 4 * ((chunk * VPT + 4 * g) * NT) - shift;  // position of the group's first element
          if (first < len) {
            uint32_t mask = reach16<T>(v + 4 * g, floor_f);
            if (first < 0 || first + 16 * NT > len) {  // elements outside the row
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                const int at = first + 4 * (j * NT + tid), room = len - at;
                const uint32_t ok = room >= 4 ? 15u : (room > 0 ? (1u << room) - 1u : 0u);
                mask &= ~(15u << (4 * j)) | ((at < 0 ? ok & 14u : ok) << (4 * j));
              }
            }
            if (__ballot(mask != 0u)) {
              const uint32_t mine = __popc(mask);
              const uint32_t incl = wave_prefix_sum_dpp(mine, lane);
              const uint32_t all = __builtin_amdgcn_readlane(incl, 63);
              uint32_t at = 0;
              if (lane == 0) at = atomicAdd(&L.n_cand, all);
              at = __builtin_amdgcn_readfirstlane(at);
              if (kFits || at + all <= (uint32_t)CAP) {  // else counted, not listed
                at += incl - mine;
                while (mask) {
                  const int i = __builtin_ctz(mask);
                  mask &= mask - 1u;
                  L.pos[at++] = (typename Lds::pos_t)(first + 4 * tid + (i & 12) * NT + (i & 3));
                }
              }
            }
          }
          if ((chunk + 1) * CHUNK < len + shift) load_group(chunk + 1, g);
        }
      }
      __syncthreads();
      C = __builtin_amdgcn_readfirstlane(L.n_cand);
      if (above || (C >= (uint32_t)k && (!kTied || C <= kMost))) break;
      if (C >= (uint32_t)k)
        above = true;
      else
        rank = 2u * rank + 64u;  // an unlucky sample: the k-th largest lies below the floor
#pragma unroll
      for (int g = 0; g < VPT / 4; ++g) load_group(0, g);
      __syncthreads();
      if (tid == 0) L.n_cand = 0;  // (added to again behind the barriers of the next level)
    }
    if constexpr (kTied) {
      if (__builtin_expect(above && C < (uint32_t)k, 0)) {
        // The list holds what is above the ties, and the ties make up the rest: the first of them by position.
        const float tie_f = key_to_float(tie);
        for (int vec0 = 0; vec0 < nvec; vec0 += 4 * NT) {
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = rv.load(tid, vec0 + j * NT);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int at = 4 * (vec0 + j * NT + tid) - shift;
            uint32_t four = 0;
#pragma unroll
            for (int c = 0; c < 4; ++c)
              four |= RowVectors<T>::element(v[j], c) == tie_f && (uint32_t)(at + c) < (uint32_t)len ? 1u << c : 0u;
            if (four) {
              const int word = at < 0 ? 0 : at >> 5, bit = at & 31;
              if (at < 0)
                atomicOr(&L.bits[0], four >> 1);
              else
                atomicOr(&L.bits[word], four << bit);
              if (bit > 28 && at >= 0 && (four >> (32 - bit))) atomicOr(&L.bits[word + 1], four >> (32 - bit));
            }
          }
        }
        const uint32_t wanted = (uint32_t)k - C;
        if (count_words() >= wanted) {
          for (int w = tid; w < n_words; w += NT) {
            uint32_t word = L.bits[w];
            const uint32_t first = L.before[w];
            if (first + __popc(word) > wanted) {
              const int keep = first < wanted ? (int)(wanted - first) : 0;
              while (__popc(word) > keep) word &= 0x7fffffffu >> __builtin_clz(word);
              L.bits[w] = word;
            }
          }
          __syncthreads();
          for (int i = tid; i < (int)C; i += NT) atomicOr(&L.bits[L.pos[i] >> 5], 1u << (L.pos[i] & 31));
          count_words();
          for (int w = tid; w < n_words; w += NT) {  // the list again, in order
            uint32_t word = L.bits[w], at = L.before[w];
            for (; word; word &= word - 1u) L.pos[at++] = (typename Lds::pos_t)(32 * w + __builtin_ctz(word));
          }
          __syncthreads();
          int32_t* out_idx = out_row(p, p.out_idx, row);
          elem_t* out_val = p.out_values ? out_row(p, reinterpret_cast<elem_t*>(p.out_values), row) : nullptr;
          const int32_t* table = table_of(p, row);
          const int32_t* in = p.in_idx ? p.in_idx + (int64_t)row * p.in_idx_stride : nullptr;
          for (int i = tid; i < k; i += NT) {
            const int at = (int)L.pos[i];
            int32_t pay = at;
            if (in) {
              pay = in[at];
            } else if (table) {
              const int page = p.page_shift >= 0 ? at >> p.page_shift : page_of(p, at);
              pay = table[page] * p.page_size + (at - page * p.page_size);
            }
            out_idx[i] = pay;
            if (out_val) out_val[i] = vals[at];
          }
          return;
        }
        C = CAP + 1u;
      }
      if (__builtin_expect(C > (uint32_t)CAP, 0)) {
        if constexpr (!kFits) {
          const int n_runs = (len + kTopkThreads - 1) / kTopkThreads;
          for (int j_lo = 0; j_lo < n_runs; j_lo += kSliceMaxRuns) {
            __syncthreads();
            select_slice<T, 0>(p, row, j_lo, kSliceMaxRuns, lds.slice);
          }
          return;
        } else {  // the list holds the whole row
          for (int i = tid; i < len; i += NT) L.pos[i] = (typename Lds::pos_t)i;
          for (int i = tid; i < n_words; i += NT) L.bits[i] = 0;
          C = (uint32_t)len;
          kbase = kKeyNegInf;
          __syncthreads();
        }
      }
    }
    // ---- 3. the k-th largest of them: the (C - k + 1)-th smallest distance above the floor -----------
    n = (int)C;
#pragma unroll
    for (int u = 0; u < CPT; ++u) x[u] = kNoElement;
    each_slot([&](int u) {
      const int i = u * NT + tid;
      pos[u] = (int32_t)L.pos[i < n ? i : 0];
    });
    elem_t raw[CPT];
    each_slot([&](int u) { raw[u] = vals[pos[u]]; });
    each_slot([&](int u) {
      float f;
      if constexpr (std::is_same<T, F32>::value) f = raw[u];
      else f = to_float<T>(raw[u]);
      x[u] = u * NT + tid < n ? KeyTraits<F32>::key(f) - kbase : kNoElement;
    });
    krem = krem0 = C - (uint32_t)k + 1u;
    narrow(kmax > kbase ? kmax - kbase : 0u, equal, false, [&](auto f) { each_slot([&](int u) { f(x[u]); }); });
  }
  uint32_t below = krem0 - krem;  // smaller than the bin's members

  // ---- the payloads (in flight from here on), and the members of the bin against each other --------
  const int32_t* table = table_of(p, row);
  int32_t pay[CPT];
  if (p.in_idx) {
    const int32_t* in = p.in_idx + (int64_t)row * p.in_idx_stride;
    each_slot([&](int u) { pay[u] = in[pos[u]]; });
  } else if (p.page_table) {
    int32_t entry[CPT];
    each_slot([&](int u) {
      const int page = p.page_shift >= 0 ? pos[u] >> p.page_shift : page_of(p, pos[u]);
      entry[u] = pos[u] - page * p.page_size;
      pay[u] = table[page];
    });
    each_slot([&](int u) { pay[u] = pay[u] * p.page_size + entry[u]; });
  } else {
    each_slot([&](int u) { pay[u] = pos[u]; });
  }
  uint32_t thr = lo, ties = n_in;  // s == 0: the members are equal
  if (s > 0u) {
    each_slot([&](int u) {
      if (x[u] - lo < (1u << s)) L.mem[atomicAdd(&L.n_mem, 1u)] = x[u];
    });
    __syncthreads();
    const uint32_t mine = lane < (int)n_in ? L.mem[lane] : kNoElement;
    uint32_t lt = 0, le = 0;
    for (int i = 0; i < (int)n_in; ++i) {
      const uint32_t other = __builtin_amdgcn_readlane(mine, i);
      lt += other < mine ? 1u : 0u;
      le += other <= mine ? 1u : 0u;
    }
    // krem <= n_in: some member has that rank
    const int src = __builtin_ctzll(__ballot(lane < (int)n_in && lt < krem && krem <= le));
    thr = __builtin_amdgcn_readlane(mine, src);
    lt = __builtin_amdgcn_readlane(lt, src);
    ties = __builtin_amdgcn_readlane(le, src) - lt;
    below += lt;
  }
  // how many of the ties are taken; the sample counts down from the reference, the survivors up from
  // the floor
  const uint32_t r = whole ? (uint32_t)k - below : (uint32_t)k - (C - below - ties);

  // ---- 4. places in position order ---------------------------------------------------------------
  auto place_of = [&](int32_t at) -> uint32_t {
    return (uint32_t)L.before[at >> 5] + __popc(L.bits[at >> 5] & ((1u << (at & 31)) - 1u));
  };
  const uint32_t flip = whole ? ~0u : 0u;  // selected: (x ^ flip) above (thr ^ flip)
  uint32_t take = 0;                       // bit u: slot u of this thread
  each_slot([&](int u) {
    if (x[u] != kNoElement && ((x[u] ^ flip) > (thr ^ flip) || (x[u] == thr && r == ties))) take |= 1u << u;
  });
  if (kTieRank && r != ties && ties <= (uint32_t)kFilterRank) {
    // the first r of a few ties: their positions against each other in the lanes of every wave (the bitmap below
    // takes three barriers and two scans more: bf16, 32 x 640 -> 128 5.5 -> 5.1 us; fp32 scores
    // seldom tie, and the branch costs their rows 0.1)
    each_slot([&](int u) {
      if (x[u] == thr) L.hist[1u + atomicAdd(&L.hist[0], 1u)] = (uint32_t)pos[u];  // (zero since the last level)
    });
    __syncthreads();
    const uint32_t mine = lane < (int)ties ? L.hist[1 + lane] : 0u;
    uint32_t earlier = 0;
    for (int i = 0; i < (int)ties; ++i) earlier += (uint32_t)__builtin_amdgcn_readlane(mine, i) < mine ? 1u : 0u;
    const int last = __builtin_ctzll(__ballot(lane < (int)ties && earlier == r - 1u));  // 1 <= r < ties
    const uint32_t until = __builtin_amdgcn_readlane(mine, last);
    each_slot([&](int u) {
      if (x[u] == thr && (uint32_t)pos[u] <= until) take |= 1u << u;
    });
  } else if (r != ties) {  // the first r of the ties
    each_slot([&](int u) {
      if (x[u] == thr) atomicOr(&L.bits[pos[u] >> 5], 1u << (pos[u] & 31));
    });
    count_words();
    each_slot([&](int u) {
      if (x[u] == thr && place_of(pos[u]) < r) take |= 1u << u;
    });
    __syncthreads();
    for (int i = tid; i < n_words; i += NT) L.bits[i] = 0;
    __syncthreads();
  }
  each_slot([&](int u) {
    if ((take >> u) & 1u) atomicOr(&L.bits[pos[u] >> 5], 1u << (pos[u] & 31));
  });
  count_words();
  int32_t* out_idx = out_row(p, p.out_idx, row);
  elem_t* out_val = p.out_values ? out_row(p, reinterpret_cast<elem_t*>(p.out_values), row) : nullptr;
  each_slot([&](int u) {
    if ((take >> u) & 1u) {
      const uint32_t at = place_of(pos[u]);
      out_idx[at] = pay[u];
      if (out_val) out_val[at] = vals[pos[u]];
    }
  });
}

constexpr int kFilterCap = 8192;

// Whether the survivors of a row of `len` elements fit the list with room to spare: the sample's
// count, five standard deviations of the margin put on it and five of its own spread, scaled to the row.
static bool filter_fits(int len, int k, int threads) {
  const double m = 4.0 * threads;
  if (len <= kFilterCap) return true;
  const double mu = (double)k * m / len, want = mu + 5.0 * __builtin_sqrt(mu) + 5.0;
  return (want + 5.0 * __builtin_sqrt(want)) * len / m <= 0.95 * kFilterCap;
}

// Whether a row's only workgroup here is faster than the slices, whose workgroups (up to eight a row, 256 in all)
// each go through the whole row: what grows with k is done by one workgroup here, and 16-bit scores nearly always
// tie at the threshold, which costs another bitmap (3 us).  One MI355X, rows of N(0, 1) with a bound and a page
// table, slices | one pass, us: fp32, 32 rows 8192 -> 1024 9.3 | 8.8, -> 2048 9.0 | 10.7, 12288 -> 1536 10.7 | 10.6,
// -> 4096 10.2 | 14.3, 16384 -> 2048 10.5 | 10.7, 32768 -> 3072 14.9 | 13.9, 65536 -> 4096 27 | 18; 128 rows 16384
// -> 2048 1.09 times, -> 3072 0.97 times as fast; 256 rows 12288 -> 3072 1.11, -> 4096 0.93; bf16, 32 rows 8192 ->
// 512 1.00, 16384 -> 512 0.97, 24576 -> 512 0.99, 32768 -> 1536 1.01, 49152 -> 3072 0.98; 256 rows 12288 -> 2048 1.01.
// More than 256 rows: a compute unit holds two of the 512-thread workgroups here and one of the slices' 1024: fp32 |
// bf16, 512 rows 3000 -> 1024 | 15.1 | 10.7, 8192 -> 2048 18.2 | 12.8, 8192 -> 2500 18.3 | 14.1 and 18.6 | 16.2, 5000
// -> 2500 18.7 | 16.5 and 18.9 | 17.2, 8192 -> 4096 20.9 | 20.7 and 21.3 | 21.7.  bf16 rows of up to kMidLen: 128 rows
// 8193 -> 512 10.4 | 9.6, 10240 -> 800 10.7 | 10.4, -> 1000 10.7 | 10.8; 256 rows 9000 -> 1500 12.9 | 12.6.
// (Over 480 shapes of more than 256 rows, 3000 to 10240 long: 0.68 to 1.0, but bf16 rows of 3000 to 4600 -> 1800 to 2500,
// whose survivors just pass a multiple of four a thread, 0.84 to 1.06, and 512 fp32 rows of 8193 -> 3300 23.2 | 25.2.)
// Rows of up to 2048 elements gain at any k (bf16 1500 -> 1024, a tie and as many survivors as there can be, 0.96),
// rows of more than 65536, which the slices read again in every pass, too.
static bool filter_pays(int len, int k, int rows, bool half) {
  if (len <= 2048 || len > 65536) return true;
  int most;
  if (len <= 8192)
    most = rows > 256 ? 2500 : (half ? 600 : 1300);
  else if (half && len <= kMidLen && rows > 64)
    most = rows < 256 ? 800 : 1500;
  else if (rows <= 64)
    most = half ? (len - 16384) / 12 : (len < 14400 ? 1600 : len / 9);
  else if (rows < 256)
    most = half ? (len - 8192) / 8 : (len < 10000 ? 2000 : len / 5);
  else
    most = half ? 1500 + (len - 10240) / 4 : (len < 13200 ? 3300 : len / 4);
  return k <= most;
}

// True: launched.  Threads by row length: the fewer, the cheaper the barriers and scans that make up
// most of a short row's time; 1024 are needed where the row's elements are (32 x 8192 -> 512: 7.1 us
// with 512, 9.3 at 10000 with 1024).  Up to kMidLen the registers of 512 hold a list of the whole row and still two
// workgroups a compute unit: fp32, with 1024 | 512 threads: 32 x 8193 -> 512 8.7 | 7.6, 256 x 10240 -> 800 9.3 | 8.8,
// 512 x 8193 -> 512 16.6 | 10.4, 1000 x 10240 -> 2000 41.3 | 30.2; where a row has a compute unit to itself the larger
// selections gain nothing (256 x 9000 -> 1200 9.8 | 9.4, -> 1500 10.1 | 10.2).  Longer rows in 512 threads leave one
// workgroup there (16384: 170 registers): 8% at k <= 1024, -12% at 3300, not taken.  The limits of 65536 and 262144 are the LDS of the bitmap.
template <typename T>
static bool launch_topk_filter(const TopkParams& p, int rows, hipStream_t st) {
  const dim3 grid(rows);
  if (!filter_pays(p.len, p.k, rows, !std::is_same<T, F32>::value)) return false;
  if (p.len <= 1024 - 4)
    hipLaunchKernelGGL((topk_filter_kernel<T, 256, 4, 1024, 1024>), grid, dim3(256), 0, st, p);
  else if (p.len <= 8192)
    hipLaunchKernelGGL((topk_filter_kernel<T, 512, 4, 8192, 8192>), grid, dim3(512), 0, st, p);
  else if (p.len <= kMidLen && (p.k <= 1200 || rows > 256))
    hipLaunchKernelGGL((topk_filter_kernel<T, 512, 4, kMidLen, kMidLen>), grid, dim3(512), 0, st, p);
  else if (!filter_fits(p.len, p.k, 1024))
    return false;
  else if (p.len <= 65536)
    hipLaunchKernelGGL((topk_filter_kernel<T, 1024, 8, kFilterCap, 65536>), grid, dim3(1024), 0, st, p);
  else if (p.len <= 262144)
    hipLaunchKernelGGL((topk_filter_kernel<T, 1024, 8, kFilterCap, 262144>), grid, dim3(1024), 0, st, p);
  else
    return false;
  return true;
}

}  // namespace tidal
