// A strip of columns of a prompt's product out = x w^T (16-bit operands, fp32 sums) for gfx950 (MI355X).
//
// The library multiplies in tiles of 256 x 256, so a product takes whole rounds of the 256 compute units, and a last
// round with a few tiles costs as much as a full one.  There the caller leaves the last strip of 256 columns out of
// the product and multiplies it here in small tiles, which takes a fifth of a round.  One MI355X, bf16, inner
// dimension 4096, us, cold weights, whole product -> without the strip + strip: 2900 x 22016 (4.03 rounds)
// 471 -> 384, 1388 x 22016 (2.02) 289 -> 206, 700 x 22016 (1.01) 158 -> 121, 3700 x 22016 (5.04) 574 -> 495.

#include "common.cuh"

namespace tidal {

constexpr int kGemmK = 64;  // elements of the inner dimension per stage: rows of 128 bytes in LDS
constexpr int kStripTile = 64, kStripGroups = 2, kStripStages = 4;
constexpr int kStripOperand = kStripTile * kGemmK * 2, kStripStage = 2 * kStripOperand * kStripGroups;  // bytes

struct StripParams {
  const uint16_t *x, *w;  // [m, k], [n, k]
  uint16_t* out;          // [m, n], rows out_stride elements apart
  int32_t m, n, k, m_tiles;
  int64_t out_stride;
};

// 16 bytes per lane to LDS bytes lds + 16 lane.  The asm holds the wait states itself: between m0 and the load,
// and between a vector instruction that wrote the scalar base and the load that reads it.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_lds(uint32_t lds, uint64_t base, uint32_t offset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(lds), "v"(offset), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop

// Bound by latency: 2900 rows are 184 tiles of 64 x 64 for 256 compute units, and each walks the whole inner
// dimension.  So the eight wavefronts of a workgroup walk it in two halves that alternate by stage, and four steps
// of 32 KB are on their way to LDS (256 columns of 4096: 25 us with one group of four, 16 - 19 with two, 18 - 21
// with four, whose two steps are all that LDS holds; the library's product of the strip 21 - 23).
// grid: tiles of 64 x 64, rows first, so that the workgroups on a strip of w run together.
template <typename T>
__global__ __launch_bounds__(kStripGroups * 256) void gemm_strip_kernel(StripParams p) {
  extern __shared__ __align__(1024) uint8_t strip_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave >> 2, in = wave & 3;  // four wavefronts share a tile's product over their stages
  const int m0 = (int)blockIdx.x % p.m_tiles * kStripTile, n0 = (int)blockIdx.x / p.m_tiles * kStripTile;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)strip_lds +
                        group * 2 * kStripOperand;
  // A row's eight 16-byte pieces are permuted by its number: eight rows that lanes read together lie in
  // different banks.  Rows past the end read the last one; what comes of them is not stored.
  uint32_t woff[2], xoff[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = (j * 4 + in) * 8 + (lane >> 3), piece = ((lane & 7) ^ (r & 7)) * 16;
    woff[j] = (uint32_t)(min(n0 + r, p.n - 1) - n0) * (uint32_t)(p.k * 2) + piece;
    xoff[j] = (uint32_t)(min(m0 + r, p.m - 1) - m0) * (uint32_t)(p.k * 2) + piece;
  }
  const uint64_t wb = (uint64_t)(p.w + (int64_t)n0 * p.k), xb = (uint64_t)(p.x + (int64_t)m0 * p.k);
  const int stages = p.k / kGemmK, steps = (stages + kStripGroups - 1) / kStripGroups;
  auto load = [&](int s) {  // a stage past the end reads the last one again and is not multiplied
    const int st = min(s * kStripGroups + group, stages - 1);
    const uint32_t to = lds0 + s % kStripStages * kStripStage + in * 1024;
    const uint64_t at = (uint64_t)st * kGemmK * 2;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      load_lds(to + j * 4096, wb + at, woff[j]);
      load_lds(to + kStripOperand + j * 4096, xb + at, xoff[j]);
    }
  };
  const int a = lane & 15, g = lane >> 4, wm = in & 1, wn = in >> 1;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < kStripStages - 1; ++s)
    if (s < steps) load(s);
  for (int s = 0; s < steps; ++s) {
    // the step's loads are there when no more than those of later steps are on their way; every wavefront has
    // read the step before it, whose buffer is filled next
    if (kStripStages > 2 && s + kStripStages - 2 < steps)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((kStripStages - 2) * 4) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (s + kStripStages - 1 < steps) load(s + kStripStages - 1);
    if (s * kStripGroups + group >= stages) continue;
    const uint8_t* at = strip_lds + s % kStripStages * kStripStage + group * 2 * kStripOperand;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int piece = ((half * 4 + g) ^ (a & 7)) * 16;
      u32x4 wf[2], xf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        wf[i] = *reinterpret_cast<const u32x4*>(at + (wn * 32 + i * 16 + a) * 128 + piece);
        xf[i] = *reinterpret_cast<const u32x4*>(at + kStripOperand + (wm * 32 + i * 16 + a) * 128 + piece);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma_16x16x32<T>(wf[i], xf[j], acc[i][j]);
    }
  }
  // the groups' sums, in their order
  f32x4* sums = reinterpret_cast<f32x4*>(strip_lds);
  __syncthreads();
  if (group) {
#pragma unroll
    for (int i = 0; i < 4; ++i) sums[((group - 1) * 4 + i) * 256 + in * 64 + lane] = acc[i >> 1][i & 1];
  }
  __syncthreads();
  if (group) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f32x4 v = acc[i >> 1][i & 1];
#pragma unroll
    for (int o = 0; o < kStripGroups - 1; ++o) v += sums[(o * 4 + i) * 256 + in * 64 + lane];
    const int col = n0 + wn * 32 + (i >> 1) * 16 + g * 4, row = m0 + wm * 32 + (i & 1) * 16 + a;
    if (row < p.m && col < p.n)
      *reinterpret_cast<u32x2*>(p.out + (int64_t)row * p.out_stride + col) =
          u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
  }
}

// The product of a short prompt, out = x w^T for up to 144 rows of x: all rows against 64 columns a workgroup, so that
// the weights come from memory once.  Few columns (an output or a down projection) leave the chip idle and each
// workgroup a long walk of the inner dimension, so that is cut (splits), and the four waves of a workgroup share a step
// of it: wave w multiplies a quarter of 32, every element of a step is read from LDS once, and the four sums meet at
// the end.  Bound by latency: three steps of up to 53 KB are all that LDS holds, and 30 bytes a cycle arrive of 64
// (walks that start at different steps change nothing; steps of 32 a wave, 64 bytes a row, take half as long again).
// bf16, cold weights, us, the library -> here: 4096 columns of 11008, 64 rows 35.5 -> 25.1, 93 41.3 -> 30.6, 138 44.5 ->
// 34.8; of 14336, 138 rows 55.5 -> 40.8; of 4096 15.6 -> 14.8, 17.5 -> 17.0, 22.3 -> 20.6; 6144 columns of 4096, 64 rows
// 18.5 -> 19.1, 93 23.4 -> 22.3, 138 39.5 -> 28.4.  Two row tiles (200 rows) and wide products stay the library's: 200 x
// 4096 of 11008 45 -> 43 to 66, 138 x 12288 of 4096 39.0 -> 38.6, x 22016 52 -> 73.
constexpr int kRowsN = 64, kRowsStages = 3, kRowsPitch = kRowsN + 4;  // columns of a tile; floats a row of its sums

struct RowsParams {
  const uint16_t *x, *w;  // [m, k], [n, k]
  uint16_t* out;          // [m, n]
  float* parts;           // [splits, m, n], splits > 1
  int32_t m, n, k, m_tiles, splits, strips;  // strips: n / 64 times splits
};

template <typename T, int MT>
__global__ __launch_bounds__(256, 1) void gemm_rows_kernel(const RowsParams p) {
  constexpr int BM = 16 * MT, NL = MT + 4, STAGE = (BM + kRowsN) * 256;  // bytes of a step of 128 in LDS
  extern __shared__ __align__(1024) uint8_t rows_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // eight strips at a time, one an XCD (workgroups go to the XCDs round-robin), their row tiles one after the other
  const int lin = blockIdx.x, strip = lin / (8 * p.m_tiles) * 8 + (lin & 7);
  if (strip >= p.strips) return;
  const int m0 = lin / 8 % p.m_tiles * BM, split = strip % p.splits, n0 = strip / p.splits * kRowsN;
  const int steps_all = p.k / 128, first = steps_all * split / p.splits;
  const int steps = steps_all * (split + 1) / p.splits - first;

  // ---- loads: four rows of 256 bytes per instruction, straight to LDS; piece s ^ r % 16 of row r lies in place s, so
  //      that sixteen rows read at one piece fall on different banks.  Wave w brings the rows 16 x + 4 w + 0 .. 3.
  const int lr = 4 * wave + (lane >> 4), piece = (lane & 15) ^ lr;
  uint32_t xoff[MT], woff = (uint32_t)lr * (uint32_t)(p.k * 2) + piece * 16;
#pragma unroll
  for (int x = 0; x < MT; ++x)
    xoff[x] = (uint32_t)(min(m0 + 16 * x + lr, p.m - 1) - m0) * (uint32_t)(p.k * 2) + piece * 16;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)rows_lds + wave * 1024;
  const uint64_t xb = (uint64_t)(p.x + (int64_t)m0 * p.k) + (uint64_t)first * 256;
  const uint64_t wb = (uint64_t)(p.w + (int64_t)n0 * p.k) + (uint64_t)first * 256;
  const uint32_t wrow = (uint32_t)p.k * 32;  // bytes of 16 rows
  auto load = [&](int i, uint32_t slot) __attribute__((always_inline)) {  // a step past the end reads the last one again
    const uint64_t at = (uint64_t)(i < steps ? i : steps - 1) * 256;
    const uint32_t to = lds0 + slot;
#pragma unroll
    for (int x = 0; x < 4; ++x) load_lds(to + (MT + x) * 4096, wb + at + (uint64_t)x * wrow, woff);
#pragma unroll
    for (int x = 0; x < MT; ++x) load_lds(to + x * 4096, xb + at, xoff[x]);
  };
  // ---- operands: wave w multiplies the elements 32 w .. 32 w + 31 of a step
  const int c16 = lane & 15, g = lane >> 4;
  const uint8_t* const mine = rows_lds + c16 * 256 + 16 * ((4 * wave + g) ^ c16);
  u32x4 xf[2][MT], wf[2][4];
  auto read = [&](int to, uint32_t slot) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < 4; ++x) wf[to][x] = *reinterpret_cast<const u32x4*>(mine + slot + (MT + x) * 4096);
#pragma unroll
    for (int x = 0; x < MT; ++x) xf[to][x] = *reinterpret_cast<const u32x4*>(mine + slot + x * 4096);
  };
  f32x4 acc[MT][4];
#pragma unroll
  for (int i = 0; i < MT * 4; ++i) acc[i >> 2][i & 3] = f32x4{0.f, 0.f, 0.f, 0.f};

  load(0, 0);
  load(1, STAGE);
  load(2, 2 * STAGE);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * NL) : "memory");
  read(0, 0);
  uint32_t slot = 0;
  auto step = [&](int i, int cur) __attribute__((always_inline)) {
    // The wave's operands of step i are in registers and its share of step i + 1 is there when no more than its
    // loads of step i + 2 are on their way; behind the barrier that holds for all waves, and the place of step i is
    // free for step i + 3.
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NL) : "memory");
    load(i + 3, slot);
    slot = slot == 2 * STAGE ? 0 : slot + STAGE;
    read(cur ^ 1, slot);
#pragma unroll
    for (int x = 0; x < MT; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y) acc[x][y] = mfma_16x16x32<T>(xf[cur][x], wf[cur][y], acc[x][y]);
  };
  int i = 0;
  for (; i + 1 < steps; i += 2) {
    step(i, 0);
    step(i + 1, 1);
  }
  if (i < steps) step(i, 0);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __syncthreads();

  // ---- the four waves' sums meet in LDS: a lane holds rows 4 g + i of a block, column c16 of another
  float* const sums = reinterpret_cast<float*>(rows_lds);
#pragma unroll
  for (int x = 0; x < MT; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        sums[(wave * BM + 16 * x + 4 * g + e) * kRowsPitch + 16 * y + c16] = acc[x][y][e];
  __syncthreads();
  for (int at = tid; at < BM * 16; at += 256) {
    const int r = at >> 4, c = (at & 15) * 4, row = m0 + r;
    if (row >= p.m) break;  // rows only grow
    f32x4 v = *reinterpret_cast<const f32x4*>(sums + r * kRowsPitch + c);
#pragma unroll
    for (int q = 1; q < 4; ++q) v += *reinterpret_cast<const f32x4*>(sums + (q * BM + r) * kRowsPitch + c);
    const int64_t to = (int64_t)row * p.n + n0 + c;
    if (p.splits == 1)
      *reinterpret_cast<u32x2*>(p.out + to) = u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
    else
      *reinterpret_cast<f32x4*>(p.parts + (int64_t)split * p.m * p.n + to) = v;
  }
}

// the sum of the splits' partial products
template <typename T>
__global__ __launch_bounds__(256) void gemm_sum_kernel(const float* parts, uint16_t* out, int64_t n, int splits) {
  const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (at >= n) return;
  f32x4 v = *reinterpret_cast<const f32x4*>(parts + at);
  for (int s = 1; s < splits; ++s) v += *reinterpret_cast<const f32x4*>(parts + s * n + at);
  *reinterpret_cast<u32x2*>(out + at) = u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
}

template <typename T, int MT>
static int launch_rows(const RowsParams& p, hipStream_t st) {
  constexpr int kStages = kRowsStages * (16 * MT + kRowsN) * 256, kSums = 4 * 16 * MT * kRowsPitch * 4;
  constexpr int kBytes = kStages > kSums ? kStages : kSums;
  static_assert(kBytes <= 160 * 1024, "a tile's steps and sums fit LDS");
  auto kernel = gemm_rows_kernel<T, MT>;
  TD_HIP_CHECK(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kBytes));
  hipLaunchKernelGGL(kernel, dim3((p.strips + 7) / 8 * 8 * p.m_tiles), dim3(256), kBytes, st, p);
  if (p.splits > 1) {
    const int64_t n = (int64_t)p.m * p.n;
    hipLaunchKernelGGL(gemm_sum_kernel<T>, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, st, p.parts, p.out, n,
                       p.splits);
  }
  return TD_OK;
}

template <typename T>
static int launch_rows_of(const RowsParams& p, int mt, hipStream_t st) {
  if (mt == 3) return launch_rows<T, 3>(p, st);
  if (mt == 5) return launch_rows<T, 5>(p, st);
  if (mt == 7) return launch_rows<T, 7>(p, st);
  return launch_rows<T, 9>(p, st);
}

template <typename T>
static int launch_strip(const StripParams& p, hipStream_t st) {
  auto kernel = gemm_strip_kernel<T>;
  constexpr int kBytes = kStripStages * kStripStage;
  TD_HIP_CHECK(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kBytes));
  hipLaunchKernelGGL(kernel, dim3(p.m_tiles * ((p.n + kStripTile - 1) / kStripTile)), dim3(kStripGroups * 256),
                     kBytes, st, p);
  return TD_OK;
}

}  // namespace tidal

using namespace tidal;

extern "C" int td_gemm_strip(const void* x, const void* w, void* out, int32_t m, int32_t n, int32_t k,
                             int64_t out_stride, int32_t dtype, void* stream) {
  TD_REQUIRE(x && w && out, "td_gemm_strip: NULL argument");
  TD_REQUIRE(m >= 1 && n >= 4 && n % 4 == 0 && k >= kGemmK && k % kGemmK == 0 && k <= (1 << 24),
             "td_gemm_strip: %d rows, %d columns (multiple of 4), inner %d (multiple of %d)", m, n, k, kGemmK);
  TD_REQUIRE(out_stride >= n && out_stride % 4 == 0, "td_gemm_strip: row stride %lld", (long long)out_stride);
  TD_REQUIRE((((uintptr_t)x | (uintptr_t)w) & 15) == 0 && ((uintptr_t)out & 7) == 0,
             "td_gemm_strip: x and w must be 16-byte aligned, out 8-byte");
  StripParams p;
  p.x = (const uint16_t*)x;
  p.w = (const uint16_t*)w;
  p.out = (uint16_t*)out;
  p.m = m;
  p.n = n;
  p.k = k;
  p.m_tiles = (m + kStripTile - 1) / kStripTile;
  p.out_stride = out_stride;
  TD_REQUIRE((int64_t)p.m_tiles * ((n + kStripTile - 1) / kStripTile) < ((int64_t)1 << 31),
             "td_gemm_strip: %d x %d is too large", m, n);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  int rc;
  if (dtype == TD_F16)
    rc = launch_strip<F16>(p, st);
  else if (dtype == TD_BF16)
    rc = launch_strip<BF16>(p, st);
  else
    return fail(TD_ERR_UNSUPPORTED, "td_gemm_strip failed to dispatch with dtype %d", dtype);
  if (rc != TD_OK) return rc;
  TD_HIP_CHECK(hipGetLastError());
  return TD_OK;
}

extern "C" int td_gemm_rows(const void* x, const void* w, void* out, int32_t m, int32_t n, int32_t k, int32_t splits,
                            void* parts, int64_t parts_bytes, int32_t dtype, void* stream) {
  TD_REQUIRE(x && w && out, "td_gemm_rows: NULL argument");
  TD_REQUIRE(m >= 1 && n >= kRowsN && n % kRowsN == 0 && k >= 128 && k % 128 == 0 && k <= (1 << 20),
             "td_gemm_rows: %d rows, %d columns (multiple of 64), inner %d (multiple of 128)", m, n, k);
  TD_REQUIRE(splits >= 1 && splits <= k / 128 && splits <= 16, "td_gemm_rows: %d splits of %d", splits, k);
  TD_REQUIRE((((uintptr_t)x | (uintptr_t)w | (uintptr_t)parts) & 15) == 0 && ((uintptr_t)out & 7) == 0,
             "td_gemm_rows: x, w and parts must be 16-byte aligned, out 8-byte");
  TD_REQUIRE(splits == 1 || (parts && parts_bytes >= (int64_t)splits * m * n * 4), "td_gemm_rows: parts hold %lld bytes",
             (long long)parts_bytes);
  RowsParams p;
  p.x = (const uint16_t*)x;
  p.w = (const uint16_t*)w;
  p.out = (uint16_t*)out;
  p.parts = (float*)parts;
  p.m = m;
  p.n = n;
  p.k = k;
  p.splits = splits;
  p.strips = n / kRowsN * splits;
  const int tiles = (m + 143) / 144, blocks = ((m + tiles - 1) / tiles + 15) / 16;  // of 16 rows, a tile
  const int mt = blocks <= 3 ? 3 : (blocks <= 5 ? 5 : (blocks <= 7 ? 7 : 9));
  p.m_tiles = (m + 16 * mt - 1) / (16 * mt);
  TD_REQUIRE((int64_t)p.m_tiles * (p.strips + 7) < ((int64_t)1 << 31), "td_gemm_rows: %d x %d is too large", m, n);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  int rc;
  if (dtype == TD_F16)
    rc = launch_rows_of<F16>(p, mt, st);
  else if (dtype == TD_BF16)
    rc = launch_rows_of<BF16>(p, mt, st);
  else
    return fail(TD_ERR_UNSUPPORTED, "td_gemm_rows failed to dispatch with dtype %d", dtype);
  if (rc != TD_OK) return rc;
  TD_HIP_CHECK(hipGetLastError());
  return TD_OK;
}
