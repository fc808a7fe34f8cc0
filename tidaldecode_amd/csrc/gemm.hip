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
