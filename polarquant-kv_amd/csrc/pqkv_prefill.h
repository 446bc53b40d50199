// Shared by the prefill attention kernels (pqkv_prefill.hip, which decodes the
// cache's tiles per row block, and pqkv_prefill_planes.hip, over tiles decoded
// once per call): the tile, the split of fp32 operands into fp16 pairs and the
// row reductions of the 16x16x32 accumulator layout.
#pragma once
#include "pqkv_device.h"
#include "pqkv_launch.h"

namespace pqkv {
namespace {

constexpr int kPT = 64;                   // kv tokens per tile
constexpr int kPW = 8;                    // waves per workgroup
constexpr float kPlaneScale = kPrefillPlaneScale;              // codebook planes and queries, x 2^6
constexpr float kScoreUnscale = 1.0f / (kPlaneScale * kPlaneScale);

// four floats on a dword boundary
typedef float float4_dw __attribute__((ext_vector_type(4), aligned(4)));

// x is made opaque first: otherwise the compiler rounds a product once for lo's
// hi (v_fma_mixlo_f16) and twice for the stored one, and where they differ the
// pair is off by an fp16 step (1e-3 of a weight, in one of some thousands).
__device__ __forceinline__ void split2(float x, half_t *hi, half_t *lo) {
  asm("" : "+v"(x));
  const half_t h = (half_t)x;
  *hi = h;
  *lo = (half_t)(x - (float)h);
}

// The same of two products a b, as packed pairs: lo is taken from the exact
// product (a mixed fused multiply-add), so a pair also holds what rounding the
// product lost. The hi halves are made opaque, which keeps one rounding of each.
// With the products opaque instead, which costs a widening and a subtraction per
// weight, a prefill of 509 tokens against 32 000 cached ones (batch 32, 32 query
// / 8 kv heads, d = 128) takes 22.6 ms in place of 21.5.
__device__ __forceinline__ void split2_products(float a0, float b0, float a1, float b1, half2_t *hi, half2_t *lo) {
  half2_t h = {(half_t)(a0 * b0), (half_t)(a1 * b1)};
  asm("" : "+v"(h));
  *hi = h;
  *lo = half2_t{(half_t)__builtin_fmaf(a0, b0, -(float)h[0]), (half_t)__builtin_fmaf(a1, b1, -(float)h[1])};
}

__device__ __forceinline__ float4_t mfma16(half8_t a, half8_t b, float4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// First tile of share sp when `all` tiles are cut into `splits` shares:
// floor(all sp / splits), without the 64-bit division.
__host__ __device__ __forceinline__ int share_begin(int all, int sp, int splits) {
  const int q = all / splits, r = all - q * splits;
  return q * sp + r * sp / splits;
}

// max / sum of a value over the four lanes of a column (l, l ^ 16, l ^ 32, l ^ 48)
__device__ __forceinline__ float rows_max(float x) {
  auto a = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
  x = fmaxf(__builtin_bit_cast(float, (uint32_t)a[0]), __builtin_bit_cast(float, (uint32_t)a[1]));
  auto b = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
  return fmaxf(__builtin_bit_cast(float, (uint32_t)b[0]), __builtin_bit_cast(float, (uint32_t)b[1]));
}
__device__ __forceinline__ float rows_sum(float x) {
  auto a = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
  x = __builtin_bit_cast(float, (uint32_t)a[0]) + __builtin_bit_cast(float, (uint32_t)a[1]);
  auto b = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
  return __builtin_bit_cast(float, (uint32_t)b[0]) + __builtin_bit_cast(float, (uint32_t)b[1]);
}

// Value of lane `row` (0..15) for output row 4 grp + i (v is the same in
// the four lanes of a column): one lane gather per i.
__device__ __forceinline__ void per_row(float v, int grp, float (&f)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    f[i] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * (4 * grp + i), __builtin_bit_cast(int, v)));
}

}  // namespace
}  // namespace pqkv
