// The GPU group (min / scale) encoder with its rotations on the fp32 matrix
// cores (pqkv_fma_mfma.h): the arithmetic of group_gpu_compress_kernel
// (pqkv_group_gpu.hip), bit for bit, for d = 64 and 128 and groups of 8 .. d
// coordinates (a power of two).
//
// That kernel takes one vector per wave and reads all of R from the L2 for
// each (64 KB per 512 bytes of output at d = 128): 383 us for 131 072 vectors,
// 11 TFLOP/s. Here a workgroup of four waves takes 32 vectors per step (64 at
// d = 64), each wave computes 32 coordinates of 32 vectors from its rows of R
// in registers, and the rotated vectors go through LDS to d / 16 threads per
// vector, 16 consecutive coordinates each, which find the norm, the groups'
// minima and scales and the codes. The step's quantiser runs beside the other
// workgroups' matrix products (three per compute unit). 57 us for the same
// vectors (the products alone would take 30; 64 us with an IEEE division per
// coordinate and per code instead of the Markstein quotients).
//
// With a residual (QJL keys) the quantiser's rotated residuals are staged
// like the input and rotated back by a second product.
#include "pqkv_cells.h"
#include "pqkv_device.h"
#include "pqkv_fma_mfma.h"
#include "pqkv_launch.h"

namespace pqkv {

namespace {

struct GroupCompressArgs {
  const void *x;
  const float *R, *Rt;           // R may be null without a residual (Rt is then used)
  int64_t n;
  int x_dtype, bits, gs_shift, pdt;
  void *radius, *mins, *scales;
  uint8_t *codes;
  float *resid;
};

__device__ __forceinline__ float clamp_in(float x) { return x > 65000.0f ? 65000.0f : x < -65000.0f ? -65000.0f : x; }

__device__ __forceinline__ void put_param(void *p, int dt, int64_t i, float v) {
  if (dt == PQKV_F16) ((half_t *)p)[i] = (half_t)v;
  else ((float *)p)[i] = v;
}

}  // namespace

template <int D, bool RESID>
__global__ void __launch_bounds__(256, RESID ? 2 : 3) group_compress_mfma_kernel(const GroupCompressArgs a) {
  constexpr int NJ = D / 32, VS = 32 * (4 / NJ), PITCH = ChainRow<D>::kPitch;
  constexpr int ITEMS = VS * (D / 8) / 256;   // 8-coordinate pieces per thread and step
  constexpr int T = D / 16;                   // quantiser threads per vector
  constexpr int NM = 64 / T;                  // norm slots per thread
  __shared__ __attribute__((aligned(16))) float xs[2][VS * PITCH];
  __shared__ __attribute__((aligned(16))) float ys[VS * PITCH];    // the step's rotated vectors, natural order
  __shared__ __attribute__((aligned(16))) float es[RESID ? VS * PITCH : 4];   // its residuals, staged order
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int jt = wave % NJ, vh = wave / NJ;
  const int64_t n = a.n, steps = (n + VS - 1) / VS;
  const int gs_shift = a.gs_shift, ng = D >> gs_shift;
  const int cb = a.bits == 4 ? 4 : a.bits == 2 ? 2 : 8;
  const float L = (float)((1 << a.bits) - 1);

  // ---- input: pieces of 8 coordinates, raw words one step ahead ----
  u32x4 raw[ITEMS][2];
  auto load = [&](int64_t step) {
#pragma unroll
    for (int u = 0; u < ITEMS; ++u) {
      const int item = tid + 256 * u;
      int64_t v = step * VS + item / (D / 8);
      v = v < n ? v : n - 1;
      const int64_t e = v * D + 8 * (item % (D / 8));
      if (a.x_dtype == PQKV_F32) {
        const u32x4 *p = (const u32x4 *)((const float *)a.x + e);
        raw[u][0] = p[0];
        raw[u][1] = p[1];
      } else {
        raw[u][0] = *(const u32x4 *)((const uint16_t *)a.x + e);
      }
    }
  };
  auto stage = [&](int b) {
#pragma unroll
    for (int u = 0; u < ITEMS; ++u) {
      const int item = tid + 256 * u;
      float o[8];
      if (a.x_dtype == PQKV_F32) {
        const float4_t f0 = __builtin_bit_cast(float4_t, raw[u][0]), f1 = __builtin_bit_cast(float4_t, raw[u][1]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o[e] = f0[e];
          o[4 + e] = f1[e];
        }
      } else if (a.x_dtype == PQKV_F16) {
        const half8_t h = __builtin_bit_cast(half8_t, raw[u][0]);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (float)h[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t w = raw[u][0][e];
          o[2 * e] = bf16_to_float(w & 0xFFFFu);
          o[2 * e + 1] = bf16_to_float(w >> 16);
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = clamp_in(o[e]);   // NaN stays NaN
      chain_put8<D>(&xs[b][(item / (D / 8)) * PITCH], item % (D / 8), o);
    }
  };
  // the chains of 32 staged vectors (rows of `src`) against r[]; VROWS: the
  // vectors are the accumulator's rows (else its columns)
  auto product = [&](auto vrows, const float *src, const float (&r)[D / 2]) {
    constexpr bool VROWS = decltype(vrows)::value;
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    const float *row = src + (32 * vh + col) * PITCH + half * (D / 2);
#pragma unroll
    for (int s4 = 0; s4 < D / 8; ++s4) {
      const float4_t v = *(const float4_t *)(row + 4 * s4);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = VROWS ? mfma_fma2(v[e], r[4 * s4 + e], acc) : mfma_fma2(r[4 * s4 + e], v[e], acc);
    }
    return acc;
  };

  int64_t step = blockIdx.x;
  load(step);
  float r[D / 2], ri[RESID ? D / 2 : 1];
  if (a.R != nullptr) chain_load_rows<D>(a.R, tid, 32 * jt + col, half, &xs[0][0], r);
  else chain_load_columns<D>(a.Rt, 32 * jt + col, half, r);
  if constexpr (RESID) chain_load_columns<D>(a.R, 32 * jt + col, half, ri);
  stage(0);
  lds_barrier();
  const int qv = tid / T, qt = tid % T;       // quantiser: vector of the step, coordinates 16 qt ..
  for (int b = 0; step < steps; step += gridDim.x, b ^= 1) {
    const bool more = step + gridDim.x < steps;
    if (more) load(step + gridDim.x);
    {
      // rows = coordinates: a lane holds runs of four of one vector
      const f32x16 acc = product(std::integral_constant<bool, false>{}, xs[b], r);
      float *dst = ys + (32 * vh + col) * PITCH + 32 * jt + 4 * half;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *(float4_t *)(dst + 8 * q) = float4_t{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    }
    lds_barrier();
    const int64_t v = step * VS + qv;
    const bool live = v < n;
    {
#pragma clang fp contract(off)
      const float *yv = ys + qv * PITCH;
      // |y|^2 in fp64 (the squares are exact): slots l = 0..63 hold
      // y_l^2 (+ y_{l+64}^2), added by a tree over l's bits 5 .. 0
      double sq[NM];
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const double y0 = (double)yv[qt + T * m];
        sq[m] = y0 * y0;
        if constexpr (D == 128) {
          const double y1 = (double)yv[64 + qt + T * m];
          sq[m] = sq[m] + y1 * y1;
        }
      }
#pragma unroll
      for (int w = NM / 2; w > 0; w >>= 1)
#pragma unroll
        for (int m = 0; m < w; ++m) sq[m] = sq[m] + sq[m + w];
      double tot = sq[0];
#pragma unroll
      for (int s = T / 2; s > 0; s >>= 1) tot = tot + __shfl_xor(tot, s, 64);
      const float rad = (float)__builtin_sqrt(tot);
      const bool zero = rad < 1e-30f;
      const float safe = zero ? 1e-30f : rad;
      float u[16], y[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4_t y4 = *(const float4_t *)(yv + 16 * qt + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[4 * q + e] = y4[e];
      }
      // u = RN(y / safe): the Markstein quotient of pqkv_cells.h where it is
      // exact (safe in [2^-40, inf), no quotient below 2^-60, where the
      // residual could round), else a division per coordinate
      const float inv = __fdiv_rn(1.0f, safe);
      float least = 1.0f;
#pragma unroll
      for (int e = 0; e < 16; ++e) least = fminf(least, fabsf(y[e] * inv));
      if (__builtin_amdgcn_ballot_w64(!(least >= 0x1p-60f && rad >= 0x1p-40f && rad < __builtin_inff())) == 0) {
#pragma unroll
        for (int e = 0; e < 16; ++e) u[e] = dir_markstein(y[e], safe, inv);
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) u[e] = zero ? 0.0f : __fdiv_rn(y[e], safe);
      }
      // minima and maxima of the two halves of eight, joined up to the group
      float lo[2], hi[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        lo[q] = hi[q] = u[8 * q];
#pragma unroll
        for (int e = 1; e < 8; ++e) {
          lo[q] = fminf(lo[q], u[8 * q + e]);
          hi[q] = fmaxf(hi[q], u[8 * q + e]);
        }
      }
      if (gs_shift >= 4) {
        lo[0] = fminf(lo[0], lo[1]);
        hi[0] = fmaxf(hi[0], hi[1]);
        for (int s = 1; s < (1 << (gs_shift - 4)); s <<= 1) {
          lo[0] = fminf(lo[0], shfl_xor_f(lo[0], s));
          hi[0] = fmaxf(hi[0], shfl_xor_f(hi[0], s));
        }
        lo[1] = lo[0];
        hi[1] = hi[0];
      }
      float sc[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float range = hi[q] - lo[q];
        sc[q] = range > 0.0f ? __fdiv_rn(range, L) : 1.0f;
      }
      // t = RN((u - lo) / s), clamped, rounded half to even. The Markstein
      // quotient is exact for s in [2^-40, inf) and t >= 2^-60, and a smaller
      // t rounds to 0 in either form.
      uint32_t code[16];
      const bool plain = sc[0] >= 0x1p-40f && sc[1] >= 0x1p-40f && sc[0] < __builtin_inff() && sc[1] < __builtin_inff();
      auto code_of = [&](float t) {
        t = t < 0.0f ? 0.0f : t > L ? L : t;
        return (uint32_t)(uint8_t)rintf(t);
      };
      if (__builtin_amdgcn_ballot_w64(!plain) == 0) {
        const float is[2] = {__fdiv_rn(1.0f, sc[0]), __fdiv_rn(1.0f, sc[1])};
#pragma unroll
        for (int e = 0; e < 16; ++e) code[e] = code_of(dir_markstein(u[e] - lo[e >> 3], sc[e >> 3], is[e >> 3]));
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) code[e] = code_of(__fdiv_rn(u[e] - lo[e >> 3], sc[e >> 3]));
      }
      if (live) {
        if (qt == 0) put_param(a.radius, a.pdt, v, rad > 65504.0f ? 65504.0f : rad);
        if (gs_shift == 3) {
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            put_param(a.mins, a.pdt, v * ng + 2 * qt + q, lo[q]);
            put_param(a.scales, a.pdt, v * ng + 2 * qt + q, sc[q]);
          }
        } else if ((qt & ((1 << (gs_shift - 4)) - 1)) == 0) {
          const int g = qt >> (gs_shift - 4);
          put_param(a.mins, a.pdt, v * ng + g, lo[0]);
          put_param(a.scales, a.pdt, v * ng + g, sc[0]);
        }
        uint8_t *row = a.codes + v * (D * cb / 8) + 2 * cb * qt;
        if (cb == 4) {
          uint32_t w[2] = {0, 0};
#pragma unroll
          for (int e = 0; e < 16; ++e) w[e >> 3] |= code[e] << (4 * (e & 7));
          *(uint2 *)row = make_uint2(w[0], w[1]);
        } else if (cb == 2) {
          uint32_t w = 0;
#pragma unroll
          for (int e = 0; e < 16; ++e) w |= code[e] << (2 * e);
          *(uint32_t *)row = w;
        } else {
          u32x4 w = {0, 0, 0, 0};
#pragma unroll
          for (int e = 0; e < 16; ++e) w[e >> 2] |= code[e] << (8 * (e & 3));
          *(u32x4 *)row = w;
        }
      }
      if constexpr (RESID) {
        // rotated-space residual with the unrounded lo / s
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float er[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float dq = (float)code[8 * q + e] * sc[q] + lo[q];
            const float hat = dq * safe;
            er[e] = y[8 * q + e] - hat;
          }
          chain_put8<D>(es + qv * PITCH, 2 * qt + q, er);
        }
      }
    }
    if (more) stage(b ^ 1);
    lds_barrier();
    if constexpr (RESID) {
      // e = er R; rows = vectors: 32 consecutive coordinates per store
      const f32x16 acc = product(std::integral_constant<bool, true>{}, es, ri);
      const int64_t v0 = step * VS;
      const int left = (int)(n - v0 < VS ? n - v0 : VS);
      const __amdgpu_buffer_rsrc_t out =
          __builtin_amdgcn_make_buffer_rsrc((void *)(a.resid + v0 * D), (short)0, left * D * 4, 0x00020000);
      const int off = ((32 * vh + 4 * half) * D + 32 * jt + col) * 4;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float t = acc[i];
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, t), out, off + mfma32_row(i, 0) * D * 4, 0, 0);
      }
      // (the next step's residuals are written after its first barrier)
    }
  }
}

bool group_compress_mfma_ok(const void *x, const float *R, const float *Rt, int d, int gs, const uint8_t *codes,
                            const float *resid) {
  return (d == 64 || d == 128) && gs >= 8 && gs <= d && (gs & (gs - 1)) == 0 && (uintptr_t)x % 16 == 0 &&
         (uintptr_t)R % 16 == 0 && (uintptr_t)Rt % 4 == 0 && (uintptr_t)codes % 16 == 0 && (uintptr_t)resid % 4 == 0;
}

hipError_t launch_group_compress_mfma(const void *x, int x_dtype, const float *Rt, const float *R, int64_t n, int d,
                                      int bits, int gs, void *radius, uint8_t *codes, void *mins, void *scales,
                                      int pdt, float *resid, hipStream_t s) {
  int shift = 0;
  while ((1 << shift) < gs) ++shift;
  const GroupCompressArgs a{x, R, Rt, n, x_dtype, bits, shift, pdt, radius, mins, scales, codes, resid};
  const int vs = d == 128 ? 32 : 64;
  const int64_t steps = (n + vs - 1) / vs, cap = (resid ? 2 : 3) * (int64_t)device_compute_units();
  const int grid = (int)(steps < cap ? steps : cap);
  if (d == 128) {
    if (resid) group_compress_mfma_kernel<128, true><<<grid, 256, 0, s>>>(a);
    else group_compress_mfma_kernel<128, false><<<grid, 256, 0, s>>>(a);
  } else {
    if (resid) group_compress_mfma_kernel<64, true><<<grid, 256, 0, s>>>(a);
    else group_compress_mfma_kernel<64, false><<<grid, 256, 0, s>>>(a);
  }
  return hipGetLastError();
}

}  // namespace pqkv
