// Rotation of many vectors, y = R x or R^T x, and the decode of block-encoded
// vectors back to the original space, on the fp32 matrix cores
// (pqkv_fma_mfma.h: bit for bit the FMA chains of rotate_kernel).
//
// Work split. A workgroup of four waves takes 32 vectors per step at d = 128
// (64 at d = 64). Wave w computes the 32 output coordinates 32 (w % (d / 32))
// .. of 32 of them; its 32 rows (or columns) of R stay in registers for the
// launch (d / 2 per lane; rows come through LDS, so that R is read in runs) and the step's vectors are staged in LDS by all four
// waves, widened to fp32, double-buffered, loaded through registers one step
// ahead, one barrier per step. A wave's step is d / 2 dependent instructions
// of 64 cycles beside d / 8 LDS reads, so it is bound by the matrix cores and
// its loads, stores and address arithmetic run beside them (four waves per
// SIMD).
//
// Measured at d = 128, 400 000 fp16 vectors to fp32 (13.1 GFLOP): 103 us,
// 127 TFLOP/s of the 145 the instruction reaches alone, against 392 us for
// rotate_kernel (98 000 vectors: 30 against 103 us). The barrier of a step
// waits for LDS only: with __syncthreads, which also waits for the step's
// stores, 148 us.
//
// The vectors are rows of the MFMA's A operand, the coordinates columns, so a
// store instruction writes 32 consecutive coordinates of two vectors.
#include "pqkv_cells.h"
#include "pqkv_device.h"
#include "pqkv_fma_mfma.h"
#include "pqkv_launch.h"

namespace pqkv {

namespace {

template <int D>
struct RotShape {
  static constexpr int NJ = D / 32;              // 32-coordinate column tiles
  static constexpr int VS = 32 * (4 / NJ);       // vectors per workgroup step
  static constexpr int PITCH = ChainRow<D>::kPitch;
  static constexpr int WAVES = 4;                // per SIMD, = workgroups per compute unit
  static constexpr int ITEMS = VS * (D / 8) / 256;   // 8-coordinate pieces per thread and step
};

// Sources: the raw words of coordinates 8 j8 .. of vector v, and their values.
template <int D>
struct F32Source {
  const float *x;
  struct Raw { float4_t a, b; };
  __device__ __forceinline__ Raw load(int64_t v, int j8) const {
    const float4_t *p = (const float4_t *)(x + v * D + 8 * j8);
    return {p[0], p[1]};
  }
  __device__ __forceinline__ void values(const Raw &w, int, const float *, float (&o)[8]) const {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = w.a[e];
      o[4 + e] = w.b[e];
    }
  }
};
template <int D>
struct F16Source {
  const half_t *x;
  struct Raw { u32x4 a; };
  __device__ __forceinline__ Raw load(int64_t v, int j8) const { return {*(const u32x4 *)(x + v * D + 8 * j8)}; }
  __device__ __forceinline__ void values(const Raw &w, int, const float *, float (&o)[8]) const {
    const half8_t h = __builtin_bit_cast(half8_t, w.a);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (float)h[e];
  }
};
// fp32 rows of a strided [n_seq][Hq][n_q] arrangement taken in
// [n_seq][n_q][Hq] order (ggml's queries).
template <int D>
struct StridedSource {
  const float *x;
  int64_t s_q, s_h, s_s;
  int n_q, Hq;
  using Raw = typename F32Source<D>::Raw;
  __device__ __forceinline__ Raw load(int64_t v, int j8) const {
    const int64_t rest = v / Hq, h = v - rest * Hq;
    const int64_t sq = rest / n_q, iq = rest - sq * n_q;
    return F32Source<D>{x + sq * s_s + h * s_h + iq * s_q}.load(0, j8);
  }
  __device__ __forceinline__ void values(const Raw &w, int j8, const float *cb, float (&o)[8]) const {
    F32Source<D>{x}.values(w, j8, cb, o);
  }
};
// Block-encoded vectors: r16 c[code]. A piece is one dword of qs (4-bit) or
// half a dword (2-bit) at 2-byte alignment.
template <int D, int BITS>
struct BlocksSource {
  const uint8_t *blocks;
  int64_t outer_stride;                          // bytes between rows of n_inner vectors
  FastDiv by_inner;
  bool split;                                    // false: one row
  uint32_t n_inner;
  struct Raw { uint32_t codes, radius; };
  __device__ __forceinline__ Raw load(int64_t v, int j8) const {
    int64_t at = v * vector_bytes(D, BITS);
    if (split) {
      const uint32_t o = by_inner.div((uint32_t)v);
      at = o * outer_stride + (int64_t)((uint32_t)v - o * n_inner) * vector_bytes(D, BITS);
    }
    const uint8_t *vec = blocks + at;
    const uint8_t *qs = vec + qs_offset(j8 * BITS, BITS);
    Raw w;
    if constexpr (BITS == 4) {
      const uint16_t *q2 = (const uint16_t *)qs;
      w.codes = (uint32_t)q2[0] | ((uint32_t)q2[1] << 16);
    } else {
      w.codes = *(const uint16_t *)qs;
    }
    w.radius = *(const uint16_t *)vec;
    return w;
  }
  __device__ __forceinline__ void values(const Raw &w, int, const float *cb, float (&o)[8]) const {
    const float r = half_bits_to_float(w.radius);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = r * cb[(w.codes >> (BITS * e)) & ((1 << BITS) - 1)];
  }
};

}  // namespace

// SAT16: fp16 output saturates at +-65504 (as rotate_kernel).
template <int D, bool INVERSE, typename SRC, typename TOUT, bool SAT16>
__global__ void __launch_bounds__(256, RotShape<D>::WAVES) rotate_mfma_kernel(const SRC src, const float *__restrict__ codebook,
                                                             const float *__restrict__ R, TOUT *__restrict__ y,
                                                             int64_t n, float out_scale) {
  using S = RotShape<D>;
  __shared__ __attribute__((aligned(16))) float xs[2][S::VS * S::PITCH];
  __shared__ float cb[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int jt = wave % S::NJ, vh = wave / S::NJ;   // this wave's column tile and vector half
  const int64_t steps = (n + S::VS - 1) / S::VS;

  typename SRC::Raw raw[S::ITEMS];
  auto load = [&](int64_t step) {
#pragma unroll
    for (int u = 0; u < S::ITEMS; ++u) {
      const int item = tid + 256 * u;
      const int64_t v = step * S::VS + item / (D / 8);
      raw[u] = src.load(v < n ? v : n - 1, item % (D / 8));
    }
  };
  auto stage = [&](int b) {
#pragma unroll
    for (int u = 0; u < S::ITEMS; ++u) {
      const int item = tid + 256 * u;
      float o[8];
      src.values(raw[u], item % (D / 8), cb, o);
      chain_put8<D>(&xs[b][(item / (D / 8)) * S::PITCH], item % (D / 8), o);
    }
  };

  int64_t step = blockIdx.x;
  load(step);
  if (codebook != nullptr && tid < 16) cb[tid] = codebook[tid];
  float r[D / 2];
  if constexpr (INVERSE) chain_load_columns<D>(R, 32 * jt + col, half, r);
  else chain_load_rows<D>(R, tid, 32 * jt + col, half, &xs[0][0], r);
  lds_barrier();
  stage(0);
  lds_barrier();
  for (int b = 0; step < steps; step += gridDim.x, b ^= 1) {
    const bool more = step + gridDim.x < steps;
    if (more) load(step + gridDim.x);
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    const float *xr = &xs[b][(32 * vh + col) * S::PITCH + half * (D / 2)];
#pragma unroll
    for (int s4 = 0; s4 < D / 8; ++s4) {
      const float4_t a = *(const float4_t *)(xr + 4 * s4);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = mfma_fma2(a[e], r[4 * s4 + e], acc);
    }
    // the step's outputs, through a buffer over its valid vectors: stores past
    // the last one are dropped, so they need no branch
    const int64_t v0 = step * S::VS;
    const int left = (int)(n - v0 < S::VS ? n - v0 : S::VS);
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(y + v0 * D), (short)0, left * D * (int)sizeof(TOUT), 0x00020000);
    const int off = ((32 * vh + 4 * half) * D + 32 * jt + col) * (int)sizeof(TOUT);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float t = acc[i] * out_scale;
      if (SAT16) t = t > 65504.0f ? 65504.0f : (t < -65504.0f ? -65504.0f : t);
      const int row = mfma32_row(i, 0) * D * (int)sizeof(TOUT);
      if constexpr (sizeof(TOUT) == 4)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, t), out, off + row, 0, 0);
      else
        __builtin_amdgcn_raw_buffer_store_b16(float_to_half_bits(t), out, off + row, 0, 0);
    }
    if (more) stage(b ^ 1);
    lds_barrier();   // (not __syncthreads, which would wait for this step's stores)
  }
}

namespace {

// One resident round of workgroups loops over the steps: R is loaded once per
// workgroup.
template <int D, bool INVERSE, bool SAT16, typename SRC, typename TOUT>
hipError_t launch_one(const SRC &src, const float *cb, const float *R, TOUT *y, int64_t n, float scale,
                      hipStream_t s) {
  const int64_t steps = (n + RotShape<D>::VS - 1) / RotShape<D>::VS, cap = RotShape<D>::WAVES * (int64_t)device_compute_units();
  const int grid = (int)(steps < cap ? steps : cap);
  rotate_mfma_kernel<D, INVERSE, SRC, TOUT, SAT16><<<grid, 256, 0, s>>>(src, cb, R, y, n, scale);
  return hipGetLastError();
}

template <int D, bool INV>
hipError_t rotate_d(const void *x, int xt, const float *R, void *y, int yt, int64_t n, float sc, hipStream_t s) {
  if (xt == 0) {
    const F32Source<D> f{(const float *)x};
    if (yt == 0) return launch_one<D, INV, false>(f, nullptr, R, (float *)y, n, sc, s);
    return launch_one<D, INV, false>(f, nullptr, R, (half_t *)y, n, sc, s);
  }
  const F16Source<D> h{(const half_t *)x};
  if (yt == 0) return launch_one<D, INV, false>(h, nullptr, R, (float *)y, n, sc, s);
  return launch_one<D, INV, false>(h, nullptr, R, (half_t *)y, n, sc, s);
}

template <int D, int BITS>
hipError_t dequant_d(const uint8_t *blocks, int64_t bstride, const float *cb, const float *R, void *y, int yt,
                     int64_t n_outer, int64_t n_inner, hipStream_t s) {
  const BlocksSource<D, BITS> b{blocks, bstride, FastDiv(n_outer > 1 ? (uint32_t)n_inner : 1u), n_outer > 1,
                                (uint32_t)n_inner};
  const int64_t n = n_outer * n_inner;
  if (yt == 0) return launch_one<D, true, false>(b, cb, R, (float *)y, n, 1.0f, s);
  return launch_one<D, true, true>(b, cb, R, (half_t *)y, n, 1.0f, s);
}

}  // namespace

hipError_t launch_rotate_mfma(const void *x, int x_dtype, const float *R, void *y, int y_dtype, int64_t n, int d,
                              int inverse, float out_scale, hipStream_t s) {
  if (d == 128)
    return inverse ? rotate_d<128, true>(x, x_dtype, R, y, y_dtype, n, out_scale, s)
                   : rotate_d<128, false>(x, x_dtype, R, y, y_dtype, n, out_scale, s);
  return inverse ? rotate_d<64, true>(x, x_dtype, R, y, y_dtype, n, out_scale, s)
                 : rotate_d<64, false>(x, x_dtype, R, y, y_dtype, n, out_scale, s);
}

hipError_t launch_rotate_rows_mfma(const float *x, int64_t s_q, int64_t s_h, int64_t s_s, int n_q, int Hq, int n_seq,
                                   const float *R, float *y, int d, float out_scale, hipStream_t s) {
  const int64_t n = (int64_t)n_seq * n_q * Hq;
  if (d == 128)
    return launch_one<128, false, false>(StridedSource<128>{x, s_q, s_h, s_s, n_q, Hq}, nullptr, R, y, n, out_scale,
                                         s);
  return launch_one<64, false, false>(StridedSource<64>{x, s_q, s_h, s_s, n_q, Hq}, nullptr, R, y, n, out_scale, s);
}

hipError_t launch_dequantize(const uint8_t *blocks, int64_t blocks_outer_stride, const float *codebook, int bits,
                             const float *R, void *y, int y_dtype, int64_t y_outer_stride, int64_t n_outer,
                             int64_t n_inner, int d, hipStream_t s) {
  // one launch writes one run of vectors and splits their index with 32-bit
  // arithmetic: several rows together where the output rows follow each other,
  // else (and past 2^32 vectors) a row at a time
  int64_t per = y_outer_stride == n_inner * d ? n_outer : 1;
  if (per > 1 && per * n_inner > 0xFFFFFFFFll - 64) per = n_inner < 0xFFFFFF ? (0xFFFFFFFFll - 64) / n_inner : 1;
  const int64_t ys = y_dtype == 0 ? 4 : 2;
  for (int64_t o = 0; o < n_outer; o += per) {
    const int64_t no = n_outer - o < per ? n_outer - o : per;
    const uint8_t *b = blocks + o * blocks_outer_stride;
    void *yo = (uint8_t *)y + o * y_outer_stride * ys;
    hipError_t e;
    // Few vectors spread over more compute units in the kernel of 8 vectors by
    // 32 columns (32 or 64 vectors by all columns here). Measured crossover
    // (4-bit, fp16 out, replayed graphs, there / here): d = 128 3.0 / 4.7 us
    // for 1 vector, 4.2 / 5.0 for 1024, 5.6 / 4.8 for 1792; d = 64 2.5 / 3.6
    // for 1, 3.0 / 3.7 for 2048, 3.6 / 3.7 for 4096, 3.95 / 3.7 for 4608.
    if (no * n_inner <= (d == 128 ? 1024 : 4096))
      e = launch_dequantize_few(b, blocks_outer_stride, codebook, bits, R, yo, y_dtype, no, n_inner, d, s);
    else if (d == 128 && bits == 4) e = dequant_d<128, 4>(b, blocks_outer_stride, codebook, R, yo, y_dtype, no, n_inner, s);
    else if (d == 128) e = dequant_d<128, 2>(b, blocks_outer_stride, codebook, R, yo, y_dtype, no, n_inner, s);
    else if (bits == 4) e = dequant_d<64, 4>(b, blocks_outer_stride, codebook, R, yo, y_dtype, no, n_inner, s);
    else e = dequant_d<64, 2>(b, blocks_outer_stride, codebook, R, yo, y_dtype, no, n_inner, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace pqkv
