// The FMA-chain rotation on the fp32 matrix cores.
//
// The rotations of this library are one fp32 FMA chain per output over k
// ascending (the reference's arithmetic, csrc/flash_turboquant.cu:132-137).
// v_mfma_f32_32x32x2_f32 computes the same chain: it adds its two products to
// the accumulator one after the other, k = 0 then k = 1, each as one fused
// multiply-add rounded to nearest even, subnormals kept. Checked on the device
// against fmaf over 128-long chains (12.8 M outputs: normal data, exponents
// spread over 2^+-40, products and operands in the subnormal range, fp16
// values): every bit equal. So a chain of these instructions over ascending k
// gives the chain's bits, at 142-154 TFLOP/s measured (all CUs) without vector
// ALU work, where the vector ALU reaches 109-111 TFLOP/s of FMAs alone and
// 62 TFLOP/s in a register-blocked kernel that has to feed them from LDS
// (v_mfma_f32_16x16x4_f32 rounds alike but reaches 126-129 TFLOP/s).
//
// Operand layout (M = N = 32, K = 2): lane l holds A[row l % 32][k = l / 32]
// and B[k = l / 32][col l % 32]; accumulator register r of lane l is
// D[row 8 (r / 4) + 4 (l / 32) + r % 4][col l % 32].
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pqkv_cells.h"

namespace pqkv {

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma_fma2(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
// Row of accumulator register r in the half-wave half = lane / 32.
__device__ __forceinline__ constexpr int mfma32_row(int r, int half) { return 8 * (r >> 2) + 4 * half + (r & 3); }

// A lane's operands of the chain are every second k (k = 2 s + half), so the
// staged vectors keep their even and odd coordinates apart: one 16-byte LDS
// read then feeds four steps. Coordinate k of a D-vector sits at
// (k & 1) D / 2 + k / 2; rows are padded by 16 bytes, which spreads the 16
// rows of one 16-byte read phase over all banks.
template <int D>
struct ChainRow {
  static constexpr int kPitch = D + 4;   // floats
};

// Eight consecutive coordinates 8 j8 .. 8 j8 + 7 into a staged row.
template <int D>
__device__ __forceinline__ void chain_put8(float *row, int j8, const float (&o)[8]) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  *(f4 *)(row + 4 * j8) = f4{o[0], o[2], o[4], o[6]};
  *(f4 *)(row + D / 2 + 4 * j8) = f4{o[1], o[3], o[5], o[7]};
}

// This lane's operands of column j of R (inverse rotation):
// r[s] = R[2 s + half][j].
template <int D>
__device__ __forceinline__ void chain_load_columns(const float *__restrict__ R, int j, int half, float (&r)[D / 2]) {
#pragma unroll
  for (int s = 0; s < D / 2; ++s) r[s] = R[(2 * s + half) * D + j];
}

// This lane's operands of row j of R (forward rotation): r[s] =
// R[j][2 s + half]. A workgroup of 256 threads reads R in runs (a lane reading
// its own row would touch 32 lines per load) and hands the rows out through
// LDS, 64 rows at a time: issue() starts the loads, and spread(), which every
// thread calls, hands the rows out through `lds` (64 staged rows, whose last
// reads are done, behind an LDS barrier of its own, when it returns).
template <int D>
struct ChainRows {
  typedef float f4 __attribute__((ext_vector_type(4)));
  static constexpr int kPieces = 64 * (D / 8) / 256;   // 8-coordinate pieces per thread and pass
  f4 w[D / 64][kPieces][2];
  __device__ __forceinline__ void issue(const float *__restrict__ R, int tid) {
#pragma unroll
    for (int p = 0; p < D / 64; ++p)
#pragma unroll
      for (int u = 0; u < kPieces; ++u) {
        const f4 *src = (const f4 *)(R + (64 * p) * D + 8 * (tid + 256 * u));
        w[p][u][0] = src[0];
        w[p][u][1] = src[1];
      }
  }
  __device__ __forceinline__ void spread(int tid, int j, int half, float *lds, float (&r)[D / 2]) const {
    constexpr int PITCH = ChainRow<D>::kPitch;
#pragma unroll
    for (int p = 0; p < D / 64; ++p) {
      if (p) lds_barrier();
#pragma unroll
      for (int u = 0; u < kPieces; ++u) {
        const int item = tid + 256 * u;
        const float o[8] = {w[p][u][0][0], w[p][u][0][1], w[p][u][0][2], w[p][u][0][3],
                            w[p][u][1][0], w[p][u][1][1], w[p][u][1][2], w[p][u][1][3]};
        chain_put8<D>(lds + (item / (D / 8)) * PITCH, item % (D / 8), o);
      }
      lds_barrier();
      if (j / 64 == p) {
        const float *row = lds + (j % 64) * PITCH + half * (D / 2);
#pragma unroll
        for (int s4 = 0; s4 < D / 8; ++s4) {
          const f4 v = *(const f4 *)(row + 4 * s4);
#pragma unroll
          for (int e = 0; e < 4; ++e) r[4 * s4 + e] = v[e];
        }
      }
    }
    lds_barrier();
  }
};
template <int D>
__device__ __forceinline__ void chain_load_rows(const float *__restrict__ R, int tid, int j, int half, float *lds,
                                                float (&r)[D / 2]) {
  ChainRows<D> rows;
  rows.issue(R, tid);
  rows.spread(tid, j, half, lds, r);
}

}  // namespace pqkv
