// The exact encoder: the FMA-chain rotation of the reference's encode kernel
// (csrc/flash_turboquant.cu:132-137, rot[j] = fp32 FMA chain over k = 0..d-1
// of x[k] * R[j][k]) on the fp32 matrix cores (pqkv_fma_mfma.h, the same
// bits), then the quantiser of csrc/flash_turboquant.cu:141-170.
//
// Work split. A workgroup of four waves takes 32 vectors per step at d = 128,
// 64 at d = 64. Wave w computes the 32 coordinates 32 (w % (d / 32)) .. of 32
// of them, its rows of R in registers for the launch (d / 2 per lane). The
// input is staged in LDS one step ahead (loaded through registers, widened to
// fp32), and the rotated vectors come back through the buffer their input was
// in, to 16 threads per vector for the quantiser: lane tj of a row of 16 takes
// coordinates j = 64 g + 4 tj + i (g < d / 64, i < 4) of VT vectors. Two
// barriers per step; the quantiser of one step and the products of the next
// share the region between them, and three workgroups per compute unit fill
// the matrix cores while others quantise.
//
// Bound by the matrix cores: 2 d^2 flop per vector. Measured (d = 128, 4-bit,
// replayed graphs; in brackets the register-blocked vector-ALU kernel it took
// the place of): 2 097 152 vectors 658 us fp32, 653 us bf16 (1179, 1167), 105
// of the instruction's 145 TFLOP/s; 65 528 vectors 27-28 us (45); 64 vectors
// 9.6 us (14.6); 262 144 keys with signs 162 us (374 fp32, 345 bf16). It was
// the faster one at every count from 1 to 2 097 152, at d = 64 too. Writing
// the next step's products and this step's codes in one block, an instruction
// of each in turn, changed nothing at large counts (654-666 us) and cost
// registers.
//
// Quantiser, per vector, on its 16 lanes:
//   - radius: the reference's 128-slot tree of squares. The step s = 64
//     pairs coordinates j and j + 64 of one thread; the steps s = 32 .. 4
//     pair lanes tj and tj +- s / 4, done as DPP row rotations by 8, 4, 2, 1
//     (after the step by s the lanes' partial sums repeat with period s / 4,
//     so a rotation pairs each lane with a holder of slot t ^ s; IEEE
//     addition commutes); s = 2, 1 pair the thread's own four slots. Then
//     the correctly rounded sqrt (fp64 root rounded once);
//   - index: the switch-point cell table of pqkv_cells.h with the Markstein
//     direction (or a per-coordinate division for radii outside its range),
//     the reference's scan when the table refuses the codebook.
// Output: block_pq4 / block_pq2 vectors (fp16 radius per block) or the
// reference's SoA codes (packed[p] = code(2p) | code(2p+1) << 4) with fp32
// radii, staged in LDS and stored one step later, 16-byte pieces for one
// aligned run of vectors, dwords otherwise. QJL keys add the sign sketch of
// the residual (src/polarquant_kv_cuda/compress_kernel.py:166-175): the
// residuals e = y - r c[code] (fp32 r) go back to LDS and the projections
// P_rot e are a second chain product, P_rot's rows in registers beside R's.
#include <type_traits>

#include "pqkv_cells.h"
#include "pqkv_device.h"
#include "pqkv_fma_mfma.h"
#include "pqkv_launch.h"

namespace pqkv {

namespace {

template <int D>
struct ChainShape {
  static constexpr int NJ = D / 32;              // 32-coordinate tiles
  static constexpr int VS = 32 * (4 / NJ);       // vectors per step
  static constexpr int NG = D / 64;              // 64-coordinate groups per quantiser thread
  static constexpr int VT = VS / 16;             // vectors per quantiser thread
  static constexpr int PITCH = ChainRow<D>::kPitch;
  static constexpr int ITEMS = VS * (D / 8) / 256;   // 8-coordinate input pieces per thread and step
};

// Lane l of a 16-lane row receives lane (l + N) % 16's value (DPP row_ror).
template <int N>
__device__ __forceinline__ float row_ror(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x120 + N, 0xF, 0xF, true));
}

typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(3))) uint32_t lds_u32;

}  // namespace

// OUT: 4 / 2 = block_pq4 / block_pq2 vectors through a's output addressing;
// 0 = SoA codes at a.blocks (d / 2 bytes per vector) and fp32 radii at
// soa_radius, one run of n_inner vectors. nl levels (<= 16). QJL: keys with
// signs, m = d projections.
template <int D, int OUT, typename TIN, bool QJL>
__global__ void __launch_bounds__(256, QJL ? 2 : 3) encode_chain_kernel(const EncodeArgs a, const int nl,
                                                                         float *soa_radius, const FastDiv by_inner) {
  using S = ChainShape<D>;
  constexpr int NG = S::NG, VT = S::VT, VS = S::VS, PITCH = S::PITCH, ITEMS = S::ITEMS;
  constexpr int VB = OUT == 0 ? D / 2 : vector_bytes(D, OUT);   // output bytes per vector
  constexpr int BB = OUT == 0 ? 0 : block_bytes(OUT);
  constexpr int SB = D / 8;                                      // sign bytes per vector
  constexpr int RW = sizeof(TIN) == 4 ? 2 : 1;                   // 16-byte words per input piece
  static_assert(!QJL || OUT != 0, "QJL keys are blocks");
  __shared__ __attribute__((aligned(16))) float xs[2][VS * PITCH];   // a step's input, then its rotation
  __shared__ __attribute__((aligned(16))) float es[QJL ? VS * PITCH : 4];   // residuals, staged order
  __shared__ __attribute__((aligned(16))) uint8_t stage[VS * VB];
  __shared__ __attribute__((aligned(16))) uint8_t sstage[QJL ? VS * SB : 16];
  __shared__ uint2 cells[kECellSlots];
  __shared__ float cb[16], thr[16];
  __shared__ int ucell[16];
  __shared__ int table_ok;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int jt = wave % S::NJ, vh = wave / S::NJ;
  const int tj = tid & 15, tv = tid >> 4;
  const uint32_t n = (uint32_t)(a.n_outer * a.n_inner);
  const uint32_t steps = (n + VS - 1) / VS;
  const TIN *x = (const TIN *)a.x;
  bool use_table = false;   // whether the switch-point table holds (set after its build)

  // ---- input: piece u of this thread is coordinates 8 (item % (D / 8)) .. of
  // vector item / (D / 8) of the step, item = tid + 256 u (past the end: the
  // last vector again) ----
  u32x4 raw[ITEMS][RW];
  auto load = [&](uint32_t s) {
#pragma unroll
    for (int u = 0; u < ITEMS; ++u) {
      const int item = tid + 256 * u;
      const uint32_t v = min(s * VS + item / (D / 8), n - 1);
      const uint32_t vo = a.n_outer > 1 ? by_inner.div(v) : 0u, vi = v - vo * (uint32_t)a.n_inner;
      const u32x4 *p = (const u32x4 *)(x + (int64_t)vo * a.x_outer_stride + (int64_t)vi * D + 8 * (item % (D / 8)));
#pragma unroll
      for (int w = 0; w < RW; ++w) raw[u][w] = p[w];
    }
  };
  auto stage_x = [&](int b) {
#pragma unroll
    for (int u = 0; u < ITEMS; ++u) {
      const int item = tid + 256 * u;
      float o[8];
      if constexpr (sizeof(TIN) == 4) {
        const float4_t f0 = __builtin_bit_cast(float4_t, raw[u][0]), f1 = __builtin_bit_cast(float4_t, raw[u][RW - 1]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o[e] = f0[e];
          o[4 + e] = f1[e];
        }
      } else if constexpr (__is_same(TIN, bf16_t)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t w = raw[u][0][e];
          o[2 * e] = bf16_to_float(w & 0xFFFFu);
          o[2 * e + 1] = bf16_to_float(w >> 16);
        }
      } else {
        const half8_t h = __builtin_bit_cast(half8_t, raw[u][0]);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (float)h[e];
      }
      chain_put8<D>(&xs[b][(item / (D / 8)) * PITCH], item % (D / 8), o);
    }
  };
  // The chains of this wave's 32 staged vectors (columns) against its 32 rows
  // of r: accumulator register i of a lane is row 32 jt + mfma32_row(i, half).
  auto product = [&](const float *src, const float (&r)[D / 2]) {
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    const float *row = src + (32 * vh + col) * PITCH + half * (D / 2);
#pragma unroll
    for (int s4 = 0; s4 < D / 8; ++s4) {
      const float4_t v = *(const float4_t *)(row + 4 * s4);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = mfma_fma2(r[4 * s4 + e], v[e], acc);
    }
    return acc;
  };

  // ---- quantiser: step s's vectors from the rotation in xs[b] into stage ----
  auto quantise = [&](uint32_t s, int b) {
#pragma clang fp contract(off)
#pragma unroll
    for (int u = 0; u < VT; ++u) {
      const int vl = tv + 16 * u;
      float4_t y[NG];
#pragma unroll
      for (int g = 0; g < NG; ++g) y[g] = *(const float4_t *)&xs[b][vl * PITCH + 64 * g + 4 * tj];
      float sq[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p0 = y[0][i] * y[0][i];
        if constexpr (NG == 2) {
          const float p1 = y[NG - 1][i] * y[NG - 1][i];
          sq[i] = p0 + p1;   // tree step s = 64
        } else {
          sq[i] = p0;
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) sq[i] = sq[i] + row_ror<8>(sq[i]);   // s = 32
#pragma unroll
      for (int i = 0; i < 4; ++i) sq[i] = sq[i] + row_ror<4>(sq[i]);   // s = 16
#pragma unroll
      for (int i = 0; i < 4; ++i) sq[i] = sq[i] + row_ror<2>(sq[i]);   // s = 8
#pragma unroll
      for (int i = 0; i < 4; ++i) sq[i] = sq[i] + row_ror<1>(sq[i]);   // s = 4
      const float s2a = sq[0] + sq[2], s2b = sq[1] + sq[3];           // s = 2
      const float tot = s2a + s2b;                                    // s = 1
      const float r = (float)__builtin_sqrt((double)tot);
      int code[NG][4];
      if (use_table) {
        if (markstein_radius(r)) {
          const float inv = r > 1e-30f ? __fdiv_rn(1.0f, r) : 0.0f;
#pragma unroll
          for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) code[g][i] = table_code(cells, dir_markstein(y[g][i], r, inv));
        } else {
#pragma unroll
          for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) code[g][i] = table_code(cells, dir_divided(y[g][i], r));
        }
      } else {
        const bool nz = r > 1e-30f;
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int i = 0; i < 4; ++i) code[g][i] = scan_index_rolled(nz ? __fdiv_rn(y[g][i], r) : 0.0f, cb, nl);
      }
      lds_u8 *sv = (lds_u8 *)stage + vl * VB;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if constexpr (OUT == 0) {
          *(__attribute__((address_space(3))) uint16_t *)(sv + 32 * g + 2 * tj) =
              (uint16_t)(code[g][0] | (code[g][1] << 4) | (code[g][2] << 8) | (code[g][3] << 12));
        } else {
          const int blk = 2 * g + (tj >> 3);
          lds_u8 *bp = sv + blk * BB;
          if constexpr (OUT == 4)
            *(__attribute__((address_space(3))) uint16_t *)(bp + 2 + 2 * (tj & 7)) =
                (uint16_t)(code[g][0] | (code[g][1] << 4) | (code[g][2] << 8) | (code[g][3] << 12));
          else
            bp[2 + (tj & 7)] = (uint8_t)(code[g][0] | (code[g][1] << 2) | (code[g][2] << 4) | (code[g][3] << 6));
          if ((tj & 7) == 0) *(__attribute__((address_space(3))) uint16_t *)bp = radius_half_bits(r);
        }
      }
      if constexpr (OUT == 0) {
        const uint32_t v = s * VS + vl;
        if (tj == 0 && v < n) soa_radius[v] = r;
      }
      if constexpr (QJL) {
        // residuals of coordinates 64 g + 4 tj .. + 3 in the staged order
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          float e[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) e[i] = __builtin_fmaf(-r, cb[code[g][i]], y[g][i]);
          float *row = es + vl * PITCH + 32 * g + 2 * tj;
          *(float2 *)row = make_float2(e[0], e[2]);
          *(float2 *)(row + D / 2) = make_float2(e[1], e[3]);
        }
      }
    }
  };
  // sign bytes of the step into sstage from the projections acc (rows m): bits
  // 4 half .. of byte 4 jt + q are registers 4 q .. 4 q + 3 of the half
  auto signs = [&](const f32x16 &acc) {
    uint32_t w = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t nib = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) nib |= (acc[4 * q + i] >= 0.0f ? 1u : 0u) << i;
      w |= nib << (8 * q + 4 * half);
    }
    w |= (uint32_t)__shfl_xor((int)w, 32, 64);
    if (half == 0) *(lds_u32 *)((lds_u8 *)sstage + (32 * vh + col) * SB + 4 * jt) = w;
  };

  // ---- step s's output from a stage (W bytes per vector) to memory: one
  // run of 16-byte pieces when the outputs are one aligned run, else dwords
  // through the output addressing ----
  auto flush_any = [&](auto wc, uint32_t s, const lds_u8 *stg, uint8_t *outb, uint8_t *const *pages, int64_t stride,
                       bool r16) {
    constexpr int W = decltype(wc)::value;
    const uint32_t v0 = s * VS;
    const int nv = (int)min(n - v0, (uint32_t)VS);
    if (r16) {
      const int nbytes = nv * W;
      uint8_t *base = outb + (int64_t)v0 * W;
#pragma unroll
      for (int it = 0; it < (VS * W / 16 + 255) / 256; ++it) {
        const int p = tid + 256 * it;
        if (16 * p + 16 <= nbytes) {
          *(u32x4 *)(base + 16 * p) = *(const __attribute__((address_space(3))) u32x4 *)(stg + 16 * p);
        } else if (16 * p < nbytes) {
          for (int c = 0; c < 4 && 16 * p + 4 * c < nbytes; ++c)
            *(uint32_t *)(base + 16 * p + 4 * c) = *(const lds_u32 *)(stg + 16 * p + 4 * c);
        }
      }
      return;
    }
    constexpr int DW = W / 4;
#pragma unroll
    for (int it = 0; it < (VS * DW + 255) / 256; ++it) {
      const int q = tid + 256 * it;
      const int vl = q / DW, c = q - vl * DW;
      if (q < VS * DW && vl < nv) {
        const uint32_t v = v0 + vl;
        const uint32_t vo = a.n_outer > 1 ? by_inner.div(v) : 0u, vi = v - vo * (uint32_t)a.n_inner;
        *(uint32_t *)(encode_out_addr(a, outb, pages, stride, vo, vi, W) + 4 * c) = *(const lds_u32 *)(stg + vl * W + 4 * c);
      }
    }
  };
  const bool run16 = a.n_outer <= 1 && a.pages == nullptr && ((uintptr_t)a.blocks & 15) == 0;
  const bool srun16 = QJL && a.n_outer <= 1 && a.qjl_pages == nullptr && ((uintptr_t)a.qjl & 15) == 0;
  auto flush = [&](uint32_t s) {
    flush_any(std::integral_constant<int, VB>{}, s, (const lds_u8 *)stage, a.blocks, a.pages, a.blocks_outer_stride,
              run16);
  };
  auto flush_signs = [&](uint32_t s) {
    if constexpr (QJL)
      flush_any(std::integral_constant<int, SB>{}, s, (const lds_u8 *)sstage, a.qjl, a.qjl_pages, a.qjl_outer_stride,
                srun16);
  };

  // ---- set-up: the first step's input, R and P_rot are in flight while the
  // centroid table is built (its barriers wait for LDS only) ----
  uint32_t s = blockIdx.x;
  const float cbv = tid < nl ? a.codebook[tid] : 0.0f;   // first, so its LDS copy waits for it alone
  load(s);
  ChainRows<D> rows;
  rows.issue(a.R, tid);
  if (tid < 16) cb[tid] = cbv;
  lds_barrier();
  build_cell_table<256>(cb, nl, tid, cells, thr, ucell, &table_ok);
  use_table = table_ok != 0;
  float r[D / 2], p[QJL ? D / 2 : 1];
  rows.spread(tid, 32 * jt + col, half, &xs[0][0], r);
  if constexpr (QJL) chain_load_rows<D>(a.p_rot, tid, 32 * jt + col, half, &xs[0][0], p);
  stage_x(0);
  lds_barrier();

  // ---- pipeline. Iteration k (buffer b = k & 1): load step k + 1's input,
  // products of step k from xs[b]; [barrier: xs[b] read, step k - 1's blocks
  // staged] rotation into xs[b], step k + 1's input into xs[b ^ 1] (whose
  // rotation of step k - 1 the quantiser has read), step k - 1's blocks to
  // memory; [barrier] quantise step k from xs[b]. With QJL the projections of
  // step k follow its quantiser behind a barrier of their own, and its signs
  // go out with its blocks. ----
  for (int b = 0; s < steps; s += gridDim.x, b ^= 1) {
    const bool more = s + gridDim.x < steps;
    if (more) load(s + gridDim.x);
    const f32x16 acc = product(xs[b], r);
    lds_barrier();
    float *dst = xs[b] + (32 * vh + col) * PITCH + 32 * jt + 4 * half;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *(float4_t *)(dst + 8 * q) = float4_t{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    if (more) stage_x(b ^ 1);
    if (s != blockIdx.x) {
      flush(s - gridDim.x);
      flush_signs(s - gridDim.x);
    }
    lds_barrier();
    quantise(s, b);
    if constexpr (QJL) {
      lds_barrier();
      signs(product(es, p));
    }
  }
  lds_barrier();
  flush(s - gridDim.x);
  flush_signs(s - gridDim.x);
}

// The kernel applies to inputs it can read in 16-byte pieces and outputs it
// can write in dwords: 16-byte aligned x rows, R and P_rot, 4-byte aligned
// blocks, signs and row strides (pages are 16-byte aligned by contract), fewer
// than 2^32 vectors.
bool chain_encode_ok(const EncodeArgs &a, int x_dtype) {
  const int64_t es = x_dtype == 0 ? 4 : 2;
  const int64_t n = a.n_outer * a.n_inner;
  const bool qjl = a.qjl != nullptr || a.qjl_pages != nullptr;
  if (a.d != 64 && a.d != 128) return false;
  if (n <= 0 || n > ((int64_t)1 << 32) - 1024) return false;
  if ((uintptr_t)a.x % 16 || (uintptr_t)a.R % 16) return false;
  if (a.n_outer > 1 && (a.x_outer_stride * es) % 16) return false;
  if (a.pages == nullptr && ((uintptr_t)a.blocks % 4 || (a.n_outer > 1 && a.blocks_outer_stride % 4))) return false;
  if (qjl) {
    if (a.m != a.d || a.p_rot == nullptr || (uintptr_t)a.p_rot % 16) return false;
    if (a.qjl_pages == nullptr && ((uintptr_t)a.qjl % 4 || (a.n_outer > 1 && a.qjl_outer_stride % 4))) return false;
  }
  return true;
}

namespace {

// One resident round of workgroups loops over the steps: R and the centroid
// table are set up once per workgroup.
int chain_grid(int64_t n, int d, bool qjl) {
  const int vs = d == 128 ? ChainShape<128>::VS : ChainShape<64>::VS;
  const int64_t steps = (n + vs - 1) / vs, cap = (qjl ? 2 : 3) * (int64_t)device_compute_units();
  return (int)(steps < cap ? steps : cap);
}

template <int D, int OUT, bool QJL>
void launch_chain(const EncodeArgs &a, int x_dtype, int nl, float *soa_radius, hipStream_t s) {
  const int grid = chain_grid(a.n_outer * a.n_inner, D, QJL);
  const FastDiv by_inner(a.n_outer > 1 ? (uint32_t)a.n_inner : 1u);
  if (x_dtype == 0) encode_chain_kernel<D, OUT, float, QJL><<<grid, 256, 0, s>>>(a, nl, soa_radius, by_inner);
  else if constexpr (OUT != 0) {
    if (x_dtype == 1) encode_chain_kernel<D, OUT, half_t, QJL><<<grid, 256, 0, s>>>(a, nl, soa_radius, by_inner);
    else encode_chain_kernel<D, OUT, bf16_t, QJL><<<grid, 256, 0, s>>>(a, nl, soa_radius, by_inner);
  }
}

}  // namespace

hipError_t launch_encode_chain(const EncodeArgs &a, int x_dtype, hipStream_t s) {
  const int nl = 1 << a.bits;
  const bool qjl = a.qjl != nullptr || a.qjl_pages != nullptr;
#define PQKV_EC(DD, BB)                                             \
  do {                                                              \
    if (qjl) launch_chain<DD, BB, true>(a, x_dtype, nl, nullptr, s); \
    else launch_chain<DD, BB, false>(a, x_dtype, nl, nullptr, s);    \
  } while (0)
  if (a.d == 128 && a.bits == 4) PQKV_EC(128, 4);
  else if (a.d == 128) PQKV_EC(128, 2);
  else if (a.bits == 4) PQKV_EC(64, 4);
  else PQKV_EC(64, 2);
#undef PQKV_EC
  return hipGetLastError();
}

bool chain_soa_ok(const float *x, const float *R, const uint8_t *packed, int64_t n, int d) {
  return (d == 64 || d == 128) && n > 0 && n <= ((int64_t)1 << 32) - 1024 && (uintptr_t)x % 16 == 0 &&
         (uintptr_t)R % 16 == 0 && (uintptr_t)packed % 4 == 0;
}

hipError_t launch_encode_soa_chain(const float *x, const float *R, const float *codebook, int n_levels, float *radius,
                                   uint8_t *packed, int64_t n, int d, hipStream_t s) {
  EncodeArgs a{};
  a.x = x;
  a.x_outer_stride = 0;
  a.R = R;
  a.codebook = codebook;
  a.blocks = packed;
  a.n_outer = 1;
  a.n_inner = n;
  a.d = d;
  if (d == 128) launch_chain<128, 0, false>(a, 0, n_levels, radius, s);
  else launch_chain<64, 0, false>(a, 0, n_levels, radius, s);
  return hipGetLastError();
}

}  // namespace pqkv
