// Prefill attention over pre-decoded tiles, for launches whose query rows
// would decode every tile of the cache many times (prefill_mfma_kernel in
// pqkv_prefill.hip decodes each 64-token tile once per 256 query rows, and
// that stage, longer than its matrix stage, set its pace).
//
// Two kernels. plane_decode_kernel turns each 64-token tile of a stream into a
// record: the keys' and values' centroids as fp16 hi / lo planes in the exact
// order of the matrix operands, and fp32 radii (64.5 KB at d = 128).
// prefill_planes_kernel then copies records to LDS (buffer-to-LDS loads, no
// registers, no arithmetic) and runs the same online-softmax attention, so a
// tile is decoded once per call instead of once per 256 rows.
//
// Attention: a workgroup of 8 waves takes 256 query rows of one (batch, kv
// head), 32 per wave; row r is query token r / G, head r % G. Products are
// v_mfma_f32_16x16x32_f16. Scores are computed transposed, S^T[token][row] =
// K^ . Q^T: accumulator register i of lane l is token 4 (l / 16) + i of row l %
// 16, and with the value planes' tokens in the same order those registers are
// the A operand of P . V^: the weights never leave the lane.
// Precision is that of prefill_mfma_kernel: every fp32 operand split hi / lo,
// three products hi.hi + hi.lo + lo.hi in one fp32 accumulator, planes and
// queries scaled by 2^6 so that the lo parts stay normal numbers.
//
// Schedule: two groups of four waves, a wave of each on every SIMD. A tile
// takes two stages per wave, X(it) = values of tile it - 1 and scores of tile
// it (192 products, 3072 cycles of the matrix core at d = 128) and Y(it) =
// softmax of tile it. Group 1 runs one stage behind group 0, with a barrier
// after each stage, so one wave of a SIMD has the matrix core while the other
// has the vector ALU, and X sets the pace. Group 1 copies tiles in its Y
// stage: K(it + 1) and V(it) in Y(it - 1) (stage 2 it: their buffers were last
// read in stage 2 it - 1), complete before the barrier that ends its X(it)
// (stage 2 it + 1), read from stage 2 it + 2 on.
//
// splits > 1 (fewer workgroups than compute units): workgroup (row block,
// split) takes its share of the row block's tiles and writes an unnormalised
// partial; prefill_merge_kernel joins them.
//
// Bound by the matrix stage: 64 query / 8 kv heads, 2048 tokens against 131 072
// (26.6 TFLOP of products) take 16.9-18.5 ms box to box, 18.85-20.4 for decoding
// per row block; at 18.5 ms 1440 TFLOP/s, the matrix cores busy 71 % of the
// cycles and a quarter of the wave cycles waiting (the barriers between the
// groups' stages), at 1.89 GHz where short kernels run at 2.1-2.4, memory at 0.12
// TB/s and no bank conflicts. v_mfma_f32_16x16x32_f16 alone reaches 2390 TFLOP/s
// in a burst of 0.4 ms, a library product of two 8192 x 8192 fp16 matrices 1323.
// v_mfma_f32_32x32x16_f16 products (half the operand reads) take 18.6 ms where
// these take 16.9. The decode kernel takes 0.25 ms of it (1.10 GB of records, 4.4
// TB/s).
#include <type_traits>

#include "pqkv_device.h"
#include "pqkv_launch.h"
#include "pqkv_prefill.h"

namespace pqkv {

namespace {

constexpr int kPRows = 32 * kPW;               // query rows per workgroup
constexpr int kGroup = 32;                     // streams whose workgroups run side by side

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) const half8_t lds_chalf8;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int D>
struct PlaneRec {
  static constexpr int KS = D / 32;            // k-steps of the score product
  static constexpr int NT = D / 16;            // coordinate tiles of the value product
  static constexpr int KSEG = 4 * KS * 2;      // 1 KB segments (token tile, k-step, plane): 64 lanes x 16 bytes
  static constexpr int VSEG = NT * 2 * 2;      // (coordinate tile, k-step, plane)
  static constexpr int KBYTES = KSEG * 1024, VBYTES = VSEG * 1024;
  static constexpr int RAD = KBYTES + VBYTES;  // 64 key radii (x 2^-12), then 64 value radii, fp32
  static constexpr int BYTES = RAD + 512;
  __host__ __device__ static constexpr int kseg(int tt, int ks, int plane) { return (tt * KS + ks) * 2 + plane; }
  __host__ __device__ static constexpr int vseg(int nb, int kk, int plane) { return (nb * 2 + kk) * 2 + plane; }
};

__device__ __forceinline__ uint32_t load_u32_any(const uint8_t *p) {   // 2-byte aligned
  return (uint32_t)((const uint16_t *)p)[0] | ((uint32_t)((const uint16_t *)p)[1] << 16);
}

}  // namespace

// ---------------------------------------------------------------------------
// One 64-token tile of one stream per workgroup. Keys: thread item (token
// tile, k-step, lane) is eight coordinates of a token, one code word. Values:
// item (coordinate tile, k-step, lane) is one coordinate of eight tokens, from
// the tile's code bytes in LDS. Tokens past the end get radius 0.
template <int D, int KB, int VB>
__global__ void __launch_bounds__(256) plane_decode_kernel(const PrefillArgs a, uint8_t *planes, int64_t stream_bytes,
                                                           int stream0) {
  using P = PlaneRec<D>;
  constexpr int VBYTES = vector_bytes(D, VB), VP = VBYTES + 4;   // LDS row pitch (odd number of dwords mod banks)
  __shared__ __attribute__((aligned(16))) uint8_t vraw[kPT * VP];
  __shared__ uint32_t lk[16], lv[16];          // code -> hi | lo << 16
  const int tid = threadIdx.x;
  const int t0 = blockIdx.x * kPT;
  const int bh = stream0 + blockIdx.y;
  const int b = bh / a.n_heads, hl = bh - b * a.n_heads;
  const int h = a.listed ? a.heads[hl] : hl;
  uint8_t *rec = planes + (int64_t)blockIdx.y * stream_bytes + (int64_t)blockIdx.x * P::BYTES;
  const uint8_t *kp, *vp;                      // the tile's first vectors
  if (a.k_pages != nullptr) {
    const int pg = t0 >> a.page_shift, rel = t0 & ((1 << a.page_shift) - 1);
    const int64_t at = (int64_t)(b * a.Hkv + h) * a.max_pages + pg;
    kp = a.k_pages[at] + (int64_t)rel * vector_bytes(D, KB);
    vp = a.v_pages[at] + (int64_t)rel * VBYTES;
  } else {
    kp = a.k_cache + b * a.k_batch_stride + (a.listed ? a.k_head_off[hl] : h * a.k_head_stride) + (int64_t)t0 * a.k_tok_stride;
    vp = a.v_cache + b * a.v_batch_stride + (a.listed ? a.v_head_off[hl] : h * a.v_head_stride) + (int64_t)t0 * a.v_tok_stride;
  }
  const int64_t kts = a.k_pages != nullptr ? vector_bytes(D, KB) : a.k_tok_stride;
  const int64_t vts = a.k_pages != nullptr ? VBYTES : a.v_tok_stride;
  const int left = a.S - t0;                   // valid tokens of the tile (>= 1)
  if (tid < 32) {
    const bool isv = tid >= 16;
    const int c = tid & 15, levels = 1 << (isv ? VB : KB);
    half_t hi, lo;
    split2(c < levels ? (isv ? a.v_cb : a.k_cb)[h * a.cb_head_stride + c] * kPlaneScale : 0.0f, &hi, &lo);
    (isv ? lv : lk)[c] = (uint32_t)__builtin_bit_cast(uint16_t, hi) | ((uint32_t)__builtin_bit_cast(uint16_t, lo) << 16);
  }
  for (int q = tid; q < kPT * (VBYTES / 4); q += 256) {
    const int t = q / (VBYTES / 4), c = q - t * (VBYTES / 4);
    *(uint32_t *)(vraw + t * VP + 4 * c) = t < left ? load_u32_any(vp + t * vts + 4 * c) : 0u;
  }
  if (tid < kPT) {
    const bool ok = tid < left;
    ((float *)(rec + P::RAD))[tid] = ok ? half_bits_to_float(*(const uint16_t *)(kp + tid * kts)) * kScoreUnscale : 0.0f;
    ((float *)(rec + P::RAD))[kPT + tid] = ok ? half_bits_to_float(*(const uint16_t *)(vp + tid * vts)) : 0.0f;
  }
  uint32_t kw[P::KS * 4 * 64 / 256];           // this thread's key words, loaded before the barrier
#pragma unroll
  for (int u = 0; u < P::KS * 4 * 64 / 256; ++u) {
    const int item = tid + 256 * u, lane = item & 63, seg = item >> 6;
    const int t = 16 * (seg / P::KS) + (lane & 15), j8 = 4 * (seg % P::KS) + (lane >> 4);
    const uint8_t *qs = kp + t * kts + qs_offset(j8 * KB, KB);
    kw[u] = t >= left ? 0u : KB == 4 ? load_u32_any(qs) : (uint32_t)*(const uint16_t *)qs;
  }
  __syncthreads();
  auto put = [&](uint8_t *seg_hi, int lane, const uint32_t (&e)[8]) {
    u32x4 hi, lo;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      hi[k] = (e[2 * k] & 0xFFFFu) | (e[2 * k + 1] << 16);
      lo[k] = (e[2 * k] >> 16) | (e[2 * k + 1] & 0xFFFF0000u);
    }
    *(u32x4 *)(seg_hi + 16 * lane) = hi;
    *(u32x4 *)(seg_hi + 1024 + 16 * lane) = lo;
  };
#pragma unroll
  for (int u = 0; u < P::KS * 4 * 64 / 256; ++u) {
    const int item = tid + 256 * u, lane = item & 63, seg = item >> 6;
    uint32_t e[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) e[k] = lk[(kw[u] >> (KB * k)) & ((1 << KB) - 1)];
    put(rec + P::kseg(seg / P::KS, seg % P::KS, 0) * 1024, lane, e);
  }
#pragma unroll
  for (int u = 0; u < P::NT * 2 * 64 / 256; ++u) {
    const int item = tid + 256 * u, lane = item & 63, seg = item >> 6;
    const int nb = seg >> 1, kk = seg & 1, c = 16 * nb + (lane & 15);
    // slot k of lane group g = lane / 16 holds token 32 kk + 16 (k / 4) + 4 g + k % 4
    const uint8_t *src = vraw + (32 * kk + 4 * (lane >> 4)) * VP + qs_offset(c / (8 / VB), VB);
    const int sh = VB * (c % (8 / VB));
    uint32_t e[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) e[k] = lv[(src[(16 * (k >> 2) + (k & 3)) * VP] >> sh) & ((1 << VB) - 1)];
    put(rec + P::KBYTES + P::vseg(nb, kk, 0) * 1024, lane, e);
  }
}

// ---------------------------------------------------------------------------
// GG (llama.cpp's flash_attn_ext): queries and output [sequence][token][head],
// an additive fp16 mask in the place of the causal rule, and the operands'
// powers of two follow the data (queries per row, weights times radii by the
// largest value radius so far), since they are fp32 there and the results too. 512
// query rows (32 query / 8 kv heads, d = 128) against 4096 tokens: 143 us a
// call, 461 for the split decode kernel, which streams the cache once per row;
// the error against 64 bits is 6.4e-7 (8.1e-7 there). 123 us of it are this
// kernel, 845 TFLOP/s executed, its waves waiting for 44 % of their cycles (16
// tiles a workgroup: set-up, mask loads, barriers); the 40 bytes a lane spills at
// d = 128 buy the tile sums (1-2 %).
template <int D, bool GG>
__global__ void __launch_bounds__(kPW * 64, 1)
    prefill_planes_kernel(const PrefillArgs a, const uint8_t *planes, int64_t stream_bytes, int stream0, int ns) {
  using P = PlaneRec<D>;
  constexpr int KS = P::KS, NT = P::NT;
  constexpr int RT = 2;                        // 16-row tiles per wave
  const int qtiles = a.qtiles, splits = a.splits;
  constexpr int AHEAD = 1;
  __shared__ __attribute__((aligned(16))) uint8_t kt[2][P::KBYTES], vt[2][P::VBYTES];
  // key and value radii of tiles it % 3 (read in both groups' Y(it), so a
  // third buffer keeps tile it + 2's copy off them)
  __shared__ __attribute__((aligned(16))) float rads[3][2 * kPT];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int group = wave >= kPW / 2 ? 1 : 0, gw = wave & (kPW / 2 - 1);
  const int G = a.G;
  // Groups of kGroup streams, one after the other, in each of them the streams
  // fastest: with a multiple of eight of them the workgroups of one stream land
  // on one XCD and share its tiles in that L2, and a round of workgroups reads
  // few streams' tiles (a workgroup on each of 256 streams reads 4 TB/s in all: 24
  // row blocks of 256 streams against 2000 tokens, 32 query / 8 kv heads, d = 128,
  // 7.23 ms without groups, 6.40 with them). The longest row blocks of a group
  // (the last ones, with a causal mask) come first.
  const int per = kGroup * qtiles * splits, group0 = (int)blockIdx.x / per * kGroup;
  const int in_group = (int)blockIdx.x - group0 * qtiles * splits, members = min(kGroup, ns - group0);
  const int rest = in_group / members, sl = group0 + in_group - rest * members;
  const int sp = rest % splits, qtile = qtiles - 1 - rest / splits;
  const int bh = stream0 + sl;
  const int b = bh / a.n_heads, hl = bh - b * a.n_heads;
  const int h = a.listed ? a.heads[hl] : hl;
  const int q0 = qtile * a.qt;
  const int q_last = min(a.Sq, q0 + a.qt) - 1;
  const int kv_end = a.causal ? min(a.S, a.q_start + q_last + 1) : a.S;
  const int all = (kv_end + kPT - 1) / kPT;
  const int it0 = share_begin(all, sp, splits), it1 = share_begin(all, sp + 1, splits);

  const uint8_t *stream = planes + (int64_t)sl * stream_bytes;
  const __amdgpu_buffer_rsrc_t res =
      __builtin_amdgcn_make_buffer_rsrc((void *)stream, (short)0, (int)stream_bytes, 0x00020000);

  // queries as the B operand: column col of row tile rt = row 32 wave + 16 rt +
  // col; step ks, slot k = 8 grp + i is coordinate 32 ks + 8 grp + i
  half8_t qh[RT][KS], ql[RT][KS];
  int row_pos[RT];
  float q_un[RT];                              // GG: undoes the row's query scale (beside the radii's 2^-12)
  const uint16_t *mrow[RT];                    // GG: the row's mask
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int row = 32 * wave + 16 * rt + col;
    const int tok = q0 + row / G, head = row % G;
    const bool row_ok = row < a.qt * G && tok < a.Sq;
    row_pos[rt] = a.q_start + tok;
    const int64_t qrow = GG ? ((int64_t)b * a.Sq + (row_ok ? tok : 0)) * a.Hq + h * G + head
                            : (int64_t)(b * a.Hq + h * G + head) * a.Sq + (row_ok ? tok : 0);
    const float *qr = a.q + qrow * D;
    float q_sc = 1.0f;
    if constexpr (GG) {
      float amax = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(qr[32 * ks + 8 * grp + i]));
      // the row's largest value to [2^8, 2^9) (as it is if zero, subnormal or not finite)
      const int ex = (int)(__builtin_bit_cast(uint32_t, rows_max(amax)) >> 23);
      const int sh = ex == 0 || ex == 255 ? 0 : min(135 - ex, 100);
      q_sc = __builtin_ldexpf(1.0f, sh);
      q_un[rt] = __builtin_ldexpf(kPlaneScale, -sh);
      mrow[rt] = a.mask + b * a.mask_seq_stride + (row_ok ? tok : 0) * a.mask_row_stride;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const float4_t x0 = *(const float4_t *)(qr + 32 * ks + 8 * grp), x1 = *(const float4_t *)(qr + 32 * ks + 8 * grp + 4);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        half_t vh, vl;
        const float x = row_ok ? (i < 4 ? x0[i & 3] : x1[i & 3]) : 0.0f;
        split2(GG ? x * q_sc : x, &vh, &vl);
        qh[rt][ks][i] = vh;
        ql[rt][ks][i] = vl;
      }
    }
  }

  float m_run[RT], l_run[RT];
  float4_t oacc[RT][NT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    m_run[rt] = -INFINITY;
    l_run[rt] = 0.0f;
#pragma unroll
    for (int nb = 0; nb < NT; ++nb) oacc[rt][nb] = (float4_t){0.f, 0.f, 0.f, 0.f};
  }
  float4_t sacc[RT][4];
  half8_t ph[RT][2], pl[RT][2];
  u32x2 mk[RT][4];                             // GG: the lane's mask values of the tile
  int vexp = -40;                              // GG: weights times radii carry 2^-vexp

  // Copies of 1 KB segments: wave w of NW takes every NW-th (a compile-time
  // count). The radii come with the keys, as Y(it) reads them before V(it)
  // has to be there.
  auto copy_seg = [&](uint8_t *dst, int at, int sg) {
    at = __builtin_amdgcn_readfirstlane(at);   // (uniform: a scalar offset)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(res, (lds_void *)(dst + 1024 * sg), 16, 16 * lane, at + 1024 * sg, 0, 0);
  };
  auto copy_k = [&](auto nwc, int it, int w) {
    constexpr int NW = decltype(nwc)::value;
#pragma unroll
    for (int j = 0; j < P::KSEG / NW; ++j) copy_seg(kt[it & 1], it * P::BYTES, w + NW * j);
    if (w == 0 && lane < 32) copy_seg((uint8_t *)rads + 512 * (it % 3), it * P::BYTES + P::RAD, 0);
  };
  auto copy_v = [&](auto nwc, int it, int w) {
    constexpr int NW = decltype(nwc)::value;
#pragma unroll
    for (int j = 0; j < P::VSEG / NW; ++j) copy_seg(vt[it & 1], it * P::BYTES + P::KBYTES, w + NW * j);
  };

  // GG: four tokens' values of each row and 16-token group (S is a multiple of
  // four; the groups past it read the last four and are masked by their position)
  auto load_mask = [&](int it) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const int t = min(it * kPT + 16 * tt + 4 * grp, a.S - 4);
        mk[rt][tt] = a.mask != nullptr ? *(const u32x2 *)(mrow[rt] + t) : (u32x2){0u, 0u};
      }
  };

  // The operands of a product step are read AHEAD steps before it (the fence
  // keeps them there), so that the LDS latency hides behind 6 AHEAD products.
  auto scores = [&](int it) {
    const uint8_t *t = kt[it & 1] + 16 * lane;
    auto op = [&](int n, int plane) { return *(lds_chalf8 *)(t + P::kseg(n / KS, n % KS, plane) * 1024); };
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) sacc[rt][tt] = (float4_t){0.f, 0.f, 0.f, 0.f};
    half8_t ah[AHEAD + 1], al[AHEAD + 1];
#pragma unroll
    for (int n = 0; n < AHEAD; ++n) {
      ah[n] = op(n, 0);
      al[n] = op(n, 1);
    }
#pragma unroll
    for (int n = 0; n < 4 * KS; ++n) {
      const int tt = n / KS, ks = n % KS, c = n % (AHEAD + 1);
      if (n + AHEAD < 4 * KS) {
        ah[(n + AHEAD) % (AHEAD + 1)] = op(n + AHEAD, 0);
        al[(n + AHEAD) % (AHEAD + 1)] = op(n + AHEAD, 1);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        if (!GG) sacc[rt][tt] = mfma16(ah[c], qh[rt][ks], sacc[rt][tt]);
        sacc[rt][tt] = mfma16(al[c], qh[rt][ks], sacc[rt][tt]);
        sacc[rt][tt] = mfma16(ah[c], ql[rt][ks], sacc[rt][tt]);
        if (GG) sacc[rt][tt] = mfma16(ah[c], qh[rt][ks], sacc[rt][tt]);   // the small products first
      }
    }
  };
  auto values = [&](int it) {
    const uint8_t *t = vt[it & 1] + 16 * lane;
    auto op = [&](int n, int plane) { return *(lds_chalf8 *)(t + P::vseg(n >> 1, n & 1, plane) * 1024); };
    half8_t bh[AHEAD + 1], bl[AHEAD + 1];
    float4_t part[RT];
#pragma unroll
    for (int n = 0; n < AHEAD; ++n) {
      bh[n] = op(n, 0);
      bl[n] = op(n, 1);
    }
#pragma unroll
    for (int n = 0; n < 2 * NT; ++n) {
      const int nb = n >> 1, kk = n & 1, c = n % (AHEAD + 1);
      if (n + AHEAD < 2 * NT) {
        bh[(n + AHEAD) % (AHEAD + 1)] = op(n + AHEAD, 0);
        bl[(n + AHEAD) % (AHEAD + 1)] = op(n + AHEAD, 1);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        // GG, whose results stay fp32: the tile's sum first, so that the long
        // accumulation rounds once per tile instead of six times
        float4_t &o = GG ? part[rt] : oacc[rt][nb];
        if (GG && kk == 0) o = (float4_t){0.f, 0.f, 0.f, 0.f};
        if (!GG) o = mfma16(ph[rt][kk], bh[c], o);
        o = mfma16(ph[rt][kk], bl[c], o);
        o = mfma16(pl[rt][kk], bh[c], o);
        if (GG) o = mfma16(ph[rt][kk], bh[c], o);
        if (GG && kk == 1) oacc[rt][nb] += o;
      }
    }
  };
  auto softmax = [&](int it) {
    const int t0 = it * kPT;
    const float *rk = rads[it % 3] + 4 * grp, *rv = rk + kPT;
    float shrink = 1.0f, v_sc = 1.0f;
    if constexpr (GG) {
      float rmax = 0.0f;
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int i = 0; i < 4; ++i) rmax = fmaxf(rmax, rv[16 * tt + i]);
      // the tile's largest radius below 2^14 (the same in every lane)
      const int ex = (int)(__builtin_bit_cast(uint32_t, rows_max(rmax)) >> 23) & 0xFF;
      const int need = max(vexp, __builtin_amdgcn_readfirstlane(ex) - 127 - 13);
      shrink = __builtin_ldexpf(1.0f, vexp - need);
      vexp = need;
      v_sc = __builtin_ldexpf(1.0f, -vexp);
    }
    const bool need_mask = t0 + kPT > a.S || (a.causal && t0 + kPT - 1 > a.q_start + q0);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float s[4][4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const float4_t r4 = *(const float4_t *)(rk + 16 * tt);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[tt][i] = sacc[rt][tt][i] * r4[i];
          if constexpr (GG)   // the mask in the exp2 domain
            s[tt][i] = __builtin_fmaf(half_bits_to_float((uint16_t)(mk[rt][tt][i >> 1] >> (16 * (i & 1)))),
                                      1.4426950408889634f, s[tt][i] * q_un[rt]);
        }
      }
      if (need_mask) {
        const int last = a.causal ? min(a.S - 1, row_pos[rt]) : a.S - 1;   // last token this row sees
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (t0 + 16 * tt + 4 * grp + i > last) s[tt][i] = -INFINITY;
      }
      float cmax = s[0][0];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int i = 0; i < 4; ++i) cmax = fmaxf(cmax, s[tt][i]);
      cmax = rows_max(cmax);
      const float mnew = fmaxf(m_run[rt], cmax);
      // a row with no visible token so far (splits) keeps weight 0
      const float ref = mnew == -INFINITY ? 0.0f : mnew;
      const float alpha = __builtin_amdgcn_exp2f(m_run[rt] - ref);
      m_run[rt] = mnew;
      float psum = 0.0f;
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const float4_t r4 = *(const float4_t *)(rv + 16 * tt);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = __builtin_amdgcn_exp2f(s[tt][i] - ref);
          psum += p;
          half_t vh, vl;
          split2(GG ? p * (r4[i] * v_sc) : p * r4[i], &vh, &vl);
          ph[rt][tt >> 1][4 * (tt & 1) + i] = vh;
          pl[rt][tt >> 1][4 * (tt & 1) + i] = vl;
        }
      }
      l_run[rt] = l_run[rt] * alpha + psum;
      const float fade = GG ? alpha * shrink : alpha;
      if (__builtin_amdgcn_ballot_w64(fade != 1.0f) != 0) {
        float f[4];
        per_row(fade, grp, f);
#pragma unroll
        for (int nb = 0; nb < NT; ++nb)
#pragma unroll
          for (int i = 0; i < 4; ++i) oacc[rt][nb][i] *= f[i];
      }
    }
  };

  auto wait_copies = [] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  if (it0 < it1) {
    copy_k(std::integral_constant<int, kPW>{}, it0, wave);
    wait_copies();
    barrier();
    // X(it1), values alone, stands after the loop: with it inside, behind a
    // condition, the scores would count as live across iterations
    auto x_stage = [&](int it) {
      if constexpr (GG) load_mask(it);          // there by softmax(it)
      __builtin_amdgcn_s_setprio(1);
      if (it > it0) values(it - 1);
      __builtin_amdgcn_sched_barrier(0);
      scores(it);
      __builtin_amdgcn_s_setprio(0);
    };
    if (group == 0) {
      for (int it = it0; it < it1; ++it) {
        x_stage(it);                            // stage 2 (it - it0)
        barrier();
        softmax(it);
        barrier();
      }
      values(it1 - 1);
      barrier();
      barrier();
    } else {
      auto copies = [&](int it) {               // K(it + 1) and V(it)
        if (it + 1 < it1) copy_k(std::integral_constant<int, kPW / 2>{}, it + 1, gw);
        if (it < it1) copy_v(std::integral_constant<int, kPW / 2>{}, it, gw);
      };
      copies(it0);                              // stage 0
      barrier();
      for (int it = it0; it < it1; ++it) {
        x_stage(it);                            // stage 2 (it - it0) + 1
        wait_copies();
        barrier();
        copies(it + 1);
        softmax(it);
        barrier();
      }
      values(it1 - 1);
      barrier();
    }
  }

  // ---- normalise and write o_rot, or the split's partial ----
  // (partial rows: [stream of the pass][row block][row][split])
  const int64_t prow0 = ((int64_t)sl * qtiles + qtile) * kPRows;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const float l = rows_sum(l_run[rt]);
    if (splits > 1 && grp == 0)
      ((float2 *)a.part_ml)[(prow0 + 32 * wave + 16 * rt + col) * splits + sp] = make_float2(m_run[rt], l);
    float f[4];
    float norm = splits > 1 ? 1.0f : l > 0.0f ? 1.0f / (l * kPlaneScale) : 0.0f;       // the value planes' 2^6 as well
    if constexpr (GG) norm = __builtin_ldexpf(norm, vexp);
    per_row(norm, grp, f);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 32 * wave + 16 * rt + 4 * grp + i;
      const int tok = q0 + row / G;
      float *dst;
      if (splits > 1) dst = a.part_o + ((prow0 + row) * splits + sp) * D + col;
      else if (row < a.qt * G && tok < a.Sq)
        dst = a.o + (GG ? ((int64_t)b * a.Sq + tok) * a.Hq + h * G + row % G
                        : (int64_t)(b * a.Hq + h * G + row % G) * a.Sq + tok) * D + col;
      else continue;
#pragma unroll
      for (int nb = 0; nb < NT; ++nb) dst[16 * nb] = oacc[rt][nb][i] * f[i];
    }
  }
}

template <int D>
static hipError_t launch_planes_d(const PrefillArgs &a, int kb, int vb, const PrefillPlan &p, uint8_t *records,
                                  int stream0, int ns, hipStream_t s) {
  const int kv_end = a.causal ? (a.S < a.q_start + a.Sq ? a.S : a.q_start + a.Sq) : a.S;
  const dim3 dg((kv_end + kPT - 1) / kPT, ns);
  if (kb == 4 && vb == 4) plane_decode_kernel<D, 4, 4><<<dg, 256, 0, s>>>(a, records, p.stream_bytes, stream0);
  else if (kb == 4) plane_decode_kernel<D, 4, 2><<<dg, 256, 0, s>>>(a, records, p.stream_bytes, stream0);
  else if (vb == 4) plane_decode_kernel<D, 2, 4><<<dg, 256, 0, s>>>(a, records, p.stream_bytes, stream0);
  else plane_decode_kernel<D, 2, 2><<<dg, 256, 0, s>>>(a, records, p.stream_bytes, stream0);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int blocks = a.qtiles * a.splits * ns;
  if (a.token_major) prefill_planes_kernel<D, true><<<blocks, kPW * 64, 0, s>>>(a, records, p.stream_bytes, stream0, ns);
  else prefill_planes_kernel<D, false><<<blocks, kPW * 64, 0, s>>>(a, records, p.stream_bytes, stream0, ns);
  e = hipGetLastError();
  if (e != hipSuccess || a.splits == 1) return e;
  return launch_prefill_merge(a, stream0, ns, kPRows, s);
}

hipError_t launch_prefill_planes(PrefillArgs a, int k_bits, int v_bits, const PrefillPlan &p, uint8_t *records,
                                 hipStream_t s) {
  const int streams = a.B * a.n_heads;
  for (int s0 = 0; s0 < streams; s0 += p.streams) {
    const int ns = streams - s0 < p.streams ? streams - s0 : p.streams;
    const hipError_t e = a.d == 128 ? launch_planes_d<128>(a, k_bits, v_bits, p, records, s0, ns, s)
                                    : launch_planes_d<64>(a, k_bits, v_bits, p, records, s0, ns, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace pqkv
