// General-shape projections with fp32 activations: y = alpha * x . w^T for ANY M, N, K (no multiple-of-64 contract),
// weights bf16 or fp32 as stored ([N][K] row-major), fp32 accumulation, fp32 output - plain, and grouped over
// expert-sorted rows (one launch for all experts of a sparse feed-forward, SwiGLU optionally in the epilogue).
//
// (bf16 products of more rows than any_stream_takes says - K a multiple of 64, no segments - go to gemm_any_tile.hip.)
//
// These serve the model families whose residual stream, norms and recurrences are kept in 32-bit floats and whose
// widths are not the fragment-native kernels' (csrc/gemm_skinny*.hpp, gemm_tile.hip): eleven kernels,
//
//   gemm_any_mfma_kernel   bf16 weights: a 64 x 64 (from 512 rows: 128 x 128, with SwiGLU 128 x 64) output tile per 4-wave
//                          workgroup, x rounded to bf16 on its way into LDS, v_mfma_f32_16x16x32_bf16, the next K
//                          step's operands fetched while the current one is multiplied, edges zero-filled
//   gemm_any_skinny_kernel bf16 weights, up to 64 rows per tile (decode batches, a decode step's experts): 16 features per
//                          workgroup, the waves split K, fragments straight from memory
//   gemm_any_stream_kernel bf16 weights, 9 to 64 rows and experts of few rows each, K a multiple of 64: the same work with two 64-deep
//                          blocks in flight per wave and whole lines through LDS
//   gemm_any_stream_groups_kernel  the same for more than 96 rows of experts, whose shares may be uneven
//   gemm_any_heads_kernel  bf16 weights, the batched form over many rows (a head's projection of its own columns): the head's weight in
//                          LDS, x rows straight into operands
//   gemm_any_f32_kernel    true 32-bit: fp32 (or bf16, widened exactly) weights, x NOT rounded, on the fp32 matrix instruction
//                          - the float32 serving mode, and the routers of sparse feed-forwards in either mode
//   gemm_any_split_kernel  true 32-bit for fp32 weights and larger launches: both operands in three bf16 parts, on the bf16 instruction
//   gemm_any_fma_kernel    the same in plain FMA chains, for operands whose rows are not whole 128-byte lines
//   gemm_any_rows_kernel   M <= 8 rows, and the exact mode up to 64: one wave per (one or four output features, batch of rows)
//                          streams its weight row once, lanes split K in 16-byte pieces, butterfly reduction; both
//                          dtypes, x not rounded
//   gemm_any_rows_lds_kernel  the same sums for 2 to 8 rows and many features of bf16 weights: the rows in LDS
//   gemm_any_each_row_kernel  the same for groups that have a row or none each
//
// A row of the result is a function of its own x row and the weights only: the summation order over k does not depend
// on M, on the row's place in the batch or on the tile it falls into (each kernel has ONE fixed order), so the same
// token gives the same bits whatever it is batched with, within one kernel; between kernels (a row computed in a
// prompt's portion vs alone) results differ by rounding only.
#include <algorithm>
#include <cmath>

#include "gemm_any_stream.hpp"

namespace mi {

struct GemmAnyArgs {
  const float* x;
  int64_t ldx;
  const void* w;    // [groups][N][K]
  const void* w2;   // nullptr, or the second weight of the SwiGLU epilogue: y = silu(x w^T) * (x w2^T)
  float* y;
  int64_t ldy;
  int M, N, K;
  float alpha;
  const int32_t* group_offsets;  // nullptr: one group of M rows; else rows of group g = [off[g], off[g + 1])
  const int32_t* x_rows;         // nullptr or the x row of each (sorted) row
  const int32_t* y_rows;         // nullptr or the y row of each (sorted) row
  // epilogue: v = acc + bias[n]; with w2: v = act(v) * (acc2 + bias2[n]), else v = act(v); v *= alpha;
  // gate: v *= sigmoid(gate[y row][n])
  const float* bias;
  const float* bias2;
  int act;  // MI_ACT_*
  const float* gate;
  int64_t ldgate;
  // batched form (group_offsets == nullptr, gridDim.z > 1): batch b multiplies the M rows at x + b * x_batch with
  // w[b] into y + b * y_batch (a per-head projection of head-major rows: the batch stride is a head's width)
  int64_t x_batch, y_batch, gate_batch;
  // grouped form: sorted row m's accumulators are multiplied by row_scale[row_scale_rows ? row_scale_rows[m] : m] before
  // anything else (= its x row scaled, without touching x: an expert whose routing weight goes into its INPUT)
  const float* row_scale;
  const int32_t* row_scale_rows;
  float limit;  // MI_ACT_CLAMPED_GLU
  // extended epilogue: `act` applies to the features n >= act_from only, `act2` to those from act2_from (>= act_from) on -
  // several projections of one input, each with an activation of its own, as one product
  bool ext;
  int act_from, act2, act2_from;
  int n_groups;  // the grouped forms of gemm_any_f32_kernel and the streaming kernel
};

template <typename TW>
__device__ __forceinline__ float w_load(const TW* p);
template <>
__device__ __forceinline__ float w_load<float>(const float* p) { return *p; }
template <>
__device__ __forceinline__ float w_load<uint16_t>(const uint16_t* p) { return bf2f(*p); }

__device__ __forceinline__ bool dev_aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
__device__ __forceinline__ float silu_f(float z) { return z / (1.f + expf(-z)); }
__device__ __forceinline__ float act_f(int act, float z) {
  switch (act) {
    case MI_ACT_SILU: return silu_f(z);
    case MI_ACT_GELU_TANH: return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
    case MI_ACT_GELU_ERF: return 0.5f * z * (1.f + erff(z * 0.7071067811865476f));
    case MI_ACT_SIGMOID: return 1.f / (1.f + expf(-z));
    case MI_ACT_RELU2: return fmaxf(z, 0.f) * fmaxf(z, 0.f);
    default: return z;  // (MI_ACT_SOFTCAP is finish()'s: it needs the cap)
  }
}
// the activations of the extended epilogue
__device__ __forceinline__ float act_ext_f(int act, float z) {
  if (act == MI_ACT_TANH) return tanhf(z);
  if (act == MI_ACT_DECAY) return expf(-0.6065306597126334f / (1.f + expf(-z)));  // exp(-exp(-1/2) sigmoid(z))
  return act_f(act, z);
}
// what every kernel does to an accumulator (pair) before it stores it.  EXT: the epilogue with the activation segments and
// the activations only they use - kernels of their own, because a longer epilogue costs every tile kernel registers (7 % of
// a prefill step of models that never take these branches)
template <bool DUAL, bool EXT>
__device__ __forceinline__ float finish(const GemmAnyArgs& a, int64_t m, int64_t yrow, int n, float v, float v2) {
  if (a.row_scale) {
    const float rs = a.row_scale[a.row_scale_rows ? a.row_scale_rows[m] : m];
    v *= rs, v2 *= rs;
  }
  if (a.bias) v += a.bias[n];
  if (DUAL) {
    if (a.bias2) v2 += a.bias2[n];
    if (a.act == MI_ACT_CLAMPED_GLU) {  // g sigmoid(1.702 g) (u + 1) with g capped from above, u clamped to +-limit
      const float g = fminf(v, a.limit), u = fminf(fmaxf(v2, -a.limit), a.limit);
      v = g / (1.f + expf(-1.702f * g)) * (u + 1.f);
    } else {
      v = act_f(a.act, v) * v2;
    }
  } else if constexpr (EXT) {
    if (n >= a.act_from) v = n >= a.act2_from ? act_ext_f(a.act2, v) : act_ext_f(a.act, v);
  } else {
    v = a.act == MI_ACT_SOFTCAP ? tanhf(v / a.alpha) : act_f(a.act, v);  // (times alpha below: alpha tanh(v / alpha))
  }
  v *= a.alpha;
  if (a.gate) v *= 1.f / (1.f + expf(-a.gate[yrow * a.ldgate + n]));
  return v;
}
// the operands of this workgroup's group (grouped form) or batch (batched form)
template <typename TW, bool DUAL>
__device__ __forceinline__ void select_group(GemmAnyArgs& a, const TW*& w, const TW*& w2, int& m_lo, int& m_hi) {
  m_lo = 0, m_hi = a.M;
  w = static_cast<const TW*>(a.w);
  w2 = static_cast<const TW*>(a.w2);
  if (a.group_offsets) {
    m_lo = a.group_offsets[blockIdx.z];
    m_hi = a.group_offsets[blockIdx.z + 1];
  } else if (blockIdx.z > 0) {
    a.x += (int64_t)blockIdx.z * a.x_batch;
    a.y += (int64_t)blockIdx.z * a.y_batch;
    if (a.gate) a.gate += (int64_t)blockIdx.z * a.gate_batch;
  }
  w += (int64_t)blockIdx.z * a.N * a.K;
  if (DUAL) w2 += (int64_t)blockIdx.z * a.N * a.K;
}

// eight consecutive operands as floats: one 16-byte (bf16) / two 16-byte (fp32) loads, or element-wise at an edge
template <typename TW>
__device__ __forceinline__ void load8(const TW* p, int n_valid, bool vec, float (&v)[8]);
template <>
__device__ __forceinline__ void load8<uint16_t>(const uint16_t* p, int n_valid, bool vec, float (&v)[8]) {
  if (vec && n_valid >= 8) {
    const u32x4 w = *reinterpret_cast<const u32x4*>(p);
    v[0] = lo_bf(w[0]), v[1] = hi_bf(w[0]), v[2] = lo_bf(w[1]), v[3] = hi_bf(w[1]);
    v[4] = lo_bf(w[2]), v[5] = hi_bf(w[2]), v[6] = lo_bf(w[3]), v[7] = hi_bf(w[3]);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = i < n_valid ? bf2f(p[i]) : 0.f;
  }
}
template <>
__device__ __forceinline__ void load8<float>(const float* p, int n_valid, bool vec, float (&v)[8]) {
  if (vec && n_valid >= 8) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = i < n_valid ? p[i] : 0.f;
  }
}

// ---------------------------------------------------------------------------------------------------------------
// exact kernel for any alignment and K: 256 threads, RT x 4 outputs per thread, k ascending: a 64 x 64 tile (RT 4) or 16 x 64 (1: few
// features, many rows)
// ---------------------------------------------------------------------------------------------------------------
template <typename TW, bool DUAL, int RT, bool EXT>
__global__ __launch_bounds__(256) void gemm_any_fma_kernel(GemmAnyArgs a) {
  constexpr int BM = 16 * RT, BN = 64, BK = 32, PAD = 4;
  __shared__ float As[BK][BM + PAD];
  __shared__ float Bs[DUAL ? 2 : 1][BK][BN + PAD];
  const int tid = threadIdx.x;
  int m_lo, m_hi;
  const TW *w, *w2;
  select_group<TW, DUAL>(a, w, w2, m_lo, m_hi);
  const int m0 = m_lo + blockIdx.y * BM;
  if (m0 >= m_hi) return;
  const int n0 = blockIdx.x * BN;
  const int lr = tid >> 2, lk = (tid & 3) * 8;  // this thread stages 8 consecutive k of one row
  int64_t xrow = -1;
  if (lr < BM && m0 + lr < m_hi) xrow = a.x_rows ? a.x_rows[m0 + lr] : m0 + lr;
  const int wrow = n0 + lr < a.N ? n0 + lr : -1;
  float acc[DUAL ? 2 : 1][RT][4] = {};
  const int ty = tid >> 4, tx = tid & 15;
  for (int k0 = 0; k0 < a.K; k0 += BK) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = k0 + lk + i;
      if (lr < BM) As[lk + i][lr] = (xrow >= 0 && k < a.K) ? a.x[xrow * a.ldx + k] : 0.f;
      Bs[0][lk + i][lr] = (wrow >= 0 && k < a.K) ? w_load<TW>(w + (int64_t)wrow * a.K + k) : 0.f;
      if (DUAL) Bs[1][lk + i][lr] = (wrow >= 0 && k < a.K) ? w_load<TW>(w2 + (int64_t)wrow * a.K + k) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < BK; ++k) {
      float av[RT], bv[DUAL ? 2 : 1][4];
#pragma unroll
      for (int i = 0; i < RT; ++i) av[i] = As[k][ty * RT + i];
#pragma unroll
      for (int d = 0; d < (DUAL ? 2 : 1); ++d)
#pragma unroll
        for (int j = 0; j < 4; ++j) bv[d][j] = Bs[d][k][tx * 4 + j];
#pragma unroll
      for (int d = 0; d < (DUAL ? 2 : 1); ++d)
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[d][i][j] = fmaf(av[i], bv[d][j], acc[d][i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int m = m0 + ty * RT + i;
    if (m >= m_hi) continue;
    const int64_t yrow = a.y_rows ? a.y_rows[m] : m;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= a.N) continue;
      a.y[yrow * a.ldy + n] = finish<DUAL, EXT>(a, m, yrow, n, acc[0][i][j], acc[DUAL ? 1 : 0][i][j]);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// exact kernel on the matrix cores: v_mfma_f32_16x16x4_f32 (fp32 operands, fp32 products and sums; twice the vector rate)
// ---------------------------------------------------------------------------------------------------------------
// Four waves (WM x WN) with FM x FN fragments of 16 x 16 each.  K in steps of 32 floats = one 128-byte line of a row, by
// LDS-DMA (global_load_lds, 16 bytes a lane: eight rows an instruction; bf16 weights: sixteen rows of 64 bytes) into a ring of
// four images, so that three steps are in flight: these products are latency-bound, not rate-bound, at the sizes they come in
// (a router's 32 features, an expert's hundred rows).  A row's 16-byte chunks are XOR-swizzled by its number, on the source
// side of the DMA and at the fragment reads: sixteen rows at one chunk are sixteen different bank groups.  A lane reads four
// consecutive k of its row at once (ds_read_b128; bf16: 8 bytes, widened): element j goes into the j-th MFMA of a group
// of 16 k, which then contracts k = 4 (lane >> 4) + j - a fixed order of the sum, whatever the tile.
// Rows beyond the group's end and features beyond N are read from the last valid one and not stored.
// Needs K % 32 == 0, 16-byte aligned rows of x and w; anything else: gemm_any_fma_kernel.
// Measured against gemm_any_fma_kernel (64 x 64 tiles, element-wise loads, plain FMA chains), us: see launch_exact.
// The tile-th row tile of BM rows over all groups (group by group, a group's first SKIP rows left out): its group, its first row and the end
// of the group's rows, or false beyond the last.  Every wave for itself.
template <int BM, int SKIP = 0>
__device__ __forceinline__ bool group_tile(const int32_t* __restrict__ offsets, int groups, int tile, int& g, int& m0, int& m_hi) {
  const int lane = threadIdx.x & 63;
  for (int base = 0; base < groups; base += 64) {
    const int i = min(base + lane, groups - 1), lo = offsets[i] + SKIP, hi = offsets[i + 1];
    const int mine = base + lane < groups ? (max(hi - lo, 0) + BM - 1) / BM : 0;
    int upto = mine;
#pragma unroll
    for (int o = 1; o < 64; o *= 2) {
      const int v = __shfl_up(upto, o);
      upto += lane >= o ? v : 0;
    }
    const uint64_t behind = __ballot(upto > tile);
    if (behind) {
      const int l = __builtin_ctzll(behind);
      g = base + l;
      m0 = __builtin_amdgcn_readlane(lo, l) + (tile - (__builtin_amdgcn_readlane(upto, l) - __builtin_amdgcn_readlane(mine, l))) * BM;
      m_hi = __builtin_amdgcn_readlane(hi, l);
      return true;
    }
    tile -= __builtin_amdgcn_readlane(upto, 63);
  }
  return false;
}

// GROUPS: 0 none; 1 a workgroup for every row tile that a group can have; 2 as many as all groups' rows need, each every gridDim.y-th row tile of all
// groups, which it has to find (0.8 us)
template <typename TW, bool DUAL, int FM, int FN, int WM, int WN, bool EXT, int GROUPS, bool AHEAD>
__global__ __launch_bounds__(256) void gemm_any_f32_kernel(GemmAnyArgs a) {
  constexpr int BM = 16 * FM * WM, BN = 16 * FN * WN, BK = 32, NST = 4, ND = DUAL ? 2 : 1;
  constexpr bool WF = sizeof(TW) == 4;
  constexpr int WROW = BK * (int)sizeof(TW), WRP = 1024 / WROW;           // bytes of a weight row's step, rows of a piece
  constexpr int XB = BM * 128, WB = BN * WROW, STAGE = XB + ND * WB;
  constexpr int PIECES = STAGE / 1024, PP = (PIECES + 3) / 4;             // 1 KiB each; PP per wave (the last may repeat)
  static_assert(WM * WN == 4 && XB % 1024 == 0 && WB % 1024 == 0, "whole pieces");
  __shared__ __attribute__((aligned(1024))) char lds[NST * STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * BN, KT = a.K / BK;
  const int wm = (wave / WN) * 16 * FM, wn = (wave % WN) * 16 * FN;
  const int r16 = lane & 15, kg = lane >> 4;
  if constexpr (GROUPS == 1)   // (asked for here: behind the way out below they would be a round trip of their own)
    asm volatile("" ::"s"(a.x), "s"(a.w), "s"(a.y), "s"(a.x_rows), "s"(a.y_rows), "s"(a.ldx), "s"(a.ldy), "s"(a.row_scale), "s"(a.bias));
  for (int tile = blockIdx.y;; tile += gridDim.y) {
    int m0 = tile * BM, m_hi = a.M;
    const float* x = a.x;
    const TW *w = static_cast<const TW*>(a.w), *w2 = static_cast<const TW*>(a.w2);
    float* y = a.y;
    if constexpr (GROUPS != 0) {
      int g = blockIdx.z;
      if constexpr (GROUPS == 1) {
        m0 = a.group_offsets[g] + tile * BM, m_hi = a.group_offsets[g + 1];
        if (m0 >= m_hi) return;
      } else {
        if (!group_tile<BM>(a.group_offsets, a.n_groups, tile, g, m0, m_hi)) return;
      }
      w += (int64_t)g * a.N * a.K;
      if (DUAL) w2 += (int64_t)g * a.N * a.K;
      if (tile != (int)blockIdx.y) __syncthreads();  // (the tile before is read)
    } else {
      // (the launch has no tile beyond the rows: a way out here would put the other arguments' loads behind it, 0.3 us)
      x += (int64_t)blockIdx.z * a.x_batch;
      y += (int64_t)blockIdx.z * a.y_batch;
      if (a.gate) a.gate += (int64_t)blockIdx.z * a.gate_batch;
      w += (int64_t)blockIdx.z * a.N * a.K;
      if (DUAL) w2 += (int64_t)blockIdx.z * a.N * a.K;
    }
    const bool y_vec = (a.ldy % 4 == 0) && dev_aligned16(y);   // (a batch's rows begin where its stride says)
    const char* src[PP];
    int dst[PP];
#pragma unroll
    for (int i = 0; i < PP; ++i) {
      const int p = min(wave * PP + i, PIECES - 1);
      dst[i] = p * 1024;
      if (p < XB / 1024) {
        const int r = p * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        const int m = min(m0 + r, m_hi - 1);
        const int64_t row = a.x_rows ? a.x_rows[m] : m;
        src[i] = reinterpret_cast<const char*>(x + row * a.ldx) + c * 16;
      } else {
        const int q = p - XB / 1024, d = q / (WB / 1024);
        constexpr int CH = WROW / 16;
        const int r = (q - d * (WB / 1024)) * WRP + lane / CH;
        const int c = (lane % CH) ^ (WF ? (r >> 1) & 7 : (r >> 2) & 3);
        src[i] = reinterpret_cast<const char*>((DUAL && d ? w2 : w) + (int64_t)min(n0 + r, a.N - 1) * a.K) + c * 16;
      }
    }
    auto issue = [&](int kt) __attribute__((always_inline)) {
      char* base = lds + (kt & (NST - 1)) * STAGE;
#pragma unroll
      for (int i = 0; i < PP; ++i) {
        const bool is_x = dst[i] < XB;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + (int64_t)kt * (is_x ? 128 : WROW)),
                                         (__attribute__((address_space(3))) void*)(base + dst[i]), 16, 0, 0);
      }
    };
    f32x4 acc[ND][FM][FN];
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[d][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NST - 1; ++s)
      if (s < KT) issue(s);
    // AHEAD: a step's fragments are read during the matrix instructions of the step before: with one or two waves on a SIMD nothing else stands
    // beside the barrier and the reads' latency.  Of the time without: 32 x 32 tiles, one weight in fp32 0.91 .. 0.97 (200 x 1024 x 1024 11.7 / 10.8 us, 728 x
    // 1024 x 1024 21.4 / 20.6), in bf16 0.94 .. 0.98 and two weights 0.95 .. 0.98 up to a tile per CU, 0.98 .. 1.03 from two on; two weights in fp32 with two tiles
    // on some CUs 0.98 .. 1.06 (400 rows of 32 experts of 512 x 1024 29.0 / 30.7), with more from K 1024 on 0.97 .. 1.00.  Larger tiles keep a SIMD's
    // matrix pipe busy with the waves of a CU's other tiles: 32 x 64 one weight in fp32 0.955 .. 0.99 from K 1024 on and up to five tiles per CU, else
    // 0.98 .. 1.10 (K 512 1.00 .. 1.02, 160 1.00 .. 1.07; nine tiles 1.02), 64 x 64 1.00; and where these ran in step, a CU was given two of
    // the last tiles and its neighbour none (two weights, 1500 x 1024 x 1024 64 / 78 us; one, 2100 x 1408 x 1088 65 / 80).
    struct Frags {
      f32x4 x[2][FM];
      std::conditional_t<WF, f32x4, u32x2> w[2][ND][FN];
    } fa, fb;
    auto read = [&](int kt, Frags& f) __attribute__((always_inline)) {
      const int behind = min(KT - 1 - kt, NST - 2);  // steps requested behind this one: their pieces may still fly
      if (behind == 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * PP) : "memory");
      else if (behind == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(PP) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (kt + NST - 1 < KT) issue(kt + NST - 1);  // (into the image everybody finished reading before the barrier)
      const char* sx = lds + (kt & (NST - 1)) * STAGE;
      const char* sw = sx + XB;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const int r = wm + i * 16 + r16;
          f.x[ks][i] = *reinterpret_cast<const f32x4*>(sx + r * 128 + (((ks * 4 + kg) ^ ((r >> 1) & 7)) << 4));
        }
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            const int r = wn + j * 16 + r16;
            if constexpr (WF) f.w[ks][d][j] = *reinterpret_cast<const f32x4*>(sw + d * WB + r * 128 + (((ks * 4 + kg) ^ ((r >> 1) & 7)) << 4));
            else f.w[ks][d][j] = *reinterpret_cast<const u32x2*>(sw + d * WB + r * 64 + (((ks * 2 + (kg >> 1)) ^ ((r >> 2) & 3)) << 4) + (kg & 1) * 8);
          }
      }
      if constexpr (AHEAD) __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        f32x4 wf[ND][FN];
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            if constexpr (WF) wf[d][j] = f.w[ks][d][j];
            else wf[d][j] = f32x4{lo_bf(f.w[ks][d][j][0]), hi_bf(f.w[ks][d][j][0]), lo_bf(f.w[ks][d][j][1]), hi_bf(f.w[ks][d][j][1])};
          }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
              for (int j = 0; j < FN; ++j)
                acc[d][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[d][j][e], f.x[ks][i][e], acc[d][i][j], 0, 0, 0);
      }
    };
    if constexpr (AHEAD) {
      read(0, fa);
      int kt = 1;
      for (; kt + 1 < KT; kt += 2) {
        read(kt, fb);
        multiply(fa);
        read(kt + 1, fa);
        multiply(fb);
      }
      if (kt < KT) {
        read(kt, fb);
        multiply(fa);
        multiply(fb);
      } else {
        multiply(fa);
      }
    } else {
      for (int kt = 0; kt < KT; ++kt) {
        read(kt, fa);
        multiply(fa);
      }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = m0 + wm + i * 16 + r16;
      if (m >= m_hi) continue;
      const int64_t yrow = a.y_rows ? a.y_rows[m] : m;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int n = n0 + wn + j * 16 + kg * 4;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = n + r < a.N ? finish<DUAL, EXT>(a, m, yrow, n + r, acc[0][i][j][r], acc[ND - 1][i][j][r]) : 0.f;
        float* yp = y + yrow * a.ldy + n;
        if (n + 4 <= a.N && y_vec) {
          *reinterpret_cast<float4*>(yp) = float4{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < a.N) yp[r] = v[r];
        }
      }
    }
    if constexpr (GROUPS != 2) return;
  }
}

}  // namespace mi
#include "gemm_any_split.hpp"
namespace mi {

// ---------------------------------------------------------------------------------------------------------------
// MFMA kernel (bf16 weights): 4 waves as 2 x 2, each FM x FN fragments of 16 x 16 - a 64 x 64 tile, or 128 x 128
// (SwiGLU: 128 x 64) for prefill-sized launches, where every LDS fragment feeds four MFMAs instead of two;
// K in steps of 64 (a weight row's piece = one 128-byte line).  LDS holds the tile's x rows and weight rows as bf16
// [64][64 + 8].
// ---------------------------------------------------------------------------------------------------------------
template <bool DUAL, int FM, int FN, bool EXT>  // a wave's tile: FM x FN fragments of 16 x 16; the workgroup's: 2 x 2 waves
__global__ __launch_bounds__(256) void gemm_any_mfma_kernel(GemmAnyArgs a) {
  constexpr int BM = 32 * FM, BN = 32 * FN, BK = 64, LD = BK + 8;
  constexpr int ND = DUAL ? 2 : 1;
  __shared__ __attribute__((aligned(16))) uint16_t As[BM][LD];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[ND][BN][LD];
  const int tid = threadIdx.x;
  int m_lo, m_hi;
  const uint16_t *w, *w2;
  select_group<uint16_t, DUAL>(a, w, w2, m_lo, m_hi);
  const int m0 = m_lo + blockIdx.y * BM;
  if (m0 >= m_hi) return;
  const int n0 = blockIdx.x * BN;
  // staging: a thread takes 16 consecutive k of one row (a row's 64 k = one 128-byte line of weights), 64 rows per pass
  const int lr = tid >> 2, lk = (tid & 3) * 16;
  int64_t xrow[BM / 64];
  int wrow[BN / 64];
#pragma unroll
  for (int p = 0; p < BM / 64; ++p) {
    const int m = m0 + p * 64 + lr;
    xrow[p] = m < m_hi ? (a.x_rows ? a.x_rows[m] : m) : -1;
  }
#pragma unroll
  for (int p = 0; p < BN / 64; ++p) wrow[p] = n0 + p * 64 + lr < a.N ? n0 + p * 64 + lr : -1;
  const bool w_vec = (a.K % 8 == 0) && dev_aligned16(a.w) && (!DUAL || dev_aligned16(a.w2));
  const bool x_vec = (a.ldx % 4 == 0) && dev_aligned16(a.x);
  const int wave = tid >> 6, lane = tid & 63;
  const int wm = (wave >> 1) * 16 * FM, wn = (wave & 1) * 16 * FN;
  const int fr = lane & 15, fk = (lane >> 4) * 8;
  f32x4 acc[ND][FM][FN];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[d][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // the tile's operands travel memory -> registers -> LDS; the registers of K step k + 1 are loaded while step k's
  // MFMAs run, so the global-memory latency is not paid between the two barriers
  u32x4 xreg[2][BM / 64], wreg[ND][2][BN / 64];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int k = k0 + lk + half * 8;
#pragma unroll
      for (int p = 0; p < BM / 64; ++p) {
        float xv[8];
        if (xrow[p] >= 0) load8<float>(a.x + xrow[p] * a.ldx + k, a.K - k, x_vec, xv);
        else {
#pragma unroll
          for (int i = 0; i < 8; ++i) xv[i] = 0.f;
        }
        xreg[half][p] = u32x4{pack_bf(xv[0], xv[1]), pack_bf(xv[2], xv[3]), pack_bf(xv[4], xv[5]), pack_bf(xv[6], xv[7])};
      }
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int p = 0; p < BN / 64; ++p) {
          const uint16_t* wp = (d ? w2 : w) + (int64_t)wrow[p] * a.K + k;
          u32x4 v = {0u, 0u, 0u, 0u};
          if (wrow[p] >= 0 && k < a.K) {
            if (w_vec && k + 8 <= a.K) {
              v = *reinterpret_cast<const u32x4*>(wp);
            } else {
              uint16_t e[8];
#pragma unroll
              for (int i = 0; i < 8; ++i) e[i] = k + i < a.K ? wp[i] : (uint16_t)0;
              v = u32x4{(uint32_t)e[0] | ((uint32_t)e[1] << 16), (uint32_t)e[2] | ((uint32_t)e[3] << 16),
                        (uint32_t)e[4] | ((uint32_t)e[5] << 16), (uint32_t)e[6] | ((uint32_t)e[7] << 16)};
            }
          }
          wreg[d][half][p] = v;
        }
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < a.K; k0 += BK) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int p = 0; p < BM / 64; ++p) *reinterpret_cast<u32x4*>(&As[p * 64 + lr][lk + half * 8]) = xreg[half][p];
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int p = 0; p < BN / 64; ++p) *reinterpret_cast<u32x4*>(&Bs[d][p * 64 + lr][lk + half * 8]) = wreg[d][half][p];
    }
    __syncthreads();
    if (k0 + BK < a.K) fetch(k0 + BK);
    // D[n][m] = sum_k W[n][k] X[m][k]: weights on the MFMA's row axis, so a lane's four results are four consecutive
    // FEATURES of one x row
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 af[FM], bfr[ND][FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) af[i] = as_frag(*reinterpret_cast<const u32x4*>(&As[wm + i * 16 + fr][ks * 32 + fk]));
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          bfr[d][j] = as_frag(*reinterpret_cast<const u32x4*>(&Bs[d][wn + j * 16 + fr][ks * 32 + fk]));
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[d][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[d][j], af[i], acc[d][i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // fragment (i, j): x row = wm + i*16 + (lane & 15), features wn + j*16 + (lane >> 4) * 4 + r
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + wm + i * 16 + (lane & 15);
    if (m >= m_hi) continue;
    const int64_t yrow = a.y_rows ? a.y_rows[m] : m;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = n0 + wn + j * 16 + (lane >> 4) * 4;
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        v[r] = n + r < a.N ? finish<DUAL, EXT>(a, m, yrow, n + r, acc[0][i][j][r], acc[ND - 1][i][j][r]) : 0.f;
      float* yp = a.y + yrow * a.ldy + n;
      if (n + 4 <= a.N && (a.ldy % 4 == 0) && dev_aligned16(a.y)) {
        *reinterpret_cast<float4*>(yp) = float4{v[0], v[1], v[2], v[3]};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < a.N) yp[r] = v[r];
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// up to 64 rows per tile (decode batches, a decode step's experts): 16 output features per workgroup, so that even a
// 1024-feature projection spreads over 64 workgroups; the four waves take the K steps of 32 in turn (together they read
// 256 contiguous bytes of every weight row per round), operands go from memory straight into MFMA fragments - no LDS
// staging, no barrier inside the K loop - and the waves' accumulators are added in wave order through LDS at the end.
// ---------------------------------------------------------------------------------------------------------------
template <bool DUAL, int MF, bool EXT>  // MF fragments of 16 rows
__global__ __launch_bounds__(256) void gemm_any_skinny_kernel(GemmAnyArgs a) {
  __shared__ __attribute__((aligned(16))) float red[3][DUAL ? 2 : 1][MF][64][4];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  int m_lo, m_hi;
  const uint16_t *w, *w2;
  select_group<uint16_t, DUAL>(a, w, w2, m_lo, m_hi);
  const int m0 = m_lo + blockIdx.y * 16 * MF;
  if (m0 >= m_hi) return;
  const int n0 = blockIdx.x * 16;
  const int fr = lane & 15, kk = (lane >> 4) * 8;
  const int wrow = n0 + fr < a.N ? n0 + fr : -1;
  int64_t xrow[MF];
#pragma unroll
  for (int f = 0; f < MF; ++f) {
    const int m = m0 + f * 16 + fr;
    xrow[f] = m < m_hi ? (a.x_rows ? a.x_rows[m] : m) : -1;
  }
  const bool w_vec = (a.K % 8 == 0) && dev_aligned16(a.w) && (!DUAL || dev_aligned16(a.w2));
  const bool x_vec = (a.ldx % 4 == 0) && dev_aligned16(a.x);
  f32x4 acc[DUAL ? 2 : 1][MF];
#pragma unroll
  for (int d = 0; d < (DUAL ? 2 : 1); ++d)
#pragma unroll
    for (int f = 0; f < MF; ++f) acc[d][f] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = wave * 32; k0 < a.K; k0 += 4 * 32) {
    const int k = k0 + kk;
    bf16x8 wf[DUAL ? 2 : 1];
#pragma unroll
    for (int d = 0; d < (DUAL ? 2 : 1); ++d) {
      const uint16_t* wp = (d ? w2 : w) + (int64_t)wrow * a.K + k;
      u32x4 v = {0u, 0u, 0u, 0u};
      if (wrow >= 0 && k < a.K) {
        if (w_vec && k + 8 <= a.K) {
          v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp));
        } else {
          uint16_t e[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) e[i] = k + i < a.K ? wp[i] : (uint16_t)0;
          v = u32x4{(uint32_t)e[0] | ((uint32_t)e[1] << 16), (uint32_t)e[2] | ((uint32_t)e[3] << 16),
                    (uint32_t)e[4] | ((uint32_t)e[5] << 16), (uint32_t)e[6] | ((uint32_t)e[7] << 16)};
        }
      }
      wf[d] = as_frag(v);
    }
#pragma unroll
    for (int f = 0; f < MF; ++f) {
      float xv[8];
      if (xrow[f] >= 0) load8<float>(a.x + xrow[f] * a.ldx + k, a.K - k, x_vec, xv);
      else {
#pragma unroll
        for (int i = 0; i < 8; ++i) xv[i] = 0.f;
      }
      const bf16x8 xf = as_frag(u32x4{pack_bf(xv[0], xv[1]), pack_bf(xv[2], xv[3]), pack_bf(xv[4], xv[5]), pack_bf(xv[6], xv[7])});
#pragma unroll
      for (int d = 0; d < (DUAL ? 2 : 1); ++d)
        acc[d][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[d], xf, acc[d][f], 0, 0, 0);
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int d = 0; d < (DUAL ? 2 : 1); ++d)
#pragma unroll
      for (int f = 0; f < MF; ++f) *reinterpret_cast<f32x4*>(red[wave - 1][d][f][lane]) = acc[d][f];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int ow = 0; ow < 3; ++ow)
#pragma unroll
    for (int d = 0; d < (DUAL ? 2 : 1); ++d)
#pragma unroll
      for (int f = 0; f < MF; ++f) acc[d][f] += *reinterpret_cast<const f32x4*>(red[ow][d][f][lane]);
  // a lane holds features n0 + (lane >> 4) * 4 + r of x row (lane & 15) of every fragment
#pragma unroll
  for (int f = 0; f < MF; ++f) {
    const int m = m0 + f * 16 + fr;
    if (m >= m_hi) continue;
    const int64_t yrow = a.y_rows ? a.y_rows[m] : m;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = n0 + (lane >> 4) * 4 + r;
      if (n >= a.N) continue;
      a.y[yrow * a.ldy + n] = finish<DUAL, EXT>(a, m, yrow, n, acc[0][f][r], acc[DUAL ? 1 : 0][f][r]);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// decode batches (9 to 64 rows), and a decode step's experts: 16 RT output features (DUAL: of both weights) per workgroup, the waves take the
// 64-deep blocks of K in turn, two blocks in flight each
// ---------------------------------------------------------------------------------------------------------------
// These launches are latency-bound: a projection of 2 to 8 MB of weights has a microsecond of bytes and three of round trips.  So: one
// launch (x is rounded to bf16 on its way into LDS - every workgroup re-reads all rows, 4 bytes per element out of the L2s - instead of
// an operand pass in front), every wave's loads issued before its first use, no barrier before the waves' sums meet.  A wave asks for
// whole lines, consecutive lanes consecutive pieces, and turns them into fragments through its own part of LDS: asked for as fragments
// (16 rows an instruction, as gemm_any_skinny_kernel does) a CU's address path takes four times as long - 32 rows x 2048 x 2048 12.4 us,
// here 8.5.  Rows beyond the end are the last one again, features beyond N the last one; neither is stored.  K % 64 == 0, rows of x and w
// on 16 bytes.
// us, operand pass + tile kernel / here: 24 rows x 1024 x 1024 9.3 / 5.4, 32 x 2048 x 2048 13.0 / 8.5, 9 x 2048 x 2048 12.9 / 5.9, 48 x
// 4096 x 2048 14.3 / 11.0, 64 x 1024 x 1024 9.5 / 8.2; SwiGLU 32 x 3072 x 2048 20.8 / 11.0; both products of 256 pairs over 64 experts of
// 768 x 2048 126 / 67 + 37 (402 MB at 6.0 TB/s), of 96 over 32 of 512 x 1024 30 / 17 + 11.
constexpr int stream_slot(int nw, int mf) {  // per wave: bf16 images [16 nw weight rows | 16 mf x rows][64 k] of the block it multiplies; then its sums
  return (nw + mf) * 2048 > nw * mf * 1024 ? (nw + mf) * 2048 : nw * mf * 1024;
}
// the workgroup's features of rows m_lo .. m_hi - 1, 16 MF at a time
template <bool DUAL, int MF, int RT, int WAVES, bool EXT>
__device__ __forceinline__ void stream_rows(const GemmAnyArgs& a, char* lds, const uint16_t* w, const uint16_t* w2, int m_lo, int m_hi) {
  static_assert(RT == 1 || !DUAL, "several feature tiles: one weight");
  constexpr int NW = DUAL ? 2 : RT, SLOT = stream_slot(NW, MF);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* const slot = lds + wave * SLOT;
  auto sums = [&](int i, int t, int f) __attribute__((always_inline)) { return reinterpret_cast<f32x4*>(lds + i * SLOT + ((t * MF + f) * 64 + lane) * 16); };
  const int n0 = blockIdx.x * 16 * RT;
  const int fr = lane & 15, g = lane >> 4;
  const uint16_t* wp[NW][2];  // a request: eight weight rows of 128 bytes / four x rows of 256
#pragma unroll
  for (int t = 0; t < NW; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      wp[t][j] = (DUAL && t ? w2 : w) + (int64_t)min(n0 + (DUAL ? 0 : t * 16) + j * 8 + (lane >> 3), a.N - 1) * a.K + wave * 64 + (lane & 7) * 8;
  const int w_at = (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4);
  const int blocks = a.K >> 6, mine = (blocks - wave + WAVES - 1) / WAVES;
  for (int m0 = m_lo; m0 < m_hi; m0 += 16 * MF) {
    const float* xp[MF * 4];
#pragma unroll
    for (int q = 0; q < MF * 4; ++q) {
      const int m = min(m0 + q * 4 + g, m_hi - 1);
      xp[q] = a.x + (int64_t)(a.x_rows ? a.x_rows[m] : m) * a.ldx + wave * 64 + fr * 4;
    }
    f32x4 acc[NW][MF];
#pragma unroll
    for (int t = 0; t < NW; ++t)
#pragma unroll
      for (int f = 0; f < MF; ++f) acc[t][f] = f32x4{0.f, 0.f, 0.f, 0.f};
    struct Block {
      u32x4 w[NW][2];
      f32x4 x[MF * 4];
    };
    auto issue = [&](Block& b, int i) __attribute__((always_inline)) {
      const int k = i * (WAVES * 64);
#pragma unroll
      for (int t = 0; t < NW; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) b.w[t][j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp[t][j] + k));
#pragma unroll
      for (int q = 0; q < MF * 4; ++q) b.x[q] = *reinterpret_cast<const f32x4*>(xp[q] + k);
      __builtin_amdgcn_sched_barrier(0);  // (the next block's requests stay in front of this block's waits)
    };
    auto consume = [&](const Block& b) __attribute__((always_inline)) {  // (one wave's LDS operations are in order: no barrier)
#pragma unroll
      for (int t = 0; t < NW; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) *reinterpret_cast<u32x4*>(slot + t * 2048 + j * 1024 + w_at) = b.w[t][j];
#pragma unroll
      for (int q = 0; q < MF * 4; ++q) {
        const int r = (q * 4 + g) & 7;
        *reinterpret_cast<u32x2*>(slot + NW * 2048 + (q * 4 + g) * 128 + (((fr >> 1) ^ r) << 4) + (fr & 1) * 8) =
            u32x2{pack_bf(b.x[q][0], b.x[q][1]), pack_bf(b.x[q][2], b.x[q][3])};
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int at = fr * 128 + (((s * 4 + g) ^ (fr & 7)) << 4);
        bf16x8 wf[NW];
#pragma unroll
        for (int t = 0; t < NW; ++t) wf[t] = as_frag(*reinterpret_cast<const u32x4*>(slot + t * 2048 + at));
#pragma unroll
        for (int f = 0; f < MF; ++f) {
          const bf16x8 xf = as_frag(*reinterpret_cast<const u32x4*>(slot + (NW + f) * 2048 + at));
#pragma unroll
          for (int t = 0; t < NW; ++t) acc[t][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t], xf, acc[t][f], 0, 0, 0);
        }
      }
    };
    if (m0 > m_lo) __syncthreads();  // (the sums of the rows before are read)
    if (mine > 0) {
      Block A, B;
      issue(A, 0);
      int i = 0;
      for (; i + 2 < mine; i += 2) {
        issue(B, i + 1);
        consume(A);
        issue(A, i + 2);
        consume(B);
      }
      if (i + 1 < mine) {
        issue(B, i + 1);
        consume(A);
        consume(B);
      } else {
        consume(A);
      }
    }
#pragma unroll
    for (int t = 0; t < NW; ++t)
#pragma unroll
      for (int f = 0; f < MF; ++f) *sums(wave, t, f) = acc[t][f];
    __syncthreads();
    // a lane's four features n0 + 16 t + 4 g + r of row (lane & 15) of a fragment, the waves' sums in order
    for (int item = wave; item < (DUAL ? 1 : RT) * MF; item += WAVES) {
      const int t = item / MF, f = item % MF;
      const int m = m0 + f * 16 + fr;
      f32x4 v = *sums(0, t, f), v2 = *sums(0, DUAL ? NW - 1 : t, f);
#pragma unroll
      for (int i = 1; i < WAVES; ++i) {
        v += *sums(i, t, f);
        if (DUAL) v2 += *sums(i, NW - 1, f);
      }
      if (m >= m_hi) continue;
      const int64_t yrow = a.y_rows ? a.y_rows[m] : m;
      const int n = n0 + t * 16 + g * 4;
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = n + r < a.N ? finish<DUAL, EXT>(a, m, yrow, n + r, v[r], v2[r]) : 0.f;
      float* yp = a.y + yrow * a.ldy + n;
      if (n + 4 <= a.N && (a.ldy % 4 == 0) && dev_aligned16(a.y)) {
        *reinterpret_cast<float4*>(yp) = float4{o[0], o[1], o[2], o[3]};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < a.N) yp[r] = o[r];
      }
    }
  }
}

template <bool DUAL, int MF, int RT, int WAVES, bool EXT>
__global__ __launch_bounds__(WAVES * 64) void gemm_any_stream_kernel(GemmAnyArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[WAVES * stream_slot(DUAL ? 2 : RT, MF)];
  int m_lo, m_hi;
  const uint16_t *w, *w2;
  select_group<uint16_t, DUAL>(a, w, w2, m_lo, m_hi);
  stream_rows<DUAL, MF, RT, WAVES, EXT>(a, lds, w, w2, m_lo, m_hi);
}

// Groups, sixteen rows per workgroup: the last n_groups (blockIdx.z) take their group's first ones, the a.M in front of them share what is left - of the
// few groups that have more than the others, or of a step whose pairs go to one expert (in front: behind them it was 0.3 to 0.5 us at the
// launch's end, where there is nothing left).  us, both products, a group as one workgroup's walk | so | tile kernels: 757 pairs on one of 128 experts
// of 512 x 512 212 | 22 | 19; 512 on two of 64 of 768 x 2048 153 | 55 | 30; 32 equal tokens' 256 on eight of those 37 | 34 | 29; shared as a
// router does, 256 pairs of those 104 | 104 | 125.  32 or 64 rows at a time for what is left hold registers and LDS that the first rows then lack (512
// pairs, eight each: 126 and 160 us, so 113).
template <bool DUAL, int RT, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void gemm_any_stream_groups_kernel(GemmAnyArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[WAVES * stream_slot(DUAL ? 2 : RT, 1)];
  const int share = a.M, own = (int)blockIdx.z - share;   // (among the first arguments: the grid's size is a line of its own)
  auto weights = [&](const void* w, int g) { return static_cast<const uint16_t*>(w) + (int64_t)g * a.N * a.K; };
  int g, m_lo, m_hi;
  if (own >= 0) {
    m_lo = a.group_offsets[own], m_hi = a.group_offsets[own + 1];
    stream_rows<DUAL, 1, RT, WAVES, false>(a, lds, weights(a.w, own), DUAL ? weights(a.w2, own) : nullptr, m_lo, share ? min(m_hi, m_lo + 16) : m_hi);
    return;
  }
  for (int piece = blockIdx.z; group_tile<16, 16>(a.group_offsets, a.n_groups, piece, g, m_lo, m_hi); piece += share) {
    stream_rows<DUAL, 1, RT, WAVES, false>(a, lds, weights(a.w, g), DUAL ? weights(a.w2, g) : nullptr, m_lo, min(m_hi, m_lo + 16));
    __syncthreads();  // (the sums are read)
  }
}

// ---------------------------------------------------------------------------------------------------------------
// few rows: one wave per FT output features and batch of MT rows (blockIdx.y); the lanes take K in pieces of 8, ascending,
// 16-byte loads where the operands allow it, then a butterfly over the lanes
// ---------------------------------------------------------------------------------------------------------------
// Bound by what is asked for at a time: the rows' pieces are loaded without a branch (rows beyond the end: the last one again, not
// stored), so that a K piece is one round trip and not one per row - a router's 32 rows x 64 features x 2048 10.7 -> 6.7 us - and
// four features share the rows' pieces where there are enough features for the chip (N 32768, K 2048: 8 rows 110 us with one feature
// and a branch per row, 76 so, 4 rows 62 / 40; a single row 31 with one feature, 36 with four).
// UNROLL: K pieces that are asked for together; more than one only where all lanes have as many pieces - the last ones, which some lanes
// lack, would be a pass of their own (64 rows x 1024 features x 1000 18.5 us, one at a time 13.2).
template <typename TW, int MT, int FT, bool DUAL, bool EXT, int UNROLL = (FT == 1 ? 2 : 1)>
__global__ __launch_bounds__(256) void gemm_any_rows_kernel(GemmAnyArgs a) {
  static_assert(FT == 1 || !DUAL, "several features: one weight");
  constexpr int WN = DUAL ? 2 : FT;
  const int lane = threadIdx.x & 63;
  const int n = (blockIdx.x * 4 + (threadIdx.x >> 6)) * FT;
  int m_lo, m_hi;
  const TW *w, *w2;
  select_group<TW, DUAL>(a, w, w2, m_lo, m_hi);
  const int m0 = m_lo + blockIdx.y * MT;
  if (n >= a.N || m0 >= m_hi) return;  // (whole waves: the reductions below see all 64 lanes)
  const bool w_vec = a.K % 8 == 0 && dev_aligned16(a.w) && (!DUAL || dev_aligned16(a.w2));
  const bool x_vec = a.ldx % 4 == 0 && dev_aligned16(a.x);
  float acc[WN][MT] = {};
  const float* xp[MT];
  const TW* wp[WN];
#pragma unroll
  for (int r = 0; r < MT; ++r) {
    const int m = min(m0 + r, m_hi - 1);
    xp[r] = a.x + (int64_t)(a.x_rows ? a.x_rows[m] : m) * a.ldx;
  }
#pragma unroll
  for (int f = 0; f < FT; ++f) wp[f] = w + (int64_t)min(n + f, a.N - 1) * a.K;
  if (DUAL) wp[WN - 1] = w2 + (int64_t)n * a.K;
  auto piece = [&](int k0, bool wv_, bool xv_) __attribute__((always_inline)) {
    float wv[WN][8], xv[MT][8];
#pragma unroll
    for (int f = 0; f < WN; ++f) load8<TW>(wp[f] + k0, a.K - k0, wv_, wv[f]);
#pragma unroll
    for (int r = 0; r < MT; ++r) load8<float>(xp[r] + k0, a.K - k0, xv_, xv[r]);
#pragma unroll
    for (int r = 0; r < MT; ++r)
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int f = 0; f < WN; ++f) acc[f][r] = fmaf(xv[r][i], wv[f][i], acc[f][r]);
  };
  if (w_vec && x_vec && UNROLL > 1 && a.K % (64 * 8) == 0) {   // (K % 8 == 0: every piece is whole)
#pragma unroll UNROLL
    for (int k0 = lane * 8; k0 < a.K; k0 += 64 * 8) piece(k0, true, true);
  } else if (w_vec && x_vec) {
#pragma unroll 1
    for (int k0 = lane * 8; k0 < a.K; k0 += 64 * 8) piece(k0, true, true);
  } else {
    for (int k0 = lane * 8; k0 < a.K; k0 += 64 * 8) piece(k0, w_vec, x_vec);
  }
#pragma unroll
  for (int f = 0; f < FT; ++f)
#pragma unroll
    for (int r = 0; r < MT; ++r) {
      const float v = wave_sum(acc[f][r]);
      const float v2 = DUAL ? wave_sum(acc[WN - 1][r]) : 0.f;
      if (lane == 0 && m0 + r < m_hi && n + f < a.N) {
        const int64_t yrow = a.y_rows ? a.y_rows[m0 + r] : m0 + r;
        a.y[yrow * a.ldy + n + f] = finish<DUAL, EXT>(a, m0 + r, yrow, n + f, v, v2);
      }
    }
}

// butterfly steps OFF, OFF / 2, ... over 2 HALF sums: after a step a lane goes on with the half of them that its side keeps
template <int HALF, int OFF, int C>
__device__ __forceinline__ void halve_sums(float (&v)[C], int lane) {
  const bool up = lane & OFF;
#pragma unroll
  for (int i = 0; i < HALF; ++i) {
    if constexpr (OFF >= 16) {   // (the swap of the one's upper lanes with the other's lower ones is the exchange)
      const uint32_t lo = __float_as_uint(v[i]), hi = __float_as_uint(v[i + HALF]);
      const auto r = OFF == 32 ? __builtin_amdgcn_permlane32_swap(lo, hi, false, false) : __builtin_amdgcn_permlane16_swap(lo, hi, false, false);
      v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    } else {
      const float keep = up ? v[i + HALF] : v[i], give = up ? v[i] : v[i + HALF];
      v[i] = keep + xor_get<OFF>(give);
    }
  }
  if constexpr (HALF > 1) halve_sums<HALF / 2, OFF / 2>(v, lane);
}

// The same for 2 to 8 rows of wide products (the heads of a few sequences): the rows lie in LDS, so that a wave's only requests are its
// weights, the next piece's ahead of the arithmetic; persistent workgroups of eight waves, two per CU, so that the rows are laid out
// once.  The sums are gemm_any_rows_kernel's, in its order: a lane's pieces ascending, then the butterfly - of which a lane continues only the
// half of the sums that its side of the step keeps (32 exchanges instead of 192).  A row's pieces of eight lie as their first and
// their second halves: 16-byte reads of neighbouring lanes on neighbouring banks.
// Bound by the weights (us, weights beyond the caches, gemm_any_rows_kernel / here, TB/s here): 8 rows x 32768 x 2048 76.7 / 32.5 (4.1), x 151936
// x 1024 211 / 62.9 (4.9); 4 rows 41.7 / 28.5 (4.7) and 113 / 54.9 (5.7).
template <int MT, bool EXT>
__global__ __launch_bounds__(512, 4) void gemm_any_rows_lds_kernel(GemmAnyArgs a) {
  constexpr int FT = 4, C = FT * MT;
  extern __shared__ __attribute__((aligned(16))) f32x4 xs[];  // [MT][2][K / 8]
  const int lane = threadIdx.x & 63, np = a.K / 8, pieces = a.K / 512;
  for (int i = threadIdx.x; i < MT * 2 * np; i += 512) {
    const int r = i / (2 * np), c = i - r * 2 * np, m = min(r, a.M - 1);
    xs[r * 2 * np + (c & 1) * np + (c >> 1)] = *reinterpret_cast<const f32x4*>(a.x + (int64_t)(a.x_rows ? a.x_rows[m] : m) * a.ldx + c * 4);
  }
  __syncthreads();
  const int quads = (a.N + FT - 1) / FT, step = gridDim.x * 8;
  const uint16_t* const w = static_cast<const uint16_t*>(a.w) + lane * 8;
  u32x4 next[FT];
  auto ask = [&](int q, int p) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < FT; ++f)
      next[f] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w + (int64_t)min(q * FT + f, a.N - 1) * a.K + p * 512));
  };
  int q = blockIdx.x * 8 + (threadIdx.x >> 6);
  if (q >= quads) return;  // (whole waves, behind the only barrier)
  ask(q, 0);
  for (; q < quads; q += step) {
    float acc[C] = {};
    for (int p = 0; p < pieces; ++p) {
      u32x4 now[FT];
#pragma unroll
      for (int f = 0; f < FT; ++f) now[f] = next[f];
      const bool last = p + 1 == pieces;
      ask(last ? min(q + step, quads - 1) : q, last ? 0 : p + 1);
#pragma unroll
      for (int r = 0; r < MT; ++r) {
        const f32x4 x0 = xs[r * 2 * np + p * 64 + lane], x1 = xs[r * 2 * np + np + p * 64 + lane];
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int f = 0; f < FT; ++f)
            acc[f * MT + r] = fmaf(i < 4 ? x0[i & 3] : x1[i & 3], i & 1 ? hi_bf(now[f][i >> 1]) : lo_bf(now[f][i >> 1]), acc[f * MT + r]);
      }
    }
    halve_sums<C / 2, 32>(acc, lane);
    float v = acc[0];
    if constexpr (C == 16) v = xor_sum<2>(v);
    v = xor_sum<1>(v);
    const int idx = lane / (64 / C), m = idx % MT, n = q * FT + idx / MT;
    if (lane % (64 / C) == 0 && m < a.M && n < a.N) {
      const int64_t yrow = a.y_rows ? a.y_rows[m] : m;
      a.y[yrow * a.ldy + n] = finish<false, EXT>(a, m, yrow, n, v, 0.f);
    }
  }
}

// The same one row after the other, for groups that have one or none each (the experts of a token or two): a batch would multiply its
// empty places too, and its registers leave too few waves to keep the weights coming.  us, gate and up / down, batches of 8 | here:
// 8 pairs of 64 experts of 768 x 2048 33.7 / 37.4 | 15.2 / 14.9, 4 of 32 of 512 x 1024 6.5 / 5.6 | 5.1 / 4.7 (fp32, 8 pairs: 12.1 / 11.1 |
// 7.3 / 5.7); all eight in one expert 12.8 / 14.8 | 22.3 / 14.7.
template <typename TW, bool DUAL, bool EXT>
__global__ __launch_bounds__(256) void gemm_any_each_row_kernel(GemmAnyArgs a) {
  const int lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  int m_lo, m_hi;
  const TW *w, *w2;
  select_group<TW, DUAL>(a, w, w2, m_lo, m_hi);
  if (n >= a.N) return;  // (whole waves)
  const bool w_vec = a.K % 8 == 0 && dev_aligned16(a.w) && (!DUAL || dev_aligned16(a.w2));
  const bool x_vec = a.ldx % 4 == 0 && dev_aligned16(a.x);
  w += (int64_t)n * a.K;
  if (DUAL) w2 += (int64_t)n * a.K;
  for (int m = m_lo + blockIdx.y; m < m_hi; m += gridDim.y) {
    const float* x = a.x + (int64_t)(a.x_rows ? a.x_rows[m] : m) * a.ldx;
    float acc = 0.f, acc2 = 0.f;
    auto piece = [&](int k0, bool wv_, bool xv_) __attribute__((always_inline)) {
      float xv[8], wv[8], wv2[8];
      load8<TW>(w + k0, a.K - k0, wv_, wv);
      if (DUAL) load8<TW>(w2 + k0, a.K - k0, wv_, wv2);
      load8<float>(x + k0, a.K - k0, xv_, xv);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        acc = fmaf(xv[i], wv[i], acc);
        if (DUAL) acc2 = fmaf(xv[i], wv2[i], acc2);
      }
    };
    if (w_vec && x_vec && a.K % (64 * 8) == 0) {
#pragma unroll 2
      for (int k0 = lane * 8; k0 < a.K; k0 += 64 * 8) piece(k0, true, true);
    } else if (w_vec && x_vec) {
#pragma unroll 1
      for (int k0 = lane * 8; k0 < a.K; k0 += 64 * 8) piece(k0, true, true);
    } else {
      for (int k0 = lane * 8; k0 < a.K; k0 += 64 * 8) piece(k0, w_vec, x_vec);
    }
    const float v = wave_sum(acc), v2 = DUAL ? wave_sum(acc2) : 0.f;
    if (lane == 0) {
      const int64_t yrow = a.y_rows ? a.y_rows[m] : m;
      a.y[yrow * a.ldy + n] = finish<DUAL, EXT>(a, m, yrow, n, v, v2);
    }
  }
}

// Where the streaming kernel is the faster one of it and the tile kernels (us, tile kernels / here).  Without groups and batches every workgroup's
// copy of the rows outweighs its weights from some number of features on: 24 rows x 32768 x 2048 34.4 / 34.1, 32 x 16384 x 1024 12.0 / 11.5,
// 48 x 6144 x 2048 14.8 / 13.7, 64 x 4096 x 1024 10.3 / 8.8, 33 x 2048 x 1024 9.3 / 6.4; and, against tile kernels with a longer K loop than now, 32 x 32768 x
// 2048 36.2 / 37.0, 48 x 16384 x 1024 12.3 / 14.2, 64 x 16384 x 1024 12.8 / 19.9 (the tile kernels now 34.6, 12.1, 12.8).  So are the ratios that follow.
// Beyond 16384 features and 16 rows a short K is too little work per workgroup (24 x 18432: K 64 1.09 times the tile kernels' time, 256 1.04,
// 512 0.94, now 10.4 / 9.9 us); between 8192 and 16384 features a long one leaves a part round of long workgroups (24 x 12288: K 1024 0.95, 2048 1.02, 4096 1.15; 16
// rows: 2048 0.90, 4096 1.03; 24 x 16384 x 8192 1.07).  Two weights: 17 rows x 12288 and 16384, K to 1024 1.00 to 1.20, from 2048 on 0.78 to 0.87;
// 9 rows x 16384, K 128 1.09, 256 0.96.
// Grouped: up to ten rows a group on average, eight where K is below 1024 (64 experts of 768 x 2048, 8 each 128 / 107, now 136 / 118, 10 each 120 / 111; 128 of 256
// x 512, 10 each 31.8 / 34.6) and none of many short products (944 pairs, 128 experts of 768 x 256: 41 / 54).
bool any_stream_takes(int rows, int N, int K, int n_groups, bool dual) {
  if (rows <= 8 || K % 64) return false;
  if (n_groups) return rows <= (K < 1024 ? 8 : 10) * (int64_t)n_groups && !(K <= 256 && (int64_t)n_groups * N >= 65536);
  if (rows > 64) return false;
  const int most = rows <= 24 ? INT32_MAX : rows <= 32 ? 16384 : rows <= 48 ? 6144 : 4096;
  if (dual) return N <= std::min(most, rows <= 16 ? (K <= 128 ? 12288 : most) : K <= 1024 ? 8192 : most);
  if (rows > 16 && ((N > 16384 && K < 512) || (N > 8192 && K >= 8192))) return false;
  return N <= most && !(N > 8192 && N < 16384 && K >= (rows > 16 ? 2048 : 4096));
}

// Batches (64 rows a batch at most: the features of a head); many of one 64-deep block each are slower so (32 of 64 rows x 512 x 64: 6.9 us on
// gemm_any_skinny_kernel, 7.9)
static bool batches_stream(int rows, int N, int K, int n_batch) { return rows <= 64 && K % 64 == 0 && !(K == 64 && (int64_t)n_batch * N > 8192); }

template <bool DUAL, bool EXT>
static int launch_stream(const GemmAnyArgs& args, int groups, int rows, hipStream_t st) {
  GemmAnyArgs a = args;
  a.n_groups = groups;
  int z = groups;
  auto go = [&](auto kernel, int rt, int waves) {
    hipLaunchKernelGGL(kernel, dim3((a.N + 16 * rt - 1) / (16 * rt), 1, z), dim3(64 * waves), 0, st, a);
    return check_launch();
  };
  // groups and batches: workgroups enough, four waves each, so that several share a CU (eight: 256 pairs over 64 experts' second product 55
  // us, four 37)
  if (a.group_offsets) {   // (no group has the extended epilogue)
    // up to 96 rows a group's own workgroups walk them all, six times sixteen at most: the choice costs every launch 0.3 us (96 pairs, 32 experts of
    // 512 x 1024: 24.0 us so, 24.6)
    const bool wide = !DUAL && (int64_t)(a.N / 16) * groups >= 2048;
    if constexpr (!EXT) {
      if (rows <= 96) {
        if constexpr (!DUAL)
          if (wide) return go(gemm_any_stream_kernel<false, 1, 2, 4, false>, 2, 4);
        return go(gemm_any_stream_kernel<DUAL, 1, 1, 4, false>, 1, 4);
      }
      // (`rows` rows in all have at most twice as many sixteens beyond a group's first, and seldom as many: few stay without one)
      a.M = std::min((rows + 31) / 32, 65535 - groups);
      z = groups + a.M;
      if constexpr (!DUAL)
        if (wide) return go(gemm_any_stream_groups_kernel<false, 2, 4>, 2, 4);
      return go(gemm_any_stream_groups_kernel<DUAL, 1, 4>, 1, 4);
    }
    return MI_EUNSUPPORTED;
  }
  const int mf = (rows + 15) / 16;
  if constexpr (!DUAL && !EXT) {   // (no batch has two weights or the extended epilogue)
    if (groups > 1) {
      switch (mf) {
        case 1:
          return (int64_t)(a.N / 16) * groups >= 2048 ? go(gemm_any_stream_kernel<false, 1, 2, 4, false>, 2, 4)
                                                      : go(gemm_any_stream_kernel<false, 1, 1, 4, false>, 1, 4);
        case 2: return go(gemm_any_stream_kernel<false, 2, 1, 4, false>, 1, 4);
        case 3: return go(gemm_any_stream_kernel<false, 3, 1, 4, false>, 1, 4);
        default: return go(gemm_any_stream_kernel<false, 4, 1, 4, false>, 1, 4);
      }
    }
  }
  if constexpr (DUAL) {
    switch (mf) {
      case 1: return go(gemm_any_stream_kernel<true, 1, 1, 4, EXT>, 1, 4);
      case 2: return go(gemm_any_stream_kernel<true, 2, 1, 4, EXT>, 1, 4);
      case 3: return go(gemm_any_stream_kernel<true, 3, 1, 4, EXT>, 1, 4);
      default: return go(gemm_any_stream_kernel<true, 4, 1, 4, EXT>, 1, 4);
    }
  } else {
    // more feature tiles than CUs: two per workgroup, half as many copies of x and no part round (24 rows x 6144 x 2048 12.8 / 10.5 us, x 4096 8.6
    // / 9.8; of the tile kernels' time: 48 x 4224 x 2048 1.30 / 0.92, 24 x 5120 x 1024 0.96 / 0.72)
    if (a.N > 4096) {
      switch (mf) {
        case 1: return go(gemm_any_stream_kernel<false, 1, 2, 4, EXT>, 2, 4);
        case 2: return go(gemm_any_stream_kernel<false, 2, 2, 4, EXT>, 2, 4);
        case 3: return go(gemm_any_stream_kernel<false, 3, 2, 4, EXT>, 2, 4);
        default: break;
      }
    }
    switch (mf) {
      case 1: return go(gemm_any_stream_kernel<false, 1, 1, 8, EXT>, 1, 8);
      case 2: return go(gemm_any_stream_kernel<false, 2, 1, 8, EXT>, 1, 8);
      case 3: return go(gemm_any_stream_kernel<false, 3, 1, 8, EXT>, 1, 8);
      default: return go(gemm_any_stream_kernel<false, 4, 1, 4, EXT>, 1, 4);
    }
  }
}

// Exact mode beyond a few rows.  The tile of gemm_any_f32_kernel: a launch takes some 6 us and, per 1024 of K, 18.7 us for every 256 tiles of
// 64 x 64, 9.6 of 32 x 64, 5.05 of 32 x 32 or part of them (the matrix rate, shared by a CU's tiles): the least of the three.  us, the
// largest tile that fills 180 workgroups / this: 721 rows x 1024 x 1024 25.3 / 20.7, x 2048 42.2 / 35.1, x 3072 62.7 / 51.7, 400 rows x 3072
// 42.0 / 32.3; 1000 rows x 4096 keep 64 x 64 (81.1, 83.0, 87.1).  Groups: a last tile each that is half empty on average, and no workgroup for
// a tile that is not there: 32 experts, 1024 -> 2 x 512 / back: 256 pairs 79 / 29 -> 28 / 18, 1600 pairs 69 / 37 -> 53 / 34, 6000 pairs 176 / 92 ->
// 147 / 78; 64 experts, 2048 -> 2 x 768 / back, 512 pairs 304 / 88 -> 162 / 81.
template <typename TW, bool DUAL, bool EXT>
static int launch_exact(const GemmAnyArgs& args, int groups, int rows_per_group_max, hipStream_t st) {
  GemmAnyArgs a = args;
  a.n_groups = groups;
  constexpr int W16 = 16 / (int)sizeof(TW);
  const bool grouped = a.group_offsets != nullptr;
  const bool vec = a.K % 32 == 0 && a.ldx % 4 == 0 && aligned16(a.x) && aligned16(a.w) && (!DUAL || aligned16(a.w2)) && a.K % W16 == 0 &&
                   a.x_batch % 4 == 0;
  if (vec) {
    const auto nx = [&](int bn) { return (a.N + bn - 1) / bn; };
    // groups: a workgroup for every row tile that a group can have while they are few (32 pairs of 16 experts of 512 x 256: 14.1 us so, 16.9 where each
    // looks for its tile); else as many row tiles as rows_per_group_max rows in all groups have at most, and no fewer than four workgroups per
    // CU; what there is beyond (the bound is one group's) the workgroups take behind their first.  (A tile per group and row tile of the bound
    // were 23296 workgroups for 768 tiles: 2900 pairs over 32 experts.)
    auto grid = [&](int bm, int bn) {
      const int ny = (rows_per_group_max + bm - 1) / bm;
      if (!grouped) return dim3(nx(bn), ny, groups);
      const int64_t most = (int64_t)ny * groups;
      if (most * nx(bn) <= 1024) return dim3(nx(bn), ny, groups);
      const int64_t total = rows_per_group_max / bm + groups, fill = (1024 + nx(bn) - 1) / nx(bn);
      return dim3(nx(bn), (unsigned)std::min<int64_t>(std::min(most, std::max(total, fill)), 65535), 1);
    };
    const auto per_cu = [&](int bm, int bn) {
      const int64_t row_tiles = grouped ? rows_per_group_max / bm + (groups + 1) / 2 : (int64_t)((rows_per_group_max + bm - 1) / bm) * groups;
      return (row_tiles * nx(bn) + 255) / 256;
    };
    const auto cost = [&](int bm, int bn, double us) {
      return per_cu(bm, bn) == 1 ? 1.07 * us : (double)per_cu(bm, bn) * us;   // (alone on its CU a tile waits out its own starts)
    };
    // (two weights: 64 x 64 has a CU to itself; the small tiles read their operands most often: beyond two per CU only where it is clear)
    const double large = cost(64, 64, DUAL ? 21.0 : 18.7), medium = cost(32, 64, 9.6), one = cost(32, 32, 5.05), small = one > 11. ? 1.06 * one : one;
    const auto go = [&](auto plain, auto direct, auto found, dim3 g) {   // (no group has the extended epilogue)
      if (!grouped) hipLaunchKernelGGL(plain, g, dim3(256), 0, st, a);
      else if ((int)g.z == groups && groups > 1) hipLaunchKernelGGL(direct, g, dim3(256), 0, st, a);
      else hipLaunchKernelGGL(found, g, dim3(256), 0, st, a);
    };
#define MI_F32_TILE(FM, FN, WM, WN, AHEAD)                                                                                          \
  gemm_any_f32_kernel<TW, DUAL, FM, FN, WM, WN, EXT, 0, AHEAD>, gemm_any_f32_kernel<TW, DUAL, FM, FN, WM, WN, EXT, EXT ? 0 : 1, AHEAD>, \
      gemm_any_f32_kernel<TW, DUAL, FM, FN, WM, WN, EXT, EXT ? 0 : 2, AHEAD>
    // fp32 weights of larger launches: gemm_any_split_kernel, by a model of its own against that of the tiles above (times two for two weights).  Per 1024 of K
    // it takes some 13 us for every 256 tiles of 64 x 64 and 26 for two weights; alone on its CU a tile is a chain of read, split, write and multiply: 6 us more
    // and, two weights, 32.  Without groups from two tiles per CU on.  Two weights of groups, whose last tiles are half empty and which look for their tiles: 30
    // us a round and one round more (launches with a workgroup for every tile of a group are smaller).  One weight of groups is not taken: launches by themselves
    // were 0.92 of the time, a step of four layers with 2831 rows (354 an expert) 3068 us with them and 3003 without.  Over 5600 drawn products (64 to 9000
    // rows, 64 to 6200 features, K 64 to 4096; batches; 2 to 128 groups of up to 45000 pairs in all, even and uneven), one at a time and back to back, those
    // taken: 0.83 of the time above without groups (450 of 2091; two weights 0.77, 104 of 756), batches 0.84 (128 of 380), groups 0.79 (644 of 2115); 7 of
    // them slower by more than 1 % (6 % at most).  us, above / split: 721 rows x 1024 x 1024 25 and not taken, x 3072 61 / 57, 2831 x 1024 x 1024 69 / 58,
    // 4096 x 4096 x 4096 1127 / 991; 32 experts, 1024 -> 2 x 512, 11324 pairs 276 / 241; 64 experts, 2048 -> 2 x 768, 5768 pairs 449 / 486 and not
    // taken, 19688 pairs 1169 / 1067.
    if constexpr (sizeof(TW) == 4) {
      const double row_tiles = grouped ? std::max(rows_per_group_max / 64. + groups / 2., (double)groups) : (double)((rows_per_group_max + 63) / 64) * groups;
      const double n = row_tiles * nx(64) / 256., k = a.K / 1024.;
      const double split_us = grouped ? 30. * k * (n + 1.) : DUAL ? 32. + 26. * k * std::ceil(n) : 6. + 13. * k * std::ceil(n);
      const bool fills = grouped ? DUAL && grid(64, 64).z == 1 : rows_per_group_max / 64. * groups * nx(64) / 256. >= 2.;
      if (a.N > 32 && fills && split_us < std::min(large, std::min(medium, small)) * (DUAL ? 2. : 1.) * k) {
        constexpr bool GROUPS = DUAL && !EXT;   // (the forms that are taken)
        const dim3 g = grid(64, 64);
        if (grouped) hipLaunchKernelGGL((gemm_any_split_kernel<DUAL, EXT, GROUPS>), g, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((gemm_any_split_kernel<DUAL, EXT, false>), g, dim3(256), 0, st, a);
        return check_launch();
      }
    }
    // (fragments a step ahead: see the kernel)
    constexpr bool one_fp32 = !DUAL && sizeof(TW) == 4;
    if (a.N > 32 && large <= medium && large <= small) go(MI_F32_TILE(2, 2, 2, 2, false), grid(64, 64));
    else if (a.N > 32 && medium <= small && one_fp32 && a.K >= 1024 && per_cu(32, 64) <= 5) go(MI_F32_TILE(2, 1, 1, 4, one_fp32), grid(32, 64));
    else if (a.N > 32 && medium <= small) go(MI_F32_TILE(2, 1, 1, 4, false), grid(32, 64));
    else if (one_fp32 || (sizeof(TW) == 2 ? per_cu(32, 32) <= 2 : per_cu(32, 32) == 1 || (per_cu(32, 32) > 2 && a.K >= 1024))) go(MI_F32_TILE(1, 1, 2, 2, true), grid(32, 32));
    else go(MI_F32_TILE(1, 1, 2, 2, one_fp32), grid(32, 32));
#undef MI_F32_TILE
    return check_launch();
  }
  // a router over a prompt: one column of tiles - short tiles, more of them (us, 64 / 16 rows: 1024 rows x 64 features x 1000 93 / 75,
  // 8192 rows x 32 x 1000 100 / 84)
  if (a.N <= 64 && rows_per_group_max >= 1024) {
    hipLaunchKernelGGL((gemm_any_fma_kernel<TW, DUAL, 1, EXT>), dim3(1, (rows_per_group_max + 15) / 16, groups), dim3(256), 0, st, a);
    return check_launch();
  }
  hipLaunchKernelGGL((gemm_any_fma_kernel<TW, DUAL, 4, EXT>), dim3((a.N + 63) / 64, (rows_per_group_max + 63) / 64, groups), dim3(256), 0, st, a);
  return check_launch();
}

template <typename TW, bool DUAL, bool EXT>
static int launch_any(const GemmAnyArgs& a, int groups, int rows_per_group_max, int mode, hipStream_t st) {
  // mode 0: product (MFMA for bf16 weights, the row kernels for few rows); 1: exact (x unrounded: the row kernels, beyond them launch_exact)
  // few rows (per group): the weight-streaming row kernels.  Also the exact mode up to 64 rows: a router's few output
  // features would be one or two tiles of launch_exact's kernels, each walking all of K alone
  const bool few = rows_per_group_max <= 8 || (mode == 1 && rows_per_group_max <= 64);
  if (few) {
    const int mt = rows_per_group_max <= 1 ? 1 : rows_per_group_max <= 4 ? 4 : 8;
    if (a.group_offsets && mt > 1 && rows_per_group_max <= groups) {   // (a group of eight rows and more: over several workgroups)
      hipLaunchKernelGGL((gemm_any_each_row_kernel<TW, DUAL, EXT>), dim3((a.N + 3) / 4, (rows_per_group_max + 7) / 8, groups), dim3(256), 0, st, a);
      return check_launch();
    }
    const int ft = !DUAL && mt > 1 && a.N >= 8192 ? 4 : 1;   // (a wave per four features: from two workgroups per CU on)
    const dim3 grid((a.N + 4 * ft - 1) / (4 * ft), (rows_per_group_max + mt - 1) / mt, groups);
    // From 4096 features on and 12288 sums, in which the layout of the rows and the wide waves pay (us, gemm_any_rows_kernel / here: 2 rows x 4096 x
    // 2048 7.6 / 8.2, 3 rows 9.0 / 8.1, 8 rows 16.4 / 10.7; 2 x 6144 x 2048 9.8 / 9.0; 5 x 3072 x 2048 9.8 / 10.2), 16384 where a row of K is one piece (2 x
    // 6261 x 512 4.4 / 5.0, x 8192 x 512 0.70 of the time); 64 KB of rows at most: two workgroups on a CU.
    if constexpr (!DUAL && sizeof(TW) == 2)
      if (mt > 1 && rows_per_group_max <= 8 && a.N >= 4096 && (int64_t)a.N * rows_per_group_max >= (a.K > 512 ? 12288 : 16384) && groups == 1 && !a.group_offsets && a.K % 512 == 0 && mt * a.K * 4 <= 65536 && a.ldx % 4 == 0 &&
          aligned16(a.x) && aligned16(a.w)) {
        const dim3 persistent(std::min(512, (a.N + 31) / 32));
        if (mt == 4) hipLaunchKernelGGL((gemm_any_rows_lds_kernel<4, EXT>), persistent, dim3(512), mt * a.K * 4, st, a);
        else hipLaunchKernelGGL((gemm_any_rows_lds_kernel<8, EXT>), persistent, dim3(512), mt * a.K * 4, st, a);
        return check_launch();
      }
    if constexpr (!DUAL)
      if (ft == 4) {
        if (mt == 4) hipLaunchKernelGGL((gemm_any_rows_kernel<TW, 4, 4, DUAL, EXT>), grid, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((gemm_any_rows_kernel<TW, 8, 4, DUAL, EXT>), grid, dim3(256), 0, st, a);
        return check_launch();
      }
    const auto rows = [&](auto kernel, int batch) {
      hipLaunchKernelGGL(kernel, dim3(grid.x, (rows_per_group_max + batch - 1) / batch, groups), dim3(256), 0, st, a);
      return check_launch();
    };
    // A batch's empty places are multiplied too, and the registers of many rows and of two pieces leave few waves.  So up to seven rows are
    // a batch of their own, and from five on the lanes take a piece at a time, at eight from 4096 weight rows on.  us, four or eight rows
    // with two pieces / as here: 2 x 6144 x 2048 9.4 / 6.6, 5 x 6144 x 2048 16.8 / 11.6, 6 x 4096 x 2568 19.2 / 13.6, 8 x 8000 x 1000
    // 19.9 / 13.4; 8 x 1024 x 1024 keeps two pieces (5.5, one 5.7).  Groups, and more than one batch (exact mode): four rows, a piece at a
    // time (fp32 weights: 9 rows x 3072 x 1024 10.5 / 8.1, 64 rows 36 / 31, 64 x 1024 x 1000 18.5 / 12.9; experts' gate and up, 36 pairs
    // of 32 of 512 x 1024 34.3 / 19.4) - except over weights beyond the L2s, which would be read twice as often (64 x 6144 x 2048, 50 MB:
    // 119 / 139).
    if (mt == 1) return rows(gemm_any_rows_kernel<TW, 1, 1, DUAL, EXT>, 1);
    if (rows_per_group_max <= 8 && !a.group_offsets) {
      if (rows_per_group_max == 2) return rows(gemm_any_rows_kernel<TW, 2, 1, DUAL, EXT>, 2);
      if (rows_per_group_max == 3) return rows(gemm_any_rows_kernel<TW, 3, 1, DUAL, EXT>, 3);
      if (rows_per_group_max == 4) return rows(gemm_any_rows_kernel<TW, 4, 1, DUAL, EXT>, 4);
      if (rows_per_group_max == 5) return rows(gemm_any_rows_kernel<TW, 5, 1, DUAL, EXT, 1>, 5);
      if (rows_per_group_max == 6) return rows(gemm_any_rows_kernel<TW, 6, 1, DUAL, EXT, 1>, 6);
      if (rows_per_group_max == 7) return rows(gemm_any_rows_kernel<TW, 7, 1, DUAL, EXT, 1>, 7);
      if ((int64_t)a.N * (DUAL ? 2 : 1) >= 4096) return rows(gemm_any_rows_kernel<TW, 8, 1, DUAL, EXT, 1>, 8);
    } else if (a.group_offsets || (int64_t)a.N * a.K * (int64_t)sizeof(TW) <= (32 << 20)) {
      return rows(gemm_any_rows_kernel<TW, 4, 1, DUAL, EXT, 1>, 4);
    }
    return rows(gemm_any_rows_kernel<TW, 8, 1, DUAL, EXT>, 8);
  }
  const dim3 grid((a.N + 63) / 64, (rows_per_group_max + 63) / 64, groups);
  if constexpr (sizeof(TW) == 2) {
    const bool batches = !a.group_offsets && groups > 1;
    if (mode == 0 && (batches ? batches_stream(rows_per_group_max, a.N, a.K, groups) : any_stream_takes(rows_per_group_max, a.N, a.K, a.group_offsets ? groups : 0, DUAL)) &&
        a.ldx % 4 == 0 && a.x_batch % 4 == 0 && aligned16(a.x) && aligned16(a.w) && (!DUAL || aligned16(a.w2)))
      return launch_stream<DUAL, EXT>(a, groups, rows_per_group_max, st);
    if (mode == 0 && rows_per_group_max >= 512 && a.N >= 128) {  // prefill-sized: 128-row tiles, 128 (SwiGLU: 64) features
      if (DUAL) {
        hipLaunchKernelGGL((gemm_any_mfma_kernel<DUAL, 4, 2, EXT>), dim3((a.N + 63) / 64, (rows_per_group_max + 127) / 128, groups),
                           dim3(256), 0, st, a);
      } else {
        hipLaunchKernelGGL((gemm_any_mfma_kernel<DUAL, 4, 4, EXT>), dim3((a.N + 127) / 128, (rows_per_group_max + 127) / 128, groups),
                           dim3(256), 0, st, a);
      }
      return check_launch();
    }
    if (mode == 0 && (rows_per_group_max <= 64 || (groups > 1 && rows_per_group_max <= 8 * groups))) {
      // decode-sized: 16-feature workgroups (grouped: tiles of 32 rows, an expert's few rows fill the first)
      if (groups > 1 || rows_per_group_max <= 32) {
        const dim3 g2((a.N + 15) / 16, (rows_per_group_max + 31) / 32, groups);
        hipLaunchKernelGGL((gemm_any_skinny_kernel<DUAL, 2, EXT>), g2, dim3(256), 0, st, a);
      } else {
        const dim3 g4((a.N + 15) / 16, 1, groups);
        hipLaunchKernelGGL((gemm_any_skinny_kernel<DUAL, 4, EXT>), g4, dim3(256), 0, st, a);
      }
      return check_launch();
    }
    if (mode == 0) {
      hipLaunchKernelGGL((gemm_any_mfma_kernel<DUAL, 2, 2, EXT>), grid, dim3(256), 0, st, a);
      return check_launch();
    }
  }
  return launch_exact<TW, DUAL, EXT>(a, groups, rows_per_group_max, st);
}

// Per-head products of many rows (latent attention's: 8192 rows x 16 heads, 128 -> 256 and back).  What bounds it: memory - x in and y
// out are 24 KiB per 16 rows of a head, its 64 KiB of weights the only reuse.  So no operand pass and no x tile: a workgroup keeps ONE
// head's weight in LDS (rows padded by 16 bytes: a lane group's sixteen rows in sixteen bank slots), and its eight waves walk 16-row
// tiles, x rows from memory into the MFMA operand (rounded to bf16 once, as gemm_any_mfma_kernel does), the next tile's rows requested
// before this one is multiplied; two workgroups per CU.  gemm_any_mfma_kernel (both operands through LDS for every 64 features, two barriers per K
// step): 128 -> 256 160 us, 256 -> 128 98 us; here 48 and 43 (4.2 and 4.7 TB/s).  Same summation order (k ascending in one chain), same bits.
// Fewer rows and heads than CUs: a head's features are shared by several workgroups (blockIdx.y, n_share features each): 4 heads of 185 rows, 64 -> 512
// 5.5 us on gemm_any_mfma_kernel, 10.3 with a workgroup per 128 rows, 3.4 so; 16 of 318, 128 -> 256 8.0 / 10.4 / 6.0.
constexpr int kHeadsWeightElems = 32768, kHeadsLds = 2 * kHeadsWeightElems + 16 * 512;
template <int KF>  // K = 32 KF (256: one workgroup per CU, the next rows' registers)
__global__ __launch_bounds__(512, KF == 8 ? 2 : 4) void gemm_any_heads_kernel(GemmAnyArgs a, int n_share) {
  __shared__ __attribute__((aligned(16))) char lds[kHeadsLds];
  constexpr int K = 32 * KF, ROW = 2 * K + 16;
  const int lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int m_lo, m_hi;
  const uint16_t *w, *w2;
  select_group<uint16_t, false>(a, w, w2, m_lo, m_hi);
  const int n_lo = blockIdx.y * n_share, n_count = min(a.N - n_lo, n_share);
  for (int i = threadIdx.x; i < n_count * (K / 8); i += 512)
    *reinterpret_cast<u32x4*>(lds + (i / (K / 8)) * ROW + (i % (K / 8)) * 16) = *reinterpret_cast<const u32x4*>(w + (int64_t)n_lo * K + (int64_t)i * 8);
  f32x4 raw[KF][2];
  auto request = [&](int m0) __attribute__((always_inline)) {
    const float* xp = a.x + (int64_t)min(m0 + r16, m_hi - 1) * a.ldx + q * 8;
#pragma unroll
    for (int ks = 0; ks < KF; ++ks) {
      raw[ks][0] = *reinterpret_cast<const f32x4*>(xp + ks * 32);
      raw[ks][1] = *reinterpret_cast<const f32x4*>(xp + ks * 32 + 4);
    }
  };
  int m0 = (blockIdx.x * 8 + wave) * 16;
  const int step = gridDim.x * 128;
  request(m0);
  __syncthreads();
  for (; m0 < m_hi; m0 += step) {
    bf16x8 xf[KF];
#pragma unroll
    for (int ks = 0; ks < KF; ++ks)
      xf[ks] = as_frag(u32x4{pack_bf(raw[ks][0][0], raw[ks][0][1]), pack_bf(raw[ks][0][2], raw[ks][0][3]), pack_bf(raw[ks][1][0], raw[ks][1][1]),
                             pack_bf(raw[ks][1][2], raw[ks][1][3])});
    request(m0 + step);   // (past the last tile: the last row again)
    const int m = m0 + r16;
    float* yp = a.y + (int64_t)m * a.ldy + n_lo + q * 4;
    const float* gp = a.gate ? a.gate + (int64_t)min(m, m_hi - 1) * a.ldgate + n_lo + q * 4 : nullptr;
    for (int n = 0; n < n_count; n += 32) {
      f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int ks = 0; ks < KF; ++ks)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              as_frag(*reinterpret_cast<const u32x4*>(lds + (n + t * 16 + r16) * ROW + ks * 64 + q * 16)), xf[ks], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (gp) {
          const f32x4 g = *reinterpret_cast<const f32x4*>(gp + n + t * 16);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[t][e] *= 1.f / (1.f + expf(-g[e]));
        }
        if (m < m_hi) *reinterpret_cast<f32x4*>(yp + n + t * 16) = acc[t];
      }
    }
  }
}
// x, y and gate rows in 16-byte pieces, whole 32-feature steps, a head's weight in LDS; up to 64 rows the products stream their weights, and many heads of
// up to 128 rows stay where they were at K 256 (16 of 128 rows, 64 features: 1.20 times as long here; 8 heads 0.86)
static bool heads_takes(const GemmAnyArgs& a, int w_dtype, int n_batch, bool exact) {
  return !exact && w_dtype == MI_DTYPE_BF16 && n_batch > 1 && a.M > 64 && (a.K == 64 || a.K == 128 || a.K == 256) && a.N > 0 &&
         !(a.K == 256 && a.M <= 128 && n_batch >= 16) && a.N % 32 == 0 && a.N <= 512 && a.N * a.K <= kHeadsWeightElems && aligned16(a.x) && aligned16(a.w) && aligned16(a.y) &&
         a.ldx % 4 == 0 && a.x_batch % 4 == 0 && a.ldy % 4 == 0 && a.y_batch % 4 == 0 &&
         (!a.gate || (aligned16(a.gate) && a.ldgate % 4 == 0 && a.gate_batch % 4 == 0));
}
static int launch_heads(const GemmAnyArgs& a, int n_batch, hipStream_t st) {
  const int rows = (a.M + 127) / 128, fill = ((a.K == 256 ? 256 : 512) + n_batch - 1) / n_batch;   // (the workgroups that run together)
  const int gx = rows < fill ? rows : fill, steps = a.N / 32;
  const int slices = std::min(steps, std::max(1, 256 / (gx * n_batch))), n_share = (steps + slices - 1) / slices * 32;
  const dim3 grid(gx, (a.N + n_share - 1) / n_share, n_batch);
  if (a.K == 64) hipLaunchKernelGGL((gemm_any_heads_kernel<2>), grid, dim3(512), 0, st, a, n_share);
  else if (a.K == 128) hipLaunchKernelGGL((gemm_any_heads_kernel<4>), grid, dim3(512), 0, st, a, n_share);
  else hipLaunchKernelGGL((gemm_any_heads_kernel<8>), grid, dim3(512), 0, st, a, n_share);
  return check_launch();
}

}  // namespace mi

using namespace mi;

static int gemm_any_dispatch(const GemmAnyArgs& a, int w_dtype, int groups, int rows_max, int mode, hipStream_t st) {
  if (a.M == 0 || a.N == 0 || rows_max == 0) return MI_OK;
  if (w_dtype != MI_DTYPE_BF16 && w_dtype != MI_DTYPE_F32) return MI_EINVAL;
  const bool bf16 = w_dtype == MI_DTYPE_BF16;
  if (a.w2) return bf16 ? launch_any<uint16_t, true, false>(a, groups, rows_max, mode, st) : launch_any<float, true, false>(a, groups, rows_max, mode, st);
  if (a.ext) return bf16 ? launch_any<uint16_t, false, true>(a, groups, rows_max, mode, st) : launch_any<float, false, true>(a, groups, rows_max, mode, st);
  return bf16 ? launch_any<uint16_t, false, false>(a, groups, rows_max, mode, st) : launch_any<float, false, false>(a, groups, rows_max, mode, st);
}

static bool act_ok(int act) { return (act >= MI_ACT_NONE && act <= MI_ACT_SOFTCAP) || act == MI_ACT_RELU2; }
static bool act_ext_ok(int act) { return (act_ok(act) && act != MI_ACT_SOFTCAP) || act == MI_ACT_TANH || act == MI_ACT_DECAY; }

extern "C" int mi_gemm_any_streams(int rows, int N, int K, int n_groups) { return any_stream_takes(rows, N, K, n_groups, false) ? 1 : 0; }

extern "C" int mi_gemm_any(const float* x, int64_t ldx, const void* w, int w_dtype, float* y, int64_t ldy, int M, int N,
                           int K, float alpha, int exact, mi_stream stream) {
  return mi_gemm_any_act(x, ldx, w, nullptr, w_dtype, nullptr, nullptr, MI_ACT_NONE, y, ldy, M, N, K, alpha, exact, stream);
}

extern "C" int mi_gemm_any_act(const float* x, int64_t ldx, const void* w, const void* w2, int w_dtype, const float* bias,
                               const float* bias2, int act, float* y, int64_t ldy, int M, int N, int K, float alpha,
                               int exact, mi_stream stream) {
  if (!x || !w || !y || M < 0 || N < 0 || K < 1 || ldx < K || ldy < N || !act_ok(act) || (bias2 && !w2)) return MI_EINVAL;
  if (act == MI_ACT_SOFTCAP && (w2 || !(alpha > 0.f))) return MI_EINVAL;
  GemmAnyArgs a{x, ldx, w, w2, y, ldy, M, N, K, alpha, nullptr, nullptr, nullptr, bias, bias2, act, nullptr, 0, 0, 0, 0, nullptr, nullptr, 0.f, false, 0, 0, 0};
  return gemm_any_dispatch(a, w_dtype, 1, M, exact ? 1 : 0, S(stream));
}

extern "C" int mi_gemm_any_segments(const float* x, int64_t ldx, const void* w, int w_dtype, const float* bias, int act,
                                    int act_from, int act2, int act2_from, float* y, int64_t ldy, int M, int N, int K,
                                    int exact, mi_stream stream) {
  if (!x || !w || !y || M < 0 || N < 0 || K < 1 || ldx < K || ldy < N || !act_ext_ok(act) || !act_ext_ok(act2)) return MI_EINVAL;
  if (act_from < 0 || act2_from < act_from) return MI_EINVAL;
  GemmAnyArgs a{x, ldx, w, nullptr, y, ldy, M, N, K, 1.0f, nullptr, nullptr, nullptr, bias, nullptr, act, nullptr, 0, 0, 0, 0, nullptr, nullptr, 0.f, true, act_from, act2, act2_from};
  return gemm_any_dispatch(a, w_dtype, 1, M, exact ? 1 : 0, S(stream));
}

extern "C" int mi_gemm_any_batched(const float* x, int64_t ldx, int64_t x_batch, const void* w, int w_dtype, float* y,
                                   int64_t ldy, int64_t y_batch, const float* gate, int64_t ldgate, int64_t gate_batch,
                                   int n_batch, int M, int N, int K, int exact, mi_stream stream) {
  if (!x || !w || !y || n_batch < 1 || M < 0 || N < 0 || K < 1 || ldx < K || ldy < N) return MI_EINVAL;
  if (n_batch > 65535) return MI_EUNSUPPORTED;
  GemmAnyArgs a{x, ldx, w, nullptr, y, ldy, M, N, K, 1.0f, nullptr, nullptr, nullptr, nullptr, nullptr, MI_ACT_NONE,
                gate, ldgate, x_batch, y_batch, gate_batch, nullptr, nullptr, 0.f, false, 0, 0, 0};
  if (heads_takes(a, w_dtype, n_batch, exact != 0)) return launch_heads(a, n_batch, S(stream));
  return gemm_any_dispatch(a, w_dtype, n_batch, M, exact ? 1 : 0, S(stream));
}

extern "C" int mi_gemm_any_grouped(const float* x, int64_t ldx, const int32_t* x_rows, const void* w, const void* w2,
                                   int w_dtype, const int32_t* group_offsets, int n_groups, int rows_per_group_max,
                                   float* y, int64_t ldy, const int32_t* y_rows, int N, int K, int exact,
                                   mi_stream stream) {
  return mi_gemm_any_grouped_act(x, ldx, x_rows, w, w2, w_dtype, w2 ? MI_ACT_SILU : MI_ACT_NONE, group_offsets, n_groups,
                                 rows_per_group_max, y, ldy, y_rows, N, K, exact, stream);
}

extern "C" int mi_gemm_any_grouped_act(const float* x, int64_t ldx, const int32_t* x_rows, const void* w, const void* w2,
                                       int w_dtype, int act, const int32_t* group_offsets, int n_groups,
                                       int rows_per_group_max, float* y, int64_t ldy, const int32_t* y_rows, int N, int K,
                                       int exact, mi_stream stream) {
  if (act == MI_ACT_CLAMPED_GLU) return MI_EINVAL;  // (needs its limit: mi_gemm_any_grouped_glu)
  return mi_gemm_any_grouped_glu(x, ldx, x_rows, w, w2, w_dtype, act, 0.f, nullptr, nullptr, group_offsets, n_groups,
                                 rows_per_group_max, y, ldy, y_rows, N, K, exact, stream);
}

extern "C" int mi_gemm_any_grouped_glu(const float* x, int64_t ldx, const int32_t* x_rows, const void* w, const void* w2,
                                       int w_dtype, int act, float limit, const float* row_scale,
                                       const int32_t* row_scale_rows, const int32_t* group_offsets, int n_groups,
                                       int rows_per_group_max, float* y, int64_t ldy, const int32_t* y_rows, int N, int K,
                                       int exact, mi_stream stream) {
  if (!x || !w || !y || !group_offsets || n_groups < 1 || rows_per_group_max < 0 || N < 0 || K < 1 ||
      !(act_ok(act) || act == MI_ACT_CLAMPED_GLU) || act == MI_ACT_SOFTCAP)
    return MI_EINVAL;
  if (act == MI_ACT_CLAMPED_GLU && (!w2 || !(limit > 0.f))) return MI_EINVAL;
  if (row_scale_rows && !row_scale) return MI_EINVAL;
  if (n_groups > 65535) return MI_EUNSUPPORTED;
  GemmAnyArgs a{x, ldx, w, w2, y, ldy, rows_per_group_max, N, K, 1.0f, group_offsets, x_rows, y_rows, nullptr, nullptr,
                act, nullptr, 0, 0, 0, 0, row_scale, row_scale_rows, limit, false, 0, 0, 0};
  return gemm_any_dispatch(a, w_dtype, n_groups, rows_per_group_max, exact ? 1 : 0, S(stream));
}
