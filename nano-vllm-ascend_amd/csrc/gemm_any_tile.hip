// The projections of the 32-bit-residual model families on the MFMA tile kernels (prompt steps, decode batches of more than 8 rows,
// experts of 16 pairs and more): fp32 activations are
// rounded to bf16 once, into an operand buffer (gathered into the experts' order on the way), and multiplied by the tile
// kernels of gemm_tile.hip with an fp32 epilogue.
//
// What bounds it: the products are MFMA-bound from a few hundred rows on.  The kernel these shapes ran on before
// (gemm_any_mfma_kernel: x converted by every feature tile again, operands through registers into LDS, two barriers per K
// step) reached 200-350 TFLOP/s; the tile kernels fetch both operands with LDS-DMA, which needs them in bf16 - hence the
// pass over x, which reads and writes 6 bytes per element once and is paid back from the second feature tile on.
// Measured, 8192 rows: 2048 x 2048 207 -> 63 us + 15 us of operand pass; 64 experts x 8 per row, 2048 -> 2 x 768 with SwiGLU
// 1192 -> 355 us (1.16 PFLOP/s), back to 2048 1050 -> 280 us.  Bits: one fp32 chain over k per result, k ascending, from
// the same rounded operands as gemm_any_mfma_kernel's - the same bits (silu, a form of its own, to an ulp).
#include "gemm_any_stream.hpp"
#include "gemm_tile_args.hpp"

namespace mi {

// Table of a grouped operand: {row tiles, 0, 0, 0}, then per row tile {group, first row, end of the group's rows, 0}.
// GATHER: the (sorted) rows' activations lie at rows x_rows[.] of x, which has x_total rows.
// HALF: the results are bf16 (y16), one weight's persistent products (two weights': always, in their short epilogue).
template <int ACT, bool DUAL, bool GATHER = false, bool HALF = false>
struct AnyTileArgs : TileArgs {
  static constexpr int kAct = ACT;
  static constexpr bool kDual = DUAL, kGather = GATHER, kHalf = HALF;
  int w_rows;  // weight rows from one group's to the next (N, or 2 N where w and w2 are the halves of one matrix)
  const int32_t* x_rows;
  int x_total;
  const uint16_t* w2;
  int groups;
  const int32_t* table;  // nullptr: one group of M rows
  float* y32;
  uint16_t* y16;         // != nullptr: the results as bf16 instead
  const int32_t* y_rows;
  const float* bias1;
  const float* bias2;
  float alpha, limit;
  const float* row_scale;
  const int32_t* row_scale_rows;
};

// SiluAndMul with the roundings of a bf16 product in front of it (moe.hip): two weights only
constexpr int kActMoeGlu = 100;

// the operand's table is read through the scalar cache: it was written by an earlier launch and is the same for a whole wave
typedef const __attribute__((address_space(4))) int32_t* ConstInts;
template <class A>
__device__ __forceinline__ int any_tiles(const A& a) {
  return a.tiles_f * (a.table ? ((ConstInts)(uintptr_t)a.table)[0] : a.tiles_t);
}
// "Block" b's tile: the b & 7-th XCD takes the b & 7-th contiguous run of the tiles (workgroups go to the XCDs in turn: a speed
// assumption only; one to one for any count).  The 32 workgroups an XCD runs together then share row tiles and an expert's weights in
// its L2; with tile b each XCD read nearly every operand row for itself (64 experts of 2 x 768 x 2048 over 65536 rows 526 -> 473 us,
// 32 of 2 x 512 x 1024 over some 32000 124 -> 117).
template <class A>
__device__ __forceinline__ AnyTile any_tile(const A& a, int block, int ntiles, int tile_rows, int tile_features) {
  const int qn = ntiles >> 3, rn = ntiles & 7, xcd = block & 7;
  const int b = xcd * qn + min(xcd, rn) + (block >> 3);
  const int mt = b / a.tiles_f, nt = b - mt * a.tiles_f;
  if (!a.table) return AnyTile{0, mt * tile_rows, a.M, nt * tile_features};
  ConstInts e = (ConstInts)(uintptr_t)a.table + 4 + 4 * mt;
  return AnyTile{e[0], e[1], e[2], nt * tile_features};
}
template <class A>
__device__ __forceinline__ AnyRow any_row(const A& a, int m, int m_end) {
  AnyRow r{-1, 1.f};
  if (m >= m_end) return r;
  r.y = a.y_rows ? a.y_rows[m] : m;
  if (a.row_scale) r.scale = a.row_scale[a.row_scale_rows ? a.row_scale_rows[m] : m];
  return r;
}
// four consecutive features of one row: the epilogue of gemm_any.hip's finish(), operation for operation but for silu's form (b1, b2:
// their biases, where the operand has any)
template <class A>
__device__ __forceinline__ f32x4 any_act(const A& a, f32x4 v, f32x4 v2) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float z = v[e];
    float o = z;
    if constexpr (A::kAct == kActMoeGlu) {
      o = rbf(silu_f32(rbf(z))) * rbf(v2[e]);
    } else if constexpr (A::kAct == MI_ACT_CLAMPED_GLU) {
      const float g = fminf(z, a.limit), u = fminf(fmaxf(v2[e], -a.limit), a.limit);
      o = g / (1.f + expf(-1.702f * g)) * (u + 1.f);
    } else {
      if constexpr (A::kAct == MI_ACT_SILU) o = silu_f32(z);
      if constexpr (A::kAct == MI_ACT_GELU_TANH) o = 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
      if constexpr (A::kAct == MI_ACT_GELU_ERF) o = 0.5f * z * (1.f + erff(z * 0.7071067811865476f));
      if constexpr (A::kAct == MI_ACT_SOFTCAP) o = tanhf(z / a.alpha);   // (times alpha behind: alpha tanh(z / alpha))
      if constexpr (A::kAct == MI_ACT_RELU2) o = fmaxf(z, 0.f) * fmaxf(z, 0.f);
      if (A::kDual) o *= v2[e];
    }
    v[e] = o;
  }
  return v;
}
template <class A>
__device__ __forceinline__ f32x4 any_value(const A& a, float scale, f32x4 v, f32x4 v2, f32x4 b1, f32x4 b2) {
  if (a.row_scale) {
    v *= scale;
    if (A::kDual) v2 *= scale;
  }
  if (a.bias1) v += b1;
  if (A::kDual && a.bias2) v2 += b2;
  v = any_act(a, v, v2);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] *= a.alpha;
  return v;
}
// (a bias is added in the branch that loads it: joined behind it, every store of the lane before is waited for, 2 us of a 64-row tile each)
template <class A>
__device__ __forceinline__ void any_store(const A& a, const AnyRow& row, int n, f32x4 v, f32x4 v2) {
  if (row.y < 0 || n >= a.N) return;
  if (a.row_scale) {
    v *= row.scale;
    if (A::kDual) v2 *= row.scale;
  }
  if (a.bias1) v += *reinterpret_cast<const f32x4*>(a.bias1 + n);
  if (A::kDual && a.bias2) v2 += *reinterpret_cast<const f32x4*>(a.bias2 + n);
  v = any_act(a, v, v2);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] *= a.alpha;
  if (a.y16) *reinterpret_cast<u32x2*>(a.y16 + row.y * a.ldy + n) = u32x2{pack_bf(v[0], v[1]), pack_bf(v[2], v[3])};
  else *reinterpret_cast<f32x4*>(a.y32 + row.y * a.ldy + n) = v;
}

#include "gemm_w16_kernel.hpp"
#include "gemm_mid_kernel.hpp"

// x rows -> bf16 rows (eight elements a thread), gathered by x_rows; rows from the groups' end on are left as they are.  sorted == 0: the
// `rows` rows are those the groups lie in; else the groups lie in `sorted` rows, which the product gathers, and every row is converted.
// The grid's last workgroup writes the tile table: `table_tiles` entries at most, of rows before `rows` (`sorted`) - whatever the groups'
// ends say, nothing is written or, by the product that follows the table, read beyond the buffers.
__global__ __launch_bounds__(256) void any_operand_kernel(const float* __restrict__ x, int64_t ldx,
                                                          const int32_t* __restrict__ x_rows,
                                                          const int32_t* __restrict__ group_offsets, int n_groups,
                                                          int tile_rows, int rows, int sorted, int K, uint16_t* __restrict__ xb,
                                                          int32_t* __restrict__ table, int table_tiles) {
  __shared__ int tiles[1024];
  const int tid = threadIdx.x;
  if (table && blockIdx.x == gridDim.x - 1) {
    auto end_of = [&](int g) { return min(max(group_offsets[g], 0), sorted ? sorted : rows); };
    for (int g = tid; g < n_groups; g += 256) tiles[g] = (max(end_of(g + 1) - end_of(g), 0) + tile_rows - 1) / tile_rows;
    __syncthreads();
    for (int g = tid; g < n_groups; g += 256) {
      int at = 0;
      for (int j = 0; j < g; ++j) at += tiles[j];
      const int lo = end_of(g), hi = end_of(g + 1);
      for (int i = 0; i < tiles[g] && at + i < table_tiles; ++i)
        *reinterpret_cast<int4*>(table + 4 + 4 * (at + i)) = int4{g, lo + i * tile_rows, hi, 0};
      if (g == n_groups - 1) *reinterpret_cast<int4*>(table) = int4{min(at + tiles[g], table_tiles), 0, 0, 0};
    }
    return;
  }
  const int per_row = K >> 3;
  const int64_t i = (int64_t)blockIdx.x * 256 + tid;
  const int row = (int)(i / per_row), c = (int)(i - (int64_t)row * per_row) * 8;
  if (row >= rows || (group_offsets && !sorted && row >= group_offsets[n_groups])) return;
  const float* src = x + (int64_t)(x_rows ? x_rows[row] : row) * ldx + c;
  float4 a, b;
  if ((ldx & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0) {
    a = *reinterpret_cast<const float4*>(src), b = *reinterpret_cast<const float4*>(src + 4);
  } else {
    a = float4{src[0], src[1], src[2], src[3]}, b = float4{src[4], src[5], src[6], src[7]};
  }
  *reinterpret_cast<u32x4*>(xb + (int64_t)row * K + c) =
      u32x4{pack_bf(a.x, a.y), pack_bf(a.z, a.w), pack_bf(b.x, b.y), pack_bf(b.z, b.w)};
}

static bool tile_rows_ok(int t) { return t == 64 || t == 128 || t == 256; }

// the row tiles of `rows` rows in at most n_groups groups (0: one, its tiles known)
static int64_t row_tiles(int rows, int n_groups, int t) { return n_groups ? rows / t + n_groups : (rows + t - 1) / t; }

// (Reached by operands that the streaming kernel does not take - x off 16 bytes -, and by mi_expert_ff_bytes, which is 0 here: these products are
// two calls.)
// Few pairs over small experts: the operand pass and the rings' first round trips are longer than the general kernels' whole walk (us with
// weights not in the L2s and the tile kernels' K loop longer than now, both products, general / tile kernels: 8 experts of 256 x 1024, 64 pairs 15.8 / 18.2; 16 of 256 x 512, 96 pairs
// 12.0 / 14.8; 32 of 256 x 512, 32 pairs 13.3 / 14.7, 48 pairs 16.6 / 14.6; 128 of 256 x 256, 24 pairs 12.4 / 13.3; 8 of 512 x 1024,
// 32 pairs 17.0 / 19.1, 64 pairs 18.8 / 19.1; 128 of 192 x 512, 24 pairs 13.7 / 16.9).  Their time grows with the experts that have a pair
// (some G P / (G + P)) and their rows of weights; beyond eight pairs an expert they take other kernels.
static bool few_pairs(int64_t pairs, int N, int K, int64_t G) {
  if (pairs > 192 || pairs > 8 * G || (pairs >= 128 && N >= 256 && K >= 256) || (int64_t)N * K > (512 << 10)) return false;
  const bool narrow = pairs < 128 && (N < 256 || K < 256);   // (K < 256: on the general kernels either way, an operand pass for one product)
  return G * pairs * (N + K) <= (narrow ? 22000 : (int64_t)N * K <= (256 << 10) ? 12800 : 10240) * (G + pairs);
}

// us of a grouped product on tiles of t rows (64, 128, 256): a CU's share of the tiles, each its K steps and what lies around them, for one tile
// alone on a CU and for several (up to 64 outputs a tile of 64 rows and, of two weights, of 128; else as many as rows, of two weights half).  Fitted to 300
// drawn products from cold weights - 4 to 128 groups of 90 to 2200 rows, shares uneven by a third, 64 to 2112 outputs, K 64 to 4224 - which the choice by it
// misses the best tile's time of by 1.2 % in the mean from K 512 on, 3.7 over all with the line below; by lines in rows per group and tiles, before, 5.2: 64 groups of 276
// rows, two weights of 320 x 192 35 us for 22, 16 of 1974, 256 x 384 and back 67 for 52, 32 of 145, 1664 x 3456 and back 442 for 367.  1.1: over another 1588
// products of 24 to 112 rows the larger tile was the better one where the two are near (1.6 % missed in the mean with it, 1.8 without, 2.5 by the lines).
// The small tiles' K loop has become shorter since, all sizes alike: over 277 other products the choice misses the best tile's time by 1.1 % in the mean from
// K 512 on and by 6 over all, with the loop of the fit by 5.7.
static double grouped_us(int t, int rows, int N, int K, int G, bool dual) {
  const int f = t == 64 || !dual ? t : t / 2;
  const int64_t row_tiles = rows / t + G / 2, tiles = (row_tiles < G ? G : row_tiles) * ((N + f - 1) / f), c = (tiles + 255) / 256;
  const double kt = K / BK;
  if (t == 64) return 1.1 * (dual ? (c == 1 ? 0.63 * kt + 2.5 : c * (0.49 * kt + 1.25)) : (c == 1 ? 0.38 * kt + 2.6 : c * (0.28 * kt + 1.3)));
  if (t == 128) return dual ? (c == 1 ? 0.83 * kt + 4.7 : c * (0.75 * kt + 2.35)) : (c == 1 ? 0.77 * kt + 6.6 : c * (0.77 * kt + 3.3));
  return c * (dual ? 1.67 * kt + 10.2 : 1.6 * kt + 11.3);
}
// K below 512, -1, 0, 1 (not, by the cost, yes): 64-row tiles where a larger one would be mostly padding, and only there.  A line that leaves time: 8 groups of 122
// rows, 384 x 256 11.6 us for 7.6, 8 of 397, 448 x 256 11.8 for 9.2.
static int short_k_64(int rows, int K, int G, bool dual) { return K >= 512 ? 0 : rows < (dual ? 88 : 72) * (int64_t)G ? 1 : -1; }
// the cheapest tile by us(t); 256-row ones not for groups of less than half a tile, whose cold weights they wait for (128 of 256 x 1024, 96 rows: 100 us, 68 and 77
// with the smaller ones)
template <class F>
static int cheapest_tile(int rows, int n_groups, int take_64, F us) {
  if (take_64 > 0) return 64;
  int best = take_64 < 0 || us(128) < us(64) ? 128 : 64;
  if (rows >= 128 * (int64_t)n_groups && us(256) < us(best)) best = 256;
  return best;
}

// 0: not taken; else the rows of a tile (256: the persistent kernel, 128 and 64: the small-tile kernel).  pays: only where it is not slower
// than the general kernels
static int tile_rows_for(int rows, int N, int K, int n_groups, bool dual, int act, bool pays = true) {
  if (rows < 1 || N < 1 || K < BK || K % BK || N % 4 || n_groups < 0 || n_groups > 1024) return 0;
  const bool known = dual ? act == MI_ACT_SILU || act == MI_ACT_GELU_TANH || act == MI_ACT_CLAMPED_GLU
                          : act == MI_ACT_NONE || act == MI_ACT_GELU_ERF || act == MI_ACT_RELU2 || act == MI_ACT_SOFTCAP;
  if (!known) return 0;
  // 32-bit byte offsets from the operand bases, and 0xF0000000 beyond both (the persistent kernel's "fetch nothing")
  const int64_t limit = (int64_t)1 << 31;
  if (((int64_t)(n_groups ? n_groups : 1) * N + 256) * K * 2 >= limit || ((int64_t)rows + 256) * K * 2 >= limit) return 0;
  if (N < 64) return 0;
  // Where the lines lie (us, these kernels incl. the 2 us of the operand pass against gemm_any.hip's other than the streaming one; up to 8 rows those
  // do not round x, and they stay).  No groups, N 2048, rows off 16 bytes: K 2048 at 9 rows 11.9 / 17.2, at 32 12.7 / 33.6, at 128 14.3 / 78; K 512
  // at 16 rows not taken / 7.8, at 24 6.7 / 10.3, at 64 7.0 / 19.7; K 256 at 32 rows not taken / 7.6, at 64 6.3 / 12.5; K 64 from 65 rows on 5.5 / 6.6
  // (on rows at 16 bytes, with a longer K loop here, the kernels met at those lines: K 512 at 16 rows 7.1 / 5.9, at 24 7.2 / 7.2; K 256 at 32 rows 6.3 / 5.4).
  // Experts' pair of products, with that loop, 32 of 512 x 1024 (64 of 768 x 2048): 16 pairs 19 / 20 (32 / 50), 128 pairs 28 / 37, (64 pairs 82 / 106).
  if (n_groups ? rows < 16 || (rows < 128 && K < 256) || (pays && few_pairs(rows, N, K, n_groups))
               : !(rows > 64 || (rows > 32 && K >= 128) || (rows > 16 && K >= 512) ||
                   (rows > 8 && !dual && (K >= 2048 || N >= 8192))))
    return 0;
  if (n_groups && act == MI_ACT_SOFTCAP) return 0;   // (no group has one)
  if (n_groups)
    return cheapest_tile(rows, n_groups, short_k_64(rows, K, n_groups, dual), [=](int t) { return grouped_us(t, rows, N, K, n_groups, dual); });
  // 64-row tiles while they are few; the persistent kernel's 256-row ones where 128-row ones are more than the chip holds (two workgroups per CU).
  const auto tiles = [=](int t, int f) { return (int64_t)((rows + t - 1) / t) * ((N + f - 1) / f); };
  // us, cold weights, 64- / 128- / 256-row tiles: 2000 x 1024 x 1024 (512 / 128 / 32 tiles) 11 / 14 / 26, 2000 x 2048 x 1024 (1024 / 256 / 64) 24 / 17 / 30,
  // 4000 x 2048 x 1024 (2016 / 512 / 128) 33 / 25 / 30, 3000 x 3072 x 1024 (2256 / 576 / 144) 41 / 35 / 30; 1000 x 2048 x 2048 (512 / 128 / 32) 22 / 24 / 46,
  // 1300 (672 / 176 / 48) 30 / 22 / 44, 4000 (2016 / 512 / 128) 55 / 40 / 48, 1300 x 6144 x 2048 (2016 / 528 / 144) 77 / 59 / 47; over 200 drawn products the
  // choice misses the best tile's time by 0.4 % in the mean
  if (tiles(64, 64) <= 512) return 64;
  return act != MI_ACT_SOFTCAP && tiles(128, dual ? 64 : 128) > 512 ? 256 : 128;
}

// ... of experts' two products, which share one table of tiles
static int pair_tile_rows(int pairs, int G, int ff, int width, bool dual, int act, bool pays) {
  if (!tile_rows_for(pairs, ff, width, G, dual, act, pays) || !tile_rows_for(pairs, width, ff, G, false, MI_ACT_NONE, pays)) return 0;
  const int a = short_k_64(pairs, width, G, dual), b = short_k_64(pairs, ff, G, false);
  return cheapest_tile(pairs, G, a > 0 || b > 0 ? 1 : a < b ? a : b,
                       [=](int t) { return grouped_us(t, pairs, ff, width, G, dual) + grouped_us(t, pairs, width, ff, G, false); });
}

template <int ACT, bool DUAL, bool GATHER, bool HALF>
static int launch_any_tile(const AnyTileArgs<ACT, DUAL, GATHER, HALF>& args, int tile_rows, int64_t row_tiles_max, hipStream_t st) {
  using A = AnyTileArgs<ACT, DUAL, GATHER, HALF>;
  A a = args;
  if (tile_rows == 256) {
    a.tiles_f = (a.N + (DUAL ? 127 : 255)) / (DUAL ? 128 : 256);
    a.tiles_t = (a.M + 255) / 256;
    const int64_t tiles = row_tiles_max * a.tiles_f;
    const dim3 grid((unsigned)(tiles < kPersistentGrid ? tiles : kPersistentGrid));
    // the epilogue's short form takes what the models' projections and experts ask for
    [[maybe_unused]] const bool lean = !a.row_scale && a.alpha == 1.f && a.N % (DUAL ? 128 : 256) == 0 &&
                                       (DUAL || HALF ? a.y16 && !a.bias1 && !a.bias2 && a.ldy % 8 == 0 : !a.y16);
    if constexpr (ACT != MI_ACT_SOFTCAP) {  // (a head's product: never that many rows; it would not fit the persistent kernel's registers)
      if constexpr (DUAL ? ACT == MI_ACT_SILU || ACT == kActMoeGlu : ACT == MI_ACT_NONE)
        if (lean) {
          hipLaunchKernelGGL((gemm_w16_kernel<TEPI_ANY, false, 32768, A>), grid, dim3(256), 0, st, a);
          return check_launch();
        }
      hipLaunchKernelGGL((gemm_w16_kernel<TEPI_ANY, false, 0, A>), grid, dim3(256), 0, st, a);
    }
  } else if (tile_rows == 64) {
    // two weights: 128 feature rows (64 outputs); one: 64, or 128 where that leaves at least four tiles per CU (the experts' second
    // product, us, 64 / 128 features: 32 experts of 1024 x 512 8.9 / 9.6, 64 of 2048 x 768 41 / 39.5; with a longer K loop than now)
    const int64_t narrow = row_tiles_max * ((a.N + 63) / 64);
    const bool wide = DUAL || narrow > 4 * kPersistentGrid;
    a.tiles_f = !DUAL && wide ? (a.N + 127) / 128 : (a.N + 63) / 64;
    a.tiles_t = (a.M + 63) / 64;
    const int64_t tiles = row_tiles_max * a.tiles_f;
    if (tiles > 0x7fffffff) return MI_EUNSUPPORTED;
    if (wide) {
      hipLaunchKernelGGL((gemm_mid_kernel<TEPI_ANY, false, 3, A, MidShape<2, 2, 2, 1>>), dim3((unsigned)tiles), dim3(256), 0, st, a);
    } else {
      if constexpr (!DUAL)
        hipLaunchKernelGGL((gemm_mid_kernel<TEPI_ANY, false, 5, A, MidShape<2, 2, 1, 1>>), dim3((unsigned)tiles), dim3(256), 0, st, a);
    }
  } else {
    a.tiles_f = (a.N + (DUAL ? 63 : 127)) / (DUAL ? 64 : 128);
    a.tiles_t = (a.M + 127) / 128;
    const int64_t tiles = row_tiles_max * a.tiles_f;
    if (tiles > 0x7fffffff) return MI_EUNSUPPORTED;
    if (tiles > kPersistentGrid)
      hipLaunchKernelGGL((gemm_mid_kernel<TEPI_ANY, false, 2, A>), dim3((unsigned)tiles), dim3(256), 0, st, a);
    else
      hipLaunchKernelGGL((gemm_mid_kernel<TEPI_ANY, false, 4, A>), dim3((unsigned)tiles), dim3(256), 0, st, a);
  }
  return check_launch();
}

}  // namespace mi

using namespace mi;

extern "C" int mi_gemm_any_tile_rows(int rows, int N, int K, int n_groups, int dual, int act) {
  return tile_rows_for(rows, N, K, n_groups, dual != 0, act);
}

extern "C" int64_t mi_gemm_any_table_ints(int rows, int n_groups, int tile_rows) {
  if (rows < 0 || n_groups < 1 || !tile_rows_ok(tile_rows)) return 0;
  return 4 + 4 * row_tiles(rows, n_groups, tile_rows);
}

static int any_operand(const float* x, int64_t ldx, const int32_t* x_rows, const int32_t* group_offsets, int n_groups, int tile_rows,
                       int rows, int sorted, int K, mi_bf16* xb, int32_t* table, mi_stream stream) {
  if (!x || !xb || rows < 0 || K < 8 || K % 8 || ldx < K || !aligned16(xb)) return MI_EINVAL;
  if (n_groups < 0 || n_groups > 1024 || (n_groups > 0) != (group_offsets != nullptr)) return MI_EINVAL;
  if (table && (!n_groups || !aligned16(table) || !tile_rows_ok(tile_rows))) return MI_EINVAL;
  if (rows == 0) return MI_OK;
  const int64_t blocks = ((int64_t)rows * (K / 8) + 255) / 256 + (table ? 1 : 0);
  if (blocks > 0x7fffffff) return MI_EUNSUPPORTED;
  hipLaunchKernelGGL(any_operand_kernel, dim3((unsigned)blocks), dim3(256), 0, S(stream), x, ldx, x_rows, group_offsets, n_groups,
                     tile_rows, rows, sorted, K, xb, table, table ? (int)row_tiles(sorted ? sorted : rows, n_groups, tile_rows) : 0);
  return check_launch();
}

// the table alone
static int tile_table(const int32_t* group_offsets, int n_groups, int tile_rows, int sorted, int32_t* table, mi_stream stream) {
  hipLaunchKernelGGL(any_operand_kernel, dim3(1), dim3(256), 0, S(stream), nullptr, 0, nullptr, group_offsets, n_groups, tile_rows, 0, sorted, 8, nullptr,
                     table, (int)row_tiles(sorted, n_groups, tile_rows));
  return check_launch();
}

extern "C" int mi_gemm_any_operand(const float* x, int64_t ldx, const int32_t* x_rows, const int32_t* group_offsets,
                                   int n_groups, int tile_rows, int rows, int K, mi_bf16* xb, int32_t* table,
                                   mi_stream stream) {
  return any_operand(x, ldx, x_rows, group_offsets, n_groups, tile_rows, rows, 0, K, xb, table, stream);
}

// x_rows (two weights, groups): row m of the groups' rows is row x_rows[m] of xb's x_total
static int any_tile_product(const mi_bf16* xb, const int32_t* x_rows, int x_total, const int32_t* table, int tile_rows, const mi_bf16* w,
                            const mi_bf16* w2, const float* bias, const float* bias2, int act, float limit, const float* row_scale,
                            const int32_t* row_scale_rows, int n_groups, void* y, int y_is_bf16, int64_t ldy, const int32_t* y_rows,
                            int rows, int N, int K, float alpha, mi_stream stream) {
  if (!xb || !w || !y || rows < 0 || (n_groups > 0) != (table != nullptr) || (row_scale_rows && !row_scale)) return MI_EINVAL;
  if (act == MI_ACT_CLAMPED_GLU && !(limit > 0.f)) return MI_EINVAL;
  if (act == MI_ACT_SOFTCAP && tile_rows == 256) return MI_EUNSUPPORTED;   // (launch_any_tile)
  if (rows == 0) return MI_OK;
  if (!tile_rows_ok(tile_rows)) return MI_EINVAL;
  if (tile_rows_for(rows, N, K, n_groups, w2 != nullptr, act, false) == 0) return MI_EUNSUPPORTED;
  if (ldy < N || ldy % 4 || !aligned16(xb) || !aligned16(w) || (w2 && !aligned16(w2)) || !aligned16(y) || (bias && !aligned16(bias)) ||
      (bias2 && (!w2 || !aligned16(bias2))))
    return MI_EINVAL;
  const int64_t tiles = row_tiles(rows, n_groups, tile_rows);
  auto go = [&](auto args) {
    args.x = xb, args.w = w, args.w2 = w2, args.bias = nullptr, args.y = nullptr, args.part = nullptr;
    args.ldx = K, args.ldy = ldy, args.M = rows, args.N = N, args.K = K;
    args.groups = n_groups ? n_groups : 1, args.table = table, args.w_rows = N;
    args.y32 = y_is_bf16 ? nullptr : static_cast<float*>(y), args.y16 = y_is_bf16 ? static_cast<uint16_t*>(y) : nullptr;
    args.y_rows = y_rows, args.bias1 = bias, args.bias2 = bias2, args.alpha = alpha, args.limit = limit;
    args.row_scale = row_scale, args.row_scale_rows = row_scale_rows;
    args.x_rows = x_rows, args.x_total = x_total;
    return launch_any_tile(args, tile_rows, tiles, S(stream));
  };
  if (x_rows) {
    if (!w2 || !table || x_total < 1 || x_total > rows) return MI_EINVAL;   // (xb's rows: at most as many as the limits were taken for)
    if (act == MI_ACT_SILU) return go(AnyTileArgs<MI_ACT_SILU, true, true>{});
    if (act == MI_ACT_GELU_TANH) return go(AnyTileArgs<MI_ACT_GELU_TANH, true, true>{});
    return go(AnyTileArgs<MI_ACT_CLAMPED_GLU, true, true>{});
  }
  if (w2) {
    if (act == MI_ACT_SILU) return go(AnyTileArgs<MI_ACT_SILU, true>{});
    if (act == MI_ACT_GELU_TANH) return go(AnyTileArgs<MI_ACT_GELU_TANH, true>{});
    return go(AnyTileArgs<MI_ACT_CLAMPED_GLU, true>{});
  }
  if (act == MI_ACT_NONE) return go(AnyTileArgs<MI_ACT_NONE, false>{});
  if (act == MI_ACT_SOFTCAP) return alpha > 0.f ? go(AnyTileArgs<MI_ACT_SOFTCAP, false>{}) : MI_EINVAL;
  if (act == MI_ACT_GELU_ERF) return go(AnyTileArgs<MI_ACT_GELU_ERF, false>{});
  return go(AnyTileArgs<MI_ACT_RELU2, false>{});
}

extern "C" int mi_gemm_any_tile(const mi_bf16* xb, const int32_t* table, int tile_rows, const mi_bf16* w, const mi_bf16* w2,
                                const float* bias, const float* bias2, int act, float limit, const float* row_scale,
                                const int32_t* row_scale_rows, int n_groups, void* y, int y_is_bf16, int64_t ldy,
                                const int32_t* y_rows, int rows, int N, int K, float alpha, mi_stream stream) {
  return any_tile_product(xb, nullptr, 0, table, tile_rows, w, w2, bias, bias2, act, limit, row_scale, row_scale_rows, n_groups, y,
                          y_is_bf16, ldy, y_rows, rows, N, K, alpha, stream);
}

// ---- the two launches (operand pass, product) and the choice between these kernels and gemm_any.hip's behind one call: steps that are
// launched eagerly are bound by the host, which pays for every call (a prompt of 40 rows through 4 layers of Felolorn at width 1024: some 1330 us with four calls per product, 1110 with two) ----

extern "C" int64_t mi_gemm_any_fit_elems(int M, int N, int K, int dual, int act) {
  return tile_rows_for(M, N, K, 0, dual != 0, act) ? (int64_t)M * K : 0;
}

// ready: xb holds x rounded to bf16 already (it is written here where not)
static int any_fit(const float* x, int64_t ldx, const void* w, const void* w2, int w_dtype, const float* bias, const float* bias2, int act, float* y,
                   int64_t ldy, int M, int N, int K, float alpha, const mi_bf16* xb, int64_t xb_elems, bool ready, mi_stream stream) {
  const bool fits = xb && x && w && y && w_dtype == MI_DTYPE_BF16 && M > 0 && ldx >= K && ldy >= N && ldy % 4 == 0 && aligned16(w) &&
                    (!w2 || aligned16(w2)) && aligned16(y) && (!bias || aligned16(bias)) && (!bias2 || (w2 && aligned16(bias2))) &&
                    aligned16(xb) && xb_elems >= (int64_t)M * K && !(act == MI_ACT_SOFTCAP && !(alpha > 0.f));
  const bool streams = any_stream_takes(M, N, K, 0, w2 != nullptr) && aligned16(x) && ldx % 4 == 0;
  const int t = fits && !streams ? tile_rows_for(M, N, K, 0, w2 != nullptr, act) : 0;
  if (!t) return mi_gemm_any_act(x, ldx, w, w2, w_dtype, bias, bias2, act, y, ldy, M, N, K, alpha, 0, stream);
  const int rc = ready ? MI_OK : mi_gemm_any_operand(x, ldx, nullptr, nullptr, 0, t, M, K, const_cast<mi_bf16*>(xb), nullptr, stream);
  return rc != MI_OK ? rc
                     : mi_gemm_any_tile(xb, nullptr, t, static_cast<const mi_bf16*>(w), static_cast<const mi_bf16*>(w2), bias, bias2, act,
                                        0.f, nullptr, nullptr, 0, y, 0, ldy, nullptr, M, N, K, alpha, stream);
}
extern "C" int mi_gemm_any_fit(const float* x, int64_t ldx, const void* w, const void* w2, int w_dtype, const float* bias,
                               const float* bias2, int act, float* y, int64_t ldy, int M, int N, int K, float alpha, mi_bf16* xb,
                               int64_t xb_elems, mi_stream stream) {
  return any_fit(x, ldx, w, w2, w_dtype, bias, bias2, act, y, ldy, M, N, K, alpha, xb, xb_elems, false, stream);
}
extern "C" int mi_gemm_any_fit_rounded(const float* x, int64_t ldx, const void* w, const void* w2, int w_dtype, const float* bias, const float* bias2,
                                       int act, float* y, int64_t ldy, int M, int N, int K, float alpha, const mi_bf16* xb, int64_t xb_elems,
                                       mi_stream stream) {
  return any_fit(x, ldx, w, w2, w_dtype, bias, bias2, act, y, ldy, M, N, K, alpha, xb, xb_elems, true, stream);
}

// ---- the experts of moe.hip (bf16 activations and weights as they are stored, row-major) on the tile kernels: steps that bring prompts ----
// moe.hip's kernels keep 16 features' weights in registers and walk an expert's pairs 16 at a time, a round trip and two barriers each:
// made for the few pairs of a decode step.  us of a block (route to combine) with them / here on 64- / 128- / 256-row tiles (the first two with a longer
// K loop than now):
//   64 experts of 768 x 2048     8 pairs each 127 / 146 / 162 / 185   16 153 / 148 / 164 / 188   64 306 / 173 / 183 / 197   128 530 / 229 / 236 / 212
//                                512 1843 / 620 / 524 / 385
//   32 of 512 x 1024             8 34 / 34 / 38 / 56   16 40 / 35 / 38 / 56   64 72 / 44 / 44 / 57   192 155 / 62 / 56 / 63   512 360 / 115 / 110 / 106
//   8 of 512 x 1024              32 22 / 27 / 36 / 51   64 28 / 28 / 36 / 52   256 67 / 38 / 40 / 55   512 114 / 53 / 51 / 58
//   8 of 1536 x 4096             16 71 / 71 / 82 / 126   64 145 / 110 / 107 / 131;   128 of 768 x 2048   8 242 / 237 / 250 / 281   128 1017 / 417 / 401 / 335
// A step of 8 x 1024 tokens, four layers of 64 experts: 15.7 -> 3.9 ms.
static int moe_tile_rows(int pairs, int G, int ff, int width) {
  if (pairs < 1 || G < 1 || width % BK || ff % BK || width % 8 || ff % 8) return 0;
  if (2 * (int64_t)ff > INT32_MAX || ((int64_t)G * 2 * ff + 256) * width * 2 >= (int64_t)1 << 31) return 0;   // (32-bit offsets into gate_up)
  if (pairs < 16 * (int64_t)G || (int64_t)pairs * (ff + width) < 800000) return 0;
  return pair_tile_rows(pairs, G, ff, width, true, MI_ACT_SILU, false);
}
extern "C" int64_t mi_moe_tiles_bytes(int pairs, int n_experts, int inter, int hidden) {
  const int t = moe_tile_rows(pairs, n_experts, inter, hidden);
  return t ? 4 * mi_gemm_any_table_ints(pairs, n_experts, t) : 0;
}
extern "C" int mi_moe_tiles(const mi_bf16* x, int n_tokens, const mi_bf16* gate_up, const mi_bf16* down, const int32_t* expert_offsets,
                            const int32_t* pair_token, const int32_t* pair_index, mi_bf16* act, mi_bf16* y, int pairs, int n_experts,
                            int hidden, int inter, void* scratch, int64_t scratch_bytes, mi_stream stream) {
  if (!x || !gate_up || !down || !expert_offsets || !pair_token || !pair_index || !act || !y || !scratch) return MI_EINVAL;
  if (!aligned16(x) || !aligned16(gate_up) || !aligned16(down) || !aligned16(act) || !aligned16(y) || !aligned16(scratch)) return MI_EINVAL;
  if (n_tokens < 1 || n_tokens > pairs) return MI_EINVAL;
  const int t = moe_tile_rows(pairs, n_experts, inter, hidden);
  if (!t) return MI_EUNSUPPORTED;
  if (scratch_bytes < mi_moe_tiles_bytes(pairs, n_experts, inter, hidden)) return MI_EWORKSPACE;
  int32_t* table = static_cast<int32_t*>(scratch);
  const int64_t tiles = row_tiles(pairs, n_experts, t);
  int rc = tile_table(expert_offsets, n_experts, t, pairs, table, stream);
  if (rc != MI_OK) return rc;
  AnyTileArgs<kActMoeGlu, true, true> g{};
  g.x = x, g.w = gate_up, g.w2 = gate_up + (int64_t)inter * hidden, g.ldx = hidden, g.ldy = inter, g.M = pairs, g.N = inter, g.K = hidden;
  g.w_rows = 2 * inter, g.x_rows = pair_token, g.x_total = n_tokens, g.groups = n_experts, g.table = table, g.y16 = act, g.alpha = 1.f;
  rc = launch_any_tile(g, t, tiles, S(stream));
  if (rc != MI_OK) return rc;
  AnyTileArgs<MI_ACT_NONE, false, false, true> d{};
  d.x = act, d.w = down, d.ldx = inter, d.ldy = hidden, d.M = pairs, d.N = hidden, d.K = inter;
  d.w_rows = hidden, d.groups = n_experts, d.table = table, d.y16 = y, d.y_rows = pair_index, d.alpha = 1.f;
  return launch_any_tile(d, t, tiles, S(stream));
}

// scratch of mi_expert_ff: the gathered operand, the inner activations, the tile table (each rounded up to 16 bytes) - or, streamed, the
// inner activations in fp32
static int expert_tile_rows(int pairs, int G, int ff, int width, bool dual, int act) {
  return pair_tile_rows(pairs, G, ff, width, dual, act, true);
}
static int64_t round16(int64_t bytes) { return (bytes + 15) & ~(int64_t)15; }

extern "C" int64_t mi_expert_ff_bytes(int pairs, int G, int ff, int width, int dual, int act) {
  if (pairs < 1 || G < 1) return 0;
  const int t = expert_tile_rows(pairs, G, ff, width, dual != 0, act);
  if (!t) return 0;
  const int64_t tiles = round16((int64_t)pairs * width * 2) + round16((int64_t)pairs * ff * 2) + 4 * mi_gemm_any_table_ints(pairs, G, t);
  const int64_t inner = round16((int64_t)pairs * ff * 4);
  return tiles > inner ? tiles : inner;
}

// tokens: the rows of x (0: not known).  Where the pairs are at least as many, x is rounded to bf16 a token at a time and the first
// product's feed gathers the pairs' rows; else the operand pass writes them out in the experts' order (65536 pairs of 8192 tokens x 2048,
// us: pass 112 + product 459, now 15 + 441; 48 to 2000 pairs of 2 to 16 experts, both products: 0.97 to 1.01 of the time, 0.99 on average).
// rounded: the tokens' rows in bf16 already, or nullptr.
static int expert_ff(const float* x, int64_t ldx, const mi_bf16* rounded, int tokens, const int32_t* pair_token, const mi_bf16* w,
                     const mi_bf16* w2, const mi_bf16* down, int act, float limit, const float* row_scale,
                     const int32_t* row_scale_rows, const int32_t* offsets, const int32_t* pair_index, int pairs, int G,
                     int ff, int width, void* scratch, int64_t scratch_bytes, float* y, mi_stream stream) {
  if (!x || !w || !down || !offsets || !scratch || !y || pairs < 1 || G < 1 || !aligned16(scratch)) return MI_EINVAL;
  const int64_t need = mi_expert_ff_bytes(pairs, G, ff, width, w2 != nullptr, act);
  if (need == 0) return MI_EUNSUPPORTED;
  if (scratch_bytes < need) return MI_EWORKSPACE;
  if (any_stream_takes(pairs, ff, width, G, false) && any_stream_takes(pairs, width, ff, G, false) && aligned16(x) && ldx % 4 == 0 && aligned16(w) &&
      aligned16(down) && (!w2 || aligned16(w2))) {
    float* inner = static_cast<float*>(scratch);
    const int rc = mi_gemm_any_grouped_glu(x, ldx, pair_token, w, w2, MI_DTYPE_BF16, act, limit, row_scale, row_scale_rows, offsets, G, pairs,
                                           inner, ff, nullptr, ff, width, 0, stream);
    return rc != MI_OK ? rc : mi_gemm_any_grouped(inner, ff, nullptr, down, nullptr, MI_DTYPE_BF16, offsets, G, pairs, y, width, pair_index,
                                                  width, ff, 0, stream);
  }
  const int t = expert_tile_rows(pairs, G, ff, width, w2 != nullptr, act);
  char* p = static_cast<char*>(scratch);
  mi_bf16* xb = reinterpret_cast<mi_bf16*>(p);
  mi_bf16* inner = reinterpret_cast<mi_bf16*>(p += round16((int64_t)pairs * width * 2));
  int32_t* table = reinterpret_cast<int32_t*>(p += round16((int64_t)pairs * ff * 2));
  const bool gather = w2 && pair_token && tokens > 0 && tokens <= pairs;
  const bool ready = gather && rounded && aligned16(rounded);
  int rc = ready  ? tile_table(offsets, G, t, pairs, table, stream)
           : gather ? any_operand(x, ldx, nullptr, offsets, G, t, tokens, pairs, width, xb, table, stream)
                    : mi_gemm_any_operand(x, ldx, pair_token, offsets, G, t, pairs, width, xb, table, stream);
  if (rc == MI_OK)
    rc = any_tile_product(ready ? rounded : xb, gather ? pair_token : nullptr, gather ? tokens : 0, table, t, w, w2, nullptr, nullptr, act, limit, row_scale,
                          row_scale_rows, G, inner, 1, ff, nullptr, pairs, ff, width, 1.f, stream);
  return rc != MI_OK ? rc
                     : mi_gemm_any_tile(inner, table, t, down, nullptr, nullptr, nullptr, MI_ACT_NONE, 0.f, nullptr, nullptr, G, y, 0, width,
                                        pair_index, pairs, width, ff, 1.f, stream);
}

extern "C" int mi_expert_ff_tokens(const float* x, int64_t ldx, int tokens, const int32_t* pair_token, const mi_bf16* w,
                                   const mi_bf16* w2, const mi_bf16* down, int act, float limit, const float* row_scale,
                                   const int32_t* row_scale_rows, const int32_t* offsets, const int32_t* pair_index, int pairs, int G,
                                   int ff, int width, void* scratch, int64_t scratch_bytes, float* y, mi_stream stream) {
  return expert_ff(x, ldx, nullptr, tokens, pair_token, w, w2, down, act, limit, row_scale, row_scale_rows, offsets, pair_index, pairs, G, ff,
                   width, scratch, scratch_bytes, y, stream);
}
extern "C" int mi_expert_ff_rounded(const float* x, int64_t ldx, const mi_bf16* rounded, int tokens, const int32_t* pair_token, const mi_bf16* w,
                                    const mi_bf16* w2, const mi_bf16* down, int act, float limit, const float* row_scale,
                                    const int32_t* row_scale_rows, const int32_t* offsets, const int32_t* pair_index, int pairs, int G,
                                    int ff, int width, void* scratch, int64_t scratch_bytes, float* y, mi_stream stream) {
  return expert_ff(x, ldx, rounded, tokens, pair_token, w, w2, down, act, limit, row_scale, row_scale_rows, offsets, pair_index, pairs, G, ff,
                   width, scratch, scratch_bytes, y, stream);
}
extern "C" int mi_expert_ff(const float* x, int64_t ldx, const int32_t* pair_token, const mi_bf16* w, const mi_bf16* w2,
                            const mi_bf16* down, int act, float limit, const float* row_scale, const int32_t* row_scale_rows,
                            const int32_t* offsets, const int32_t* pair_index, int pairs, int G, int ff, int width, void* scratch,
                            int64_t scratch_bytes, float* y, mi_stream stream) {
  return mi_expert_ff_tokens(x, ldx, 0, pair_token, w, w2, down, act, limit, row_scale, row_scale_rows, offsets, pair_index, pairs, G, ff,
                             width, scratch, scratch_bytes, y, stream);
}
