// What the MFMA tile GEMM kernels (gemm_w16_kernel.hpp, gemm_mid_kernel.hpp, ...) share: arguments and tile order.
#pragma once
#include <type_traits>
#include <utility>

#include "mi_common.hpp"
#include "gemm_tile_index.hpp"

namespace mi {
using namespace gt;

typedef __attribute__((ext_vector_type(16))) float f32x16;

// TEPI_ANY: fp32 results with the epilogue of gemm_any_tile.hip (AnyTileArgs there), plain or grouped rows
enum { TEPI_NONE = 0, TEPI_SILU = 1, TEPI_PARTIAL = 2, TEPI_QKV = 3, TEPI_ANY = 4 };

struct TileArgs {
  static constexpr bool kDual = false, kGather = false, kHalf = false;
  const uint16_t* x;
  const uint16_t* w;
  const uint16_t* bias;
  uint16_t* y;
  int64_t ldx, ldy;
  int M, N, K;
  int tiles_f, tiles_t;
  // gemm_mid_kernel: the XCDs share the tiles as 2^xcd_lf runs of features times 2^(3 - xcd_lf) runs of tokens (mid_tile).  (Here, in what would be padding:
  // at the end it moved AnyTileArgs' own arguments across a 64-byte line, one more to fetch at a launch's start: 0.46 us where other kernels run between, 95 x
  // 576 x 64 3.4 / 3.9.)
  int xcd_lf;
  float* part;  // split-K (gridDim.y > 1): fp32 partial sums [gridDim.y][M][N] instead of y
  // TEPI_QKV (mi_gemm_bf16_qkv_store): the K and V heads of the packed qkv projection go straight to the paged cache
  struct QkvStore {
    const uint16_t* k_w;       // k-norm weight [128] or null
    const int64_t* positions;  // [M]
    const float* cos_sin;      // [max_position][128]
    uint16_t* k_cache;
    uint16_t* v_cache;
    const int32_t* slots;      // [M] flat slots (block * block_size + offset; negative: not stored)
    float eps;
    int n_q_heads, n_kv_heads, block_size;
  } qkv;
};

constexpr int kPersistentGrid = 256;  // one workgroup per CU

#define MI_GT_BARRIER() asm volatile("s_barrier" ::: "memory")

// tile of "block" b.  Plain order (the default): tile b, feature tiles fastest.  The dispatcher places workgroup b
// on XCD b % 8 (a speed assumption only) and a persistent workgroup keeps b % 8 - and, the feature-tile count dividing
// 256 for every shape of the path, its feature tile - over its tiles: its 256 x K weight panel stays in the XCD's L2
// while the activation panels stream through.  The alternative (rect): the 32 workgroups an XCD runs together are
// given a GT x GF rectangle of tiles, GT activation + GF weight panels per K step; measured equal or slower
// (tools/gemm_bench.py), kept as a tuning variant.
__device__ __forceinline__ int tile_of_block(int b, int tiles_t, int tiles_f, bool rect) {
  const int ntiles = tiles_t * tiles_f;
  if (!rect) return b;
  const int gf = tiles_f % 8 == 0 ? 8 : (tiles_f % 4 == 0 ? 4 : (tiles_f % 2 == 0 ? 2 : 1)), gt = 32 / gf;
  const int xcd = b & 7, idx = b >> 3;
  if (ntiles % 256 == 0 && tiles_t % gt == 0) {
    const int r = (idx >> 5) * 8 + xcd, local = idx & 31, rc = tiles_f / gf;
    return ((r / rc) * gt + local / gf) * tiles_f + (r % rc) * gf + local % gf;
  }
  // any other grid: XCD x takes the x-th contiguous run of tiles (bijective for every ntiles)
  const int qn = ntiles >> 3, rn = ntiles & 7;
  return (xcd < rn ? xcd * (qn + 1) : rn * (qn + 1) + (xcd - rn) * qn) + idx;
}


// TEPI_ANY: a tile's group (expert; 0 without groups), its first row, the end of its group's rows, its first feature; an
// output row (-1: none) with the factor on its accumulators
struct AnyTile {
  int group, m0, m_end, n0;
};
struct AnyRow {
  int64_t y;
  float scale;
};
}  // namespace mi
