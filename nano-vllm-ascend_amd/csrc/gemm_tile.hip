// bf16 MFMA tile GEMM for the compute-bound regime (M > 64 rows of activations: every prefill projection,
// large decode batches).
//
//   y[M][N] = x[M][K] @ w[N][K]^T (+ bias)        (reference: F.linear, linear.py:51,73,150)
//   epilogue 1: y[M][N/2] = SiluAndMul(x @ w^T)    (activation.py:10-12 on MergedColumnParallelLinear, linear.py:73)
//
// Both operands are K-contiguous, so both are staged the same way: whole 128-byte lines by LDS-DMA
// (global_load_lds_dwordx4) into XOR-swizzled 16 KiB half-tiles (layout and index arithmetic: gemm_tile_index.hpp).
//
// Schedule (one workgroup = 8 waves, 129 KiB of LDS, one workgroup per CU, PERSISTENT: workgroup b computes the
// 256 x 256 tiles b, b + grid, ...; the DMA stream runs on across tile seams, so only a workgroup's first tile
// pays the fill latency and a tile's stores overlap the next tile's loads):
//   * a K step t is two phases of sixteen v_mfma_f32_32x32x16_bf16 per wave (512 cycles of matrix pipe each), each
//     phase a read segment R and a matrix segment M between workgroup barriers:
//       R_P0(t): reads A half 0, B half 0, B half 1 of step t (16 ds_read_b128);
//                DMA of B half 1, A half 1 of step t + 1 (4 pieces)
//       M_P0(t): (A0 x B0, A0 x B1), sixteen MFMAs back to back
//       R_P1(t): reads A half 1 of step t (8 ds_read_b128); DMA of A half 0, B half 0 of step t + 2 (4 pieces)
//       M_P1(t): (A1 x B1, A1 x B0)
//     A DMA instruction blocks its wave for ~75 cycles: issued between MFMAs that is 75 cycles of idle matrix pipe
//     (measured: 20-26 % of the kernel), issued by the READING wave it hides under the partner's MFMA cluster.
//     Every piece has at least two segments to land.  No wait in the loop is vmcnt(0): a wave waits vmcnt(8) at the
//     end of R_P0 (A1 of this step landed) and vmcnt(6) at the end of R_P1 (A0, B0, B1 of the next step landed),
//     for its OWN pieces, and for its fragment reads (lgkmcnt(0): a slot just read may be re-filled by the partner
//     group one barrier later); the workgroup barrier behind the wait publishes the pieces to the next readers;
//   * the two waves that share a SIMD (wave w and w + 4) run one barrier apart: while one issues its MFMA cluster,
//     the other reads the next phase's fragments - the matrix pipe of a SIMD always has one wave feeding it;
//   * a workgroup's last tile requests nothing past its end; the waits of its last two K steps count accordingly.
//     The first R_P0 of every tile waits vmcnt(0): the previous tile's stores sit on the same counter.
// Tile order: plain (see tile_of_block).
//
// Summation order: one fp32 MFMA chain over K per output element (k ascending), rounded to bf16 once -
// the same rounding points as F.linear; the SwiGLU epilogue keeps the reference's three roundings
// (bf16 gate_up output, bf16 silu, bf16 product).
#include <type_traits>

#include "mi_common.hpp"
#include "gemm_tile_index.hpp"
#include "kv_store.hpp"

namespace mi {
using namespace gt;

}  // namespace mi
#include "gemm_tile_args.hpp"
namespace mi {

// Tuning variants of the eight-wave kernel below (mi_gemm_bf16_ex instantiates the combinations it lists - the staggered
// start V & 1024 and the never-waited DMA V & 256 measured no effect and are not instantiated any more; the timing-only
// ablations lived in an EXPERIMENTS=1 build flavour, since removed - their numbers are in
// profiles/r04_gemm_ablation.txt; the product entry point uses kDefaultV on the four-wave kernels):
//   V & 2    both waves of a SIMD in lockstep (no one-barrier stagger)
//   V & 4    XCD-rectangle tile order instead of the plain one (tile_of_block; measured equal or slower)
//   V & 8    8-byte stores in the epilogue (no v_permlane32_swap widening)
//   V & 16   one tile per workgroup (grid = tiles, not persistent)
//   V & 1024 workgroups start up to 6 us apart (their output bursts interleave)
//   V & 8192 output rows staged through a per-wave 4 KiB LDS buffer and stored as whole 128-byte lines (a CU's store
//            path moves 49 instead of 17 bytes per cycle that way, tools/ubench/store_pattern.hip; with every CU
//            storing at once the burst is HBM-bound either way: 130.8 vs 132.2 us on qkv, 69.5 vs 64.3 on o_proj)
//   V & 512  ABLATION: no output stores
//   V & 32 / 64 / 128   ABLATIONS for timing only (wrong results): no DMA in the K loop / no fragment reads in the K
//            loop / no workgroup barriers in the K loop
constexpr int kDefaultV = 0;
template <int EPI, bool BIAS, int V>
__global__ __launch_bounds__(512, 2) void gemm_tile_kernel(const TileArgs a) {
  // ONE LDS object (a second one makes hipcc drain the DMA queue before every fragment read)
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fh = wave >> 2, tq = wave & 3, hi = lane >> 5, l31 = lane & 31;
  // split-K: blockIdx.y takes the K steps [kbeg, kbeg + KT) of every tile it is given
  const int KT_all = a.K / BK;
  const int KT = EPI == TEPI_PARTIAL ? KT_all / (int)gridDim.y : KT_all;
  const int64_t kbeg_bytes = EPI == TEPI_PARTIAL ? (int64_t)blockIdx.y * KT * (BK * 2) : 0;
  const int ntiles = a.tiles_f * a.tiles_t, stride = (int)gridDim.x;

  // ---- LDS-DMA sources: byte offset (K step 0) of this lane's 16 bytes of piece (half-tile h, instruction i) of
  // the tile at (m0, n0) ----
  auto src_offset = [&](int h, int i, int m0, int n0) __attribute__((always_inline)) -> uint32_t {
    const int lr = dma_local_row(wave, i, lane), c = dma_chunk(wave, i, lane), r = tile_row(h, lr);
    if (is_weight_half(h)) {
      // SwiGLU: the tile's feature rows are 128 gate rows (A half 0 of both feature halves) and the 128 up rows
      // that pair with them (A half 1)
      const int row = EPI == TEPI_SILU ? ((r >> 6) & 1) * (a.N >> 1) + (n0 >> 1) + (r >> 7) * 64 + (r & 63) : n0 + r;
      return (uint32_t)(((int64_t)min(row, a.N - 1) * a.K + c * 8) * 2);
    }
    return (uint32_t)(((int64_t)min(m0 + r, a.M - 1) * a.ldx + c * 8) * 2);
  };
  int blk = (int)blockIdx.x;  // "block id" of the current tile
  auto coords = [&](int b, int& m0_, int& n0_) __attribute__((always_inline)) {
    const int tid = tile_of_block(b, a.tiles_t, a.tiles_f, (V & 4) != 0);
    m0_ = (tid / a.tiles_f) * TILE_T;
    n0_ = (tid % a.tiles_f) * TILE_F;
  };
  int m0, n0, m0_next = 0, n0_next = 0;
  coords(blk, m0, n0);
  bool has_next = blk + stride < ntiles;
  if (has_next) coords(blk + stride, m0_next, n0_next);
  // src_off[h][i] belongs to the tile that half-tile h is CURRENTLY being fetched for: the stream runs two K steps
  // ahead, so near the end of a tile the offsets of the A0 / B halves, then of A1, switch to the next tile
  uint32_t src_off[4][2];
#pragma unroll
  for (int h = 0; h < 4; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i) src_off[h][i] = src_offset(h, i, m0, n0);

  // The K steps of a workgroup form ONE stream over all its tiles; `par` is the parity of the stream position of
  // the step being computed (it selects the four LDS slots of that step) and simply keeps toggling across tiles.
  int par = 0;
  // issue piece i of half-tile h of step kt_target (< KT) of the current tile into the slots of parity p
  auto issue_cur = [&](int h, int i, int kt_target, int p) __attribute__((always_inline)) {
    if ((V & 32) && kt_target > 1) return;
    const char* src = reinterpret_cast<const char*>(is_weight_half(h) ? a.w : a.x) + kbeg_bytes + (int64_t)kt_target * (BK * 2) + src_off[h][i];
    char* dst = lds + (p * 4 + h) * HALF_BYTES + dma_block(wave, i) * 1024;
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
  };
  // the same for step ke (0 or 1) of the workgroup's NEXT tile (src_off[h] already points at it); without a next
  // tile nothing is requested, and the waits of the last two K steps ask for correspondingly fewer pieces in flight
  auto issue_next = [&](int h, int i, int ke, int p) __attribute__((always_inline)) {
    if ((V & 32) || !has_next) return;
    const char* src = reinterpret_cast<const char*>(is_weight_half(h) ? a.w : a.x) + kbeg_bytes + (int64_t)ke * (BK * 2) + src_off[h][i];
    char* dst = lds + (p * 4 + h) * HALF_BYTES + dma_block(wave, i) * 1024;
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
  };

  // ---- fragment reads: per-lane byte offsets inside a half-tile, plus the parity's 64 KiB ----
  int kxa[4], kxb[4];
  {
    const int rowoff = (l31 >> 3) * 1024 + (l31 & 7) * 128, sw = swizzle(l31);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int kx = rowoff + ((frag_chunk(kk, hi) ^ sw) << 4);
      kxa[kk] = kx + fh * 8192;  // + h * HALF_BYTES + f * 4096 as immediates
      kxb[kk] = kx + tq * 4096;  // + h * HALF_BYTES
    }
  }
  auto flip_parity = [&]() __attribute__((always_inline)) {
    par ^= 1;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      kxa[kk] ^= 4 * HALF_BYTES;
      kxb[kk] ^= 4 * HALF_BYTES;
    }
  };

  u32x4 Af[2][4], B0[4], B1[4];
  f32x16 acc[4][2];
  auto zero_acc = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][b][r] = 0.f;
  };
  zero_acc();

  bool ablate_reads = false;  // V & 64: only the first K step reads its fragments
  auto read_a = [&](int h) __attribute__((always_inline)) {
    if ((V & 64) && ablate_reads) return;
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        Af[f][kk] = *reinterpret_cast<const u32x4*>(lds + h * HALF_BYTES + f * 4096 + kxa[kk]);
  };
  auto read_b = [&](int h, u32x4 (&B)[4]) __attribute__((always_inline)) {
    if ((V & 64) && ablate_reads) return;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) B[kk] = *reinterpret_cast<const u32x4*>(lds + h * HALF_BYTES + kxb[kk]);
  };
  // the four MFMAs of k group kk of a phase: A half ah x (B half bx, B half by) - four independent accumulators
  auto mma_k = [&](int ah, int kk, const u32x4 (&Bx)[4], int bx, const u32x4 (&By)[4], int by) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      acc[ah * 2 + f][bx] =
          __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(Af[f][kk]), as_frag(Bx[kk]), acc[ah * 2 + f][bx], 0, 0, 0);
      acc[ah * 2 + f][by] =
          __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(Af[f][kk]), as_frag(By[kk]), acc[ah * 2 + f][by], 0, 0, 0);
    }
  };

  // One K step.  MODE 0: steps 0 .. KT - 3 (everything it requests belongs to this tile); MODE 1: step KT - 2 (A0, B0
  // of step kt + 2 are the next tile's step 0); MODE 2: step KT - 1 (B1, A1 of the next tile's step 0, A0, B0 of its
  // step 1).  ALL DMA is issued from the read segments, between the ds_reads: a DMA instruction blocks its wave for
  // ~75 cycles, which inside an MFMA cluster is 75 cycles of idle matrix pipe (measured: 20-26 % of the kernel),
  // while a reading wave's partner is computing.
  auto kstep = [&](int kt, auto modec) __attribute__((always_inline)) {
    constexpr int MODE = decltype(modec)::value;
    auto issue_1 = [&](int h, int i) __attribute__((always_inline)) {  // B half 1 / A half 1, one step ahead
      if (MODE == 2) issue_next(h, i, 0, par ^ 1);
      else issue_cur(h, i, kt + 1, par ^ 1);
    };
    auto issue_2 = [&](int h, int i) __attribute__((always_inline)) {  // A half 0 / B half 0, two steps ahead
      if (MODE == 0) issue_cur(h, i, kt + 2, par);
      else issue_next(h, i, MODE - 1, par);
    };
    // R_P0: A half 0, B half 0, B half 1 of this step; DMA of B half 1 and A half 1 of the next step
    if (MODE == 2 && has_next) {  // from here on B half 1 and A half 1 are fetched for the next tile
#pragma unroll
      for (int h = 2; h < 4; ++h)
#pragma unroll
        for (int i = 0; i < 2; ++i) src_off[h][i] = src_offset(h, i, m0_next, n0_next);
    }
    read_a(0);
    issue_1(2, 0);
    issue_1(2, 1);
    read_b(1, B0);
    issue_1(3, 0);
    read_b(2, B1);
    issue_1(3, 1);
    __builtin_amdgcn_sched_barrier(0);
    // a tile's first wait: the previous tile's stores share the counter with the loads, drain it once
    if (V & 128) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    else if (V & 256) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // ablation: DMA never waited for
    else if (kt == 0 || (V & 32) || (MODE == 2 && !has_next))  // (a workgroup's last K step: nothing newer is in flight)
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    // M_P0
    mma_k(0, 0, B0, 0, B1, 1);
    mma_k(0, 1, B0, 0, B1, 1);
    mma_k(0, 2, B0, 0, B1, 1);
    mma_k(0, 3, B0, 0, B1, 1);
    __builtin_amdgcn_sched_barrier(0);
    if (!(V & 128)) MI_GT_BARRIER();
    // R_P1: A half 1 of this step; DMA of A half 0 and B half 0 two steps ahead
    if ((MODE == 1 || (MODE == 2 && KT == 1)) && has_next) {  // from here on A half 0 and B half 0 are the next tile's
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 2; ++i) src_off[h][i] = src_offset(h, i, m0_next, n0_next);
    }
    read_a(3);
    issue_2(0, 0);
    issue_2(0, 1);
    issue_2(1, 0);
    issue_2(1, 1);
    __builtin_amdgcn_sched_barrier(0);
    if (V & 128) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    else if (V & 256) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else if ((V & 32) || (MODE == 2 && !has_next)) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else if (MODE == 1 && !has_next)  // the last tile's second-to-last step requested nothing here: only A1 of the last step flies
      asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    // M_P1
    mma_k(1, 0, B1, 1, B0, 0);
    mma_k(1, 1, B1, 1, B0, 0);
    mma_k(1, 2, B1, 1, B0, 0);
    mma_k(1, 3, B1, 1, B0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (!(V & 128)) MI_GT_BARRIER();
    flip_parity();
    ablate_reads = true;
  };

  // ---- epilogue of the tile at (m0, n0): lane (hi, l31) holds token acc_token(...), features 8 rq + 4 hi + {0..3} of
  // each 32-row fragment.  Two register quads (rq, rq + 1) are exchanged between the half-waves
  // (v_permlane32_swap) so that every lane stores 8 consecutive features = 16 bytes: half the store instructions
  // for the same bytes.
  const int n_out = EPI == TEPI_SILU ? a.N >> 1 : a.N;
  const bool wide = !(V & 8) && n_out % 8 == 0 && a.ldy % 8 == 0;
  char* const stg = lds + SLOTS * HALF_BYTES + wave * STAGE_BYTES;
  auto epilogue = [&]() __attribute__((always_inline)) {
    if (V & 512) {  // ablation: no output (the accumulators are kept alive by an empty asm)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < 2; ++b) asm volatile("" ::"v"(acc[j][b]));
      return;
    }
    if (EPI == TEPI_PARTIAL) {  // fp32 sums of this K slice: [slice][token][feature], 16 bytes per lane and register quad
#pragma unroll
      for (int bh = 0; bh < 2; ++bh) {
        const int tok = m0 + acc_token(tq, bh, l31);
        float* prow = a.part + ((int64_t)blockIdx.y * a.M + min(tok, a.M - 1)) * a.N;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int rq = 0; rq < 4; ++rq) {
            const int col = n0 + acc_feature(fh, j >> 1, j & 1, 4 * rq, hi);
            if (tok < a.M && col < a.N)
              *reinterpret_cast<f32x4*>(prow + col) =
                  f32x4{acc[j][bh][4 * rq], acc[j][bh][4 * rq + 1], acc[j][bh][4 * rq + 2], acc[j][bh][4 * rq + 3]};
          }
      }
      return;
    }
#pragma unroll
    for (int bh = 0; bh < 2; ++bh) {
      const int tok = m0 + acc_token(tq, bh, l31);
      const bool tok_ok = tok < a.M;
      uint16_t* yrow = a.y + (int64_t)min(tok, a.M - 1) * a.ldy;
#pragma unroll
      for (int j = 0; j < (EPI == TEPI_SILU ? 2 : 4); ++j) {
        // first column of this fragment for hi = 0, rq = 0 (tile feature row fh * 128 + (j >> 1) * 64 + (j & 1) * 32)
        const int col0 = EPI == TEPI_SILU ? (n0 >> 1) + fh * 64 + j * 32 : n0 + acc_feature(fh, j >> 1, j & 1, 0, 0);
        u32x2 pk[4];
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
          const int col = col0 + 8 * rq + 4 * hi;
          float o[4];
          if (EPI == TEPI_SILU) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              // the gate_up GEMM output rounded to bf16 as the unfused path, then silu in fp32 on the hardware
              // exp2 / reciprocal (v_exp_f32, v_rcp_f32: a few fp32 ulps, i.e. below the bf16 rounding that follows
              // except at ties; the libm expf + IEEE division of mi_silu_mul cost the 256 x 256 tile's epilogue - which
              // nothing overlaps - 15 % of the kernel)
              const float gb = rbf(acc[j][bh][4 * rq + e]);
              const float sb = rbf(gb * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gb * -1.4426950408889634f)));
              o[e] = sb * rbf(acc[2 + j][bh][4 * rq + e]);
            }
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = acc[j][bh][4 * rq + e];
            if (BIAS && col < n_out) {
              const u32x2 bw = *reinterpret_cast<const u32x2*>(a.bias + col);
              o[0] += lo_bf(bw[0]);
              o[1] += hi_bf(bw[0]);
              o[2] += lo_bf(bw[1]);
              o[3] += hi_bf(bw[1]);
            }
          }
          pk[rq] = u32x2{pack_bf(o[0], o[1]), pack_bf(o[2], o[3])};
        }
        if (wide) {
#pragma unroll
          for (int p2 = 0; p2 < 2; ++p2) {
            // lanes 32..63 of quad 2 p2 <-> lanes 0..31 of quad 2 p2 + 1: lanes < 32 then hold features
            // 16 p2 .. 16 p2 + 7 of the fragment, lanes >= 32 features 16 p2 + 8 .. 16 p2 + 15
            const auto sx = __builtin_amdgcn_permlane32_swap(pk[2 * p2][0], pk[2 * p2 + 1][0], false, false);
            const auto sy = __builtin_amdgcn_permlane32_swap(pk[2 * p2][1], pk[2 * p2 + 1][1], false, false);
            const u32x4 v = {sx[0], sy[0], sx[1], sy[1]};
            if (!(V & 8192)) {  // straight from the accumulator layout: 32 rows x 32 bytes per instruction (the default)
              const int col = col0 + 8 * (2 * p2 + hi);
              if (tok_ok && col < n_out) *reinterpret_cast<u32x4*>(yrow + col) = v;
            } else {
              // into the wave's stage: row l31, 16-byte chunk (j & 1) * 4 + 2 p2 + hi of a 128-byte line, XOR-swizzled by
              // the row so that the eight lanes of a ds_write_b128 group hit eight different chunks
              const int chunk = ((j & 1) * 4 + 2 * p2 + hi) ^ (l31 & 7);
              *reinterpret_cast<u32x4*>(stg + l31 * 128 + chunk * 16) = v;
            }
          }
          if ((V & 8192) && (j & 1)) {
            // Whole cache lines to memory.  Stored straight from the accumulator layout an instruction writes 32 bytes
            // of 32 different rows and a CU's store path moves 17 bytes per cycle; as complete 128-byte lines - eight
            // lanes per row, eight rows per instruction - it moves 49 (tools/ubench/store_pattern.hip).  The 32 x 64
            // features of two fragments pass through the wave's private 4 KiB stage; LDS operations of one wave
            // execute in order: no barrier.
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int row = 8 * r + (lane >> 3), c = lane & 7;
              const u32x4 v = *reinterpret_cast<const u32x4*>(stg + row * 128 + ((c ^ (row & 7)) << 4));
              const int t2 = m0 + acc_token(tq, bh, row), col = col0 - 32 + 8 * c;
              if (t2 < a.M && col < n_out) *reinterpret_cast<u32x4*>(a.y + (int64_t)t2 * a.ldy + col) = v;
            }
          }
        } else {
#pragma unroll
          for (int rq = 0; rq < 4; ++rq) {
            const int col = col0 + 8 * rq + 4 * hi;
            if (tok_ok && col < n_out) *reinterpret_cast<u32x2*>(yrow + col) = pk[rq];
          }
        }
      }
    }
  };

  if (V & 1024) {  // workgroups start up to 6 us apart, in four groups per XCD: their output bursts interleave
    for (int d = ((int)blockIdx.x >> 3) & 3; d > 0; --d) __builtin_amdgcn_s_sleep(63);
  }
  // prologue, in the stream's order (R_P1 issues A0, B0 two steps ahead; R_P0 issues B1, A1 one step ahead):
  // A0, B0 of step 0 | B1, A1 of step 0 | A0, B0 of step 1; everything but the six newest pieces - that is A0, B0,
  // B1 of step 0 - landed and published.  (K = 64: "step 1" is the next tile's step 0.)
#pragma unroll
  for (int h = 0; h < 4; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i) issue_cur(h, i, 0, 0);
  if (KT > 1) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) issue_cur(h, i, 1, 1);
  } else {
    if (has_next) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 2; ++i) src_off[h][i] = src_offset(h, i, m0_next, n0_next);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) issue_next(h, i, 0, 1);
  }
  __builtin_amdgcn_sched_barrier(0);
  if (KT > 1 || has_next) asm volatile("s_waitcnt vmcnt(6)\n\ts_barrier" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(2)\n\ts_barrier" ::: "memory");  // one K step, one tile: only A half 1 still flies
  if (!(V & 2) && fh == 1) MI_GT_BARRIER();  // the second wave of every SIMD runs one barrier behind the first
  __builtin_amdgcn_sched_barrier(0);

  for (;;) {
    for (int kt = 0; kt < KT - 2; ++kt) kstep(kt, std::integral_constant<int, 0>{});
    if (KT > 1) kstep(KT - 2, std::integral_constant<int, 1>{});
    kstep(KT - 1, std::integral_constant<int, 2>{});
    __builtin_amdgcn_sched_barrier(0);
    epilogue();
    __builtin_amdgcn_sched_barrier(0);
    if (!has_next) break;
    zero_acc();
    blk += stride;
    m0 = m0_next;
    n0 = n0_next;
    has_next = blk + stride < ntiles;
    if (has_next) coords(blk + stride, m0_next, n0_next);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the past-the-end loads must not outlive the workgroup's LDS
  if (!(V & 2) && fh == 0) MI_GT_BARRIER();         // barrier counts match again
}

#include "gemm_w4_kernel.hpp"
#include "gemm_w16_kernel.hpp"

#include "gemm_mid_kernel.hpp"

// sum of the split-K slices in slice order, (+ bias), one rounding to bf16: four features per thread
static __global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, int nsplit,
                                                                   const uint16_t* __restrict__ bias,
                                                                   uint16_t* __restrict__ y, int64_t ldy, int M, int N) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int nq = N >> 2;
  if (idx >= (int64_t)M * nq) return;
  const int row = (int)(idx / nq), col = (int)(idx % nq) * 4;
  f32x4 s = *reinterpret_cast<const f32x4*>(part + (int64_t)row * N + col);
  for (int k = 1; k < nsplit; ++k) s += *reinterpret_cast<const f32x4*>(part + ((int64_t)k * M + row) * N + col);
  if (bias) {
    const u32x2 bw = *reinterpret_cast<const u32x2*>(bias + col);
    s[0] += lo_bf(bw[0]);
    s[1] += hi_bf(bw[0]);
    s[2] += lo_bf(bw[1]);
    s[3] += hi_bf(bw[1]);
  }
  *reinterpret_cast<u32x2*>(y + (int64_t)row * ldy + col) = u32x2{pack_bf(s[0], s[1]), pack_bf(s[2], s[3])};
}

// K slices for a shape whose tiles cannot fill the chip (few token rows x a narrow projection): the smallest
// power of two that brings tiles x slices to ~one workgroup per CU, every slice at least four K steps deep
static int tile_ksplit(int M, int N, int K) {
  const int ntiles = ((M + TILE_T - 1) / TILE_T) * ((N + TILE_F - 1) / TILE_F), kt = K / BK;
  int ks = 1;
  while (ntiles * ks * 2 <= kPersistentGrid && kt % (ks * 2) == 0 && kt / (ks * 2) >= 4 && ks < 16) ks *= 2;
  return ks;
}

// The large-M kernel: gemm_w16_kernel (four waves, v_mfma_f32_16x16x32_bf16), with whole-line output stores
// (kLineStores) wherever the output allows it: full feature tiles (plain results: full halves, a wave's 128 features - a head of 151936 rows, us,
// 200 tokens 104 -> 97, 256 112 -> 102, 400 173 -> 163), 16-byte aligned rows, 32-bit byte offsets.
// Tuning / comparison variants: V & kDirectStores keeps the direct stores; V & kMfma32 = the same kernel on
// v_mfma_f32_32x32x16_bf16 (gemm_w4_kernel: the first form, still the qkv-store kernel); V & kEightWaves = the
// eight-wave ping-pong kernel before both.
constexpr int kEightWaves = 1 << 20, kMfma32 = 1 << 19, kLineStores = 32768, kDirectStores = 1 << 18;
template <int EPI, bool BIAS, int V = kDefaultV>
static int launch_tile(const TileArgs& a, hipStream_t st, int ksplit = 1) {
  // persistent workgroups: one per CU; the grid is a multiple of 8, so a workgroup stays in one XCD class
  const int ntiles = a.tiles_f * a.tiles_t;
  const bool persistent = !(V & 16) && ntiles > kPersistentGrid;
  const dim3 grid(persistent ? kPersistentGrid : ntiles, ksplit);
  constexpr int VK = V & ~(kDirectStores | kMfma32 | kEightWaves);  // the kernel's own flags
  const bool lines = EPI != TEPI_PARTIAL && !(V & (kDirectStores | 8 | 512)) && a.N % (EPI == TEPI_SILU || (V & kMfma32) ? TILE_F : TILE_F / 2) == 0 && a.ldy % 8 == 0 &&
                     (int64_t)a.M * a.ldy * 2 < ((int64_t)1 << 32) && (reinterpret_cast<uintptr_t>(a.y) & 15) == 0;
  if constexpr ((V & kEightWaves) != 0) {
    hipLaunchKernelGGL((gemm_tile_kernel<EPI, BIAS, VK>), grid, dim3(512), 0, st, a);
  } else if constexpr ((V & kMfma32) != 0) {
    if (lines) hipLaunchKernelGGL((gemm_w4_kernel<EPI, BIAS, VK | kLineStores>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((gemm_w4_kernel<EPI, BIAS, VK>), grid, dim3(256), 0, st, a);
  } else {
    if (lines) hipLaunchKernelGGL((gemm_w16_kernel<EPI, BIAS, VK | kLineStores>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((gemm_w16_kernel<EPI, BIAS, VK>), grid, dim3(256), 0, st, a);
  }
  return check_launch();
}

// ---- which kernel, how many K slices ----
// Where the 256-tiles are fewer than the CUs: the shape of tile (gemm_mid_kernel's, or still the large one's) and the number of K slices whose
// modelled time is the least; all give the same bits but for the slices.  Modelled: a launch, the rounds of its tiles, the K steps of a round - which take
// the longer the more of the chip's places are in use (the L2s' rate: (F + T) 128 bytes per tile and step) - and with K slices the fp32 partial sums out
// and back and the second launch.  The constants are fitted to random products (65 .. 6000 rows, K from 512 on; 64 x 128: 677 of them, 6 % off in the mean,
// the others 7 to 14 %; a launch of the two-place shapes by 500 of K 64 to 512), those of 64 x 64 and 128 x 64 corrected by whole prompt steps, whose activations another kernel has just written (1260 rows, 28
// layers, us a step with o on 128 x 64 / 64 x 64 3131 / 3084, down 3131 / 3045).  Over another 674 (K from 256 on, every launch's weights from memory) the
// choice is 1.0 % above the best shape and number of slices in the mean, SwiGLU 0.7 %, over the 500 of short K 0.8 and 0.9; without 64 x 128, the best shape
// of half of the former with SwiGLU, 2.5 % and 2.8 %.  Two-place shapes: rings of which two fit a CU; 128 x 64 and 128 x 128 have a deeper one too, a tile per CU, whose requests reach further
// ahead.  us, 64 x 64 / 128 x 64 / 128 x 128 / 128 x 192 / 256 x 256 (the better ring of each): 137 x 4096 x 1024 6.2 / 8.8 / 10.3 / 13.6 / 24, 500
// rows 10.7 / 9.8 / 12.2 / 13.8 / 26, 886 rows 16.2 / 12.9 / 12.8 / 14.4 / 25, 1260 rows 19.1 / 18.8 / 17.9 / 15.8 / 26, 2048 rows 30 / 25 / 22.1 / 28 /
// 29; 886 x 5120 x 2048 35 / 33 / 32 / 24.8 / 43; 1260 x 1024 x 2048 14.4 / 11.9 / 14.8 / 19.6 / 40, 2450 rows 21.7 / 20.7 / 16.6 / 20.2 / 40; 128 x 64 / 64 x
// 128 (another card): with SwiGLU 215 x 6400 x 832 9.6 / 7.9, 314 x 2304 x 2752 22.2 / 19.1, without 348 x 4672 x 1152 11.2 / 9.2.  Against the choice among 64 x 64,
// 64 x 128, 128 x 128 and 256 x 256 by one time per step each (and that kernel's longer steps), 500 products with weights from memory: 0.89 of the
// time in the geometric mean, 9 of them slower by more than 2 % (17 % at most).
struct MidTile {
  int f, t, places;  // features, tokens; tiles that share a CU
  double launch_us, round_us, step_us, step_load_us, pair_us, pair_load_us;
};
// (a tile's two fragments of features are a gate's and an up's with SwiGLU: 64 x 64 has one only)
enum { kMid128, kMid128Pairs, kMid128x64Pairs, kMid128x64, kMid128x192, kMid64x128, kMid64, kMidTileCount };
constexpr MidTile kMidTiles[kMidTileCount] = {{128, 128, 1, 2.2, 1.8, 0.32, 0.24, 0., 0.},     {128, 128, 2, 1.5, 1.8, 0.57, 0.27, 0.89, 0.10},
                                              {128, 64, 2, 3.3, 0., 0.29, 0.18, 0.60, 0.18},  {128, 64, 1, 2.8, 1.4, 0.21, 0.21, 0., 0.},
                                              {128, 192, 1, 1.7, 3.1, 0.43, 0.29, 0., 0.},     {64, 128, 2, 2.8, 0., 0.25, 0.10, 0.52, 0.15},
                                              {64, 64, 2, 2.75, 0., 0.14, 0.08, 0.32, 0.12}};
constexpr MidTile kLargeTile = {256, 256, 1, 3.1, 3.7, 1.04, 0.48, 0., 0.};
// the sum of K slices: its launch and its bytes (a launch of 2 us misses the best of all shapes and numbers of slices by 1.0 % over the 674 products, one of 3.2 by
// 1.3; us, best with / without: 361 x 384 x 2560 9.4 / 13.2, 127 x 1984 x 3456 13.4 / 17.4, 166 x 2048 x 3456 13.1 / 15.7)
constexpr double kLaunchUs = 2.0, kPartialBytesPerUs = 4.0e6;

// fewer 256-tiles than CUs
static bool few_tiles(int M, int N) {
  return (int64_t)((M + TILE_T - 1) / TILE_T) * ((N + TILE_F - 1) / TILE_F) < kPersistentGrid;
}
struct MidPick {
  int tile, ksplit;  // tile -1: the large kernel
};
// modelled time of `tiles` tiles of kt K steps: whole rounds of all CUs, then what is left, whose steps take the less the fewer they are
static double tiles_us(const MidTile& s, int64_t tiles, int kt) {
  const int64_t round = (int64_t)s.places * kPersistentGrid, rest = tiles % round;
  const auto step = [&](int64_t n) {
    return s.places == 2 && n > kPersistentGrid ? s.pair_us + s.pair_load_us * (n - kPersistentGrid) / kPersistentGrid
                                                : s.step_us + s.step_load_us * n / kPersistentGrid;
  };
  return s.launch_us + (double)(tiles / round) * (s.round_us + kt * step(round)) + (rest ? s.round_us + kt * step(rest) : 0.);
}
// fixed_ks: the caller wants that many slices' sums; 0: whatever is fastest, the sum of the slices included
static MidPick pick_mid(int M, int N, int K, bool silu, int fixed_ks = 0) {
  const int kt = K / BK;
  const auto tiles = [&](const MidTile& s) { return (int64_t)((M + s.t - 1) / s.t) * ((N + s.f - 1) / s.f); };
  MidPick pick{-1, 1};
  double best = fixed_ks ? 1e30 : tiles_us(kLargeTile, tiles(kLargeTile), kt);
  for (int i = 0; i < (silu ? kMid64 : kMidTileCount); ++i)
    for (int ks = fixed_ks ? fixed_ks : 1; ks <= (fixed_ks ? fixed_ks : silu ? 1 : 16); ks *= 2) {
      if (!fixed_ks && (kt % ks || (ks > 1 && kt / ks < 2))) break;
      double t = tiles_us(kMidTiles[i], tiles(kMidTiles[i]) * ks, kt / ks);
      if (!fixed_ks && ks > 1) t += 2.0 * ks * (double)M * N * sizeof(float) / kPartialBytesPerUs + kLaunchUs;
      if (t < best) best = t, pick = MidPick{i, ks};
    }
  return pick;
}

// mi_gemm_bf16's plan
static MidPick tile_plan(int M, int N, int K, bool silu) {
  if (few_tiles(M, N)) return pick_mid(M, N, K, silu);
  return MidPick{-1, silu ? 1 : tile_ksplit(M, N, K)};
}

// (log2 of the) runs of features that the XCDs share the tiles in: the fewest rows of both operands into all L2s.  us within a prompt step, eight runs / this:
// 1842 rows x 1024 features x 2048 and x 3072 21.1 / 19.9 on average, 2450 rows 22.7 / 21.7, 886 rows 13.8 / 13.2; few rows and many features keep
// eight (137 x 4096 x 1024: eight 7.0, four 6.9, two 7.4, one 7.3; 886 x 6144 x 1024 16.2 / 16.0, one 18.0).
static int xcd_features(int M, int N, int tiles_f) {
  const auto rows = [&](int lf) { return ((int64_t)M << lf) + ((int64_t)N << (3 - lf)); };
  int best = 0;
  for (int lf = 1; lf <= 3 && tiles_f % (1 << lf) == 0; ++lf)
    if (rows(lf) < rows(best)) best = lf;
  return best;
}

template <int EPI, bool BIAS>
static int launch_mid(TileArgs a, hipStream_t st, MidPick pick) {
  const MidTile& s = kMidTiles[pick.tile];
  a.tiles_f = (a.N + s.f - 1) / s.f;
  a.tiles_t = (a.M + s.t - 1) / s.t;
  a.xcd_lf = xcd_features(a.M, a.N, a.tiles_f);
  const dim3 grid((a.tiles_f * a.tiles_t + 7) / 8 * 8, pick.ksplit);
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, a);
    return check_launch();
  };
  switch (pick.tile) {
    case kMid128: return go(gemm_mid_kernel<EPI, BIAS, 4, TileArgs, Mid128>);
    case kMid128Pairs: return go(gemm_mid_kernel<EPI, BIAS, 2, TileArgs, Mid128>);
    case kMid128x64Pairs: return go(gemm_mid_kernel<EPI, BIAS, 3, TileArgs, MidShape<2, 2, 2, 1>>);
    case kMid128x64: return go(gemm_mid_kernel<EPI, BIAS, 6, TileArgs, MidShape<2, 2, 2, 1>>);
    case kMid128x192: return go(gemm_mid_kernel<EPI, BIAS, 3, TileArgs, MidShape<2, 2, 2, 3>>);
    case kMid64x128: return go(gemm_mid_kernel<EPI, BIAS, 3, TileArgs, MidShape<1, 4, 2, 1>>);
    default: break;
  }
  if constexpr (EPI != TEPI_SILU) return go(gemm_mid_kernel<EPI, BIAS, 5, TileArgs, MidShape<2, 2, 1, 1>>);
  return MI_EUNSUPPORTED;  // (never picked)
}

static int check_tile_gemm(const void* x, int64_t ldx, const void* w, const void* bias, const void* y, int64_t ldy,
                           int M, int N, int K, int epilogue) {
  if (!x || !w || !y || M < 0 || N <= 0 || K <= 0 || ldx < K) return MI_EINVAL;
  if (epilogue != 0 && epilogue != 1) return MI_EINVAL;
  if (!aligned16(x) || !aligned16(w) || !aligned16(y) || (bias && !aligned16(bias))) return MI_EINVAL;
  if (K % BK || N % 4 || ldx % 8 || ldy % 4) return MI_EUNSUPPORTED;
  if (epilogue == 1 && (bias || (N / 2) % 128)) return MI_EUNSUPPORTED;  // (the 128-tile kernel alone would take % 64)
  if (ldy < (epilogue == 1 ? N / 2 : N)) return MI_EINVAL;
  // the DMA sources are 32-bit byte offsets from the operand bases
  // (and 0xF0000000 must lie beyond both: the four-wave kernel's "fetch nothing" offset)
  if (((int64_t)N + 256) * K * 2 >= (int64_t)1 << 31 || ((int64_t)M + 256) * ldx * 2 >= (int64_t)1 << 31) return MI_EUNSUPPORTED;
  return MI_OK;
}

}  // namespace mi

using namespace mi;

// The shape contract of mi_gemm_bf16 as a query (the same tests as check_tile_gemm): the largest M one launch takes on
// a [N][K] weight with activation row stride ldx, 0 when the weight shape itself is refused.
extern "C" int64_t mi_gemm_bf16_max_rows(int N, int K, int64_t ldx) {
  if (N <= 0 || K <= 0 || K % BK || N % 4 || ldx < K || ldx % 8) return 0;
  if (((int64_t)N + 256) * K * 2 >= (int64_t)1 << 31) return 0;
  const int64_t m = (((int64_t)1 << 30) - 1) / ldx - 256;  // (M + 256) * ldx * 2 < 2^31
  return m > 0 ? m : 0;
}

extern "C" size_t mi_gemm_bf16_workspace(int M, int N, int K, int epilogue) {
  if (M <= 0 || N <= 0 || K <= 0 || K % BK || epilogue != 0) return 0;
  const int ks = tile_plan(M, N, K, false).ksplit;
  return ks > 1 ? (size_t)ks * M * N * sizeof(float) : 0;
}

extern "C" int mi_gemm_bf16(const mi_bf16* x, int64_t ldx, const mi_bf16* w, const mi_bf16* bias, mi_bf16* y,
                            int64_t ldy, int M, int N, int K, int epilogue, void* workspace, size_t ws_bytes,
                            mi_stream stream) {
  const int rc = check_tile_gemm(x, ldx, w, bias, y, ldy, M, N, K, epilogue);
  if (rc != MI_OK || M == 0) return rc;
  TileArgs a{x, w, bias, y, ldx, ldy, M, N, K, (N + TILE_F - 1) / TILE_F, (M + TILE_T - 1) / TILE_T, 0, nullptr};
  hipStream_t st = S(stream);
  const MidPick pick = tile_plan(M, N, K, epilogue == 1);
  const bool mid = pick.tile >= 0;
  if (epilogue == 1) return mid ? launch_mid<TEPI_SILU, false>(a, st, pick) : launch_tile<TEPI_SILU, false>(a, st);
  const int ks = pick.ksplit;
  if (ks > 1) {  // two launches: K slices as fp32 partial sums, then their sum (+ bias) rounded once
    if (!workspace || !aligned16(workspace) || ws_bytes < (size_t)ks * M * N * sizeof(float)) return MI_EWORKSPACE;
    a.part = static_cast<float*>(workspace);
    const int rc2 = mid ? launch_mid<TEPI_PARTIAL, false>(a, st, pick) : launch_tile<TEPI_PARTIAL, false>(a, st, ks);
    if (rc2 != MI_OK) return rc2;
    const int64_t quads = (int64_t)M * (N / 4);
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, st, a.part, ks, bias, y,
                       ldy, M, N);
    return check_launch();
  }
  if (mid) return bias ? launch_mid<TEPI_NONE, true>(a, st, pick) : launch_mid<TEPI_NONE, false>(a, st, pick);
  return bias ? launch_tile<TEPI_NONE, true>(a, st) : launch_tile<TEPI_NONE, false>(a, st);
}

// fp32 sums of `ksplit` K slices [ksplit][M][N] (mi_gemm_bf16_packed_splitk's result for the weight as stored), for the norm that adds
// them up
extern "C" int mi_gemm_bf16_splitk(const mi_bf16* x, int64_t ldx, const mi_bf16* w, float* partials, int M, int N, int K, int ksplit,
                                   mi_stream stream) {
  const int rc = check_tile_gemm(x, ldx, w, nullptr, partials, N, M, N, K, 0);
  if (rc != MI_OK) return rc;
  if (ksplit < 1 || ksplit > 65535 || K % ((int64_t)BK * ksplit)) return MI_EUNSUPPORTED;
  if (M == 0) return MI_OK;
  TileArgs a{x, w, nullptr, nullptr, ldx, N, M, N, K, 0, 0, 0, partials};
  return launch_mid<TEPI_PARTIAL, false>(a, S(stream), pick_mid(M, N, K, false, ksplit));
}

// The packed qkv projection with the K / V heads stored straight into the paged cache (TEPI_QKV, gemm_w4_kernel.hpp)
extern "C" int mi_gemm_bf16_qkv_store(const mi_bf16* x, int64_t ldx, const mi_bf16* w, const mi_bf16* bias, mi_bf16* qkv,
                                      int64_t ldy, int M, int N, int K, const mi_bf16* k_w, float eps,
                                      const int64_t* positions, const float* cos_sin, mi_bf16* k_cache,
                                      mi_bf16* v_cache, const int32_t* slots, int n_q_heads, int n_kv_heads,
                                      int head_dim, int block_size, mi_stream stream) {
  const int rc = check_tile_gemm(x, ldx, w, bias, qkv, ldy, M, N, K, 0);
  if (rc != MI_OK) return rc;
  if (!positions || !cos_sin || !k_cache || !v_cache || !slots || n_q_heads <= 0 || n_kv_heads <= 0) return MI_EINVAL;
  if (!aligned16(k_cache) || !aligned16(v_cache) || !aligned16(slots) || !aligned16(cos_sin) || (k_w && !aligned16(k_w))) return MI_EINVAL;
  // one wave = one head; whole feature tiles and 16-byte aligned output rows (the whole-line stores of the q heads)
  if (head_dim != 128 || N != (n_q_heads + 2 * n_kv_heads) * 128 || N % TILE_F || ldy % 8 || block_size <= 0 || block_size % 16)
    return MI_EUNSUPPORTED;
  if (few_tiles(M, N) || (int64_t)M * ldy * 2 >= ((int64_t)1 << 32)) return MI_EUNSUPPORTED;  // the large-M kernel only
  if (M == 0) return MI_OK;
  TileArgs a{x, w, bias, qkv, ldx, ldy, M, N, K, N / TILE_F, (M + TILE_T - 1) / TILE_T, 0, nullptr,
             {k_w, positions, cos_sin, k_cache, v_cache, slots, eps, n_q_heads, n_kv_heads, block_size}};
  const int ntiles = a.tiles_f * a.tiles_t;
  const dim3 grid(ntiles > kPersistentGrid ? kPersistentGrid : ntiles);
  // (the 32 x 32 x 16 form of the kernel: the K-head arithmetic is written for its accumulator layout)
  if (bias) hipLaunchKernelGGL((gemm_w4_kernel<TEPI_QKV, true, kLineStores>), grid, dim3(256), 0, S(stream), a);
  else hipLaunchKernelGGL((gemm_w4_kernel<TEPI_QKV, false, kLineStores>), grid, dim3(256), 0, S(stream), a);
  return check_launch();
}

// tuning entry point (tools/gemm_bench.py): variant = schedule flags V, no bias, plain epilogue
extern "C" int mi_gemm_bf16_ex(const mi_bf16* x, int64_t ldx, const mi_bf16* w, mi_bf16* y, int64_t ldy, int M, int N,
                               int K, int variant, mi_stream stream) {
  const int rc = check_tile_gemm(x, ldx, w, nullptr, y, ldy, M, N, K, 0);
  if (rc != MI_OK || M == 0) return rc;
  const TileArgs a{x, w, nullptr, y, ldx, ldy, M, N, K, (N + TILE_F - 1) / TILE_F, (M + TILE_T - 1) / TILE_T, 0, nullptr};
  hipStream_t st = S(stream);
  switch (variant) {
    // the product kernel (four waves, 16 x 16 x 32 MFMAs) and its variants
    case 0: return launch_tile<TEPI_NONE, false, 0>(a, st);
    case 4: return launch_tile<TEPI_NONE, false, 4>(a, st);
    case 8: return launch_tile<TEPI_NONE, false, 8>(a, st);
    case 16: return launch_tile<TEPI_NONE, false, 16>(a, st);
    case kDirectStores: return launch_tile<TEPI_NONE, false, kDirectStores>(a, st);
    // the same kernel on 32 x 32 x 16 MFMAs
    case kMfma32: return launch_tile<TEPI_NONE, false, kMfma32>(a, st);
    case kMfma32 + kDirectStores: return launch_tile<TEPI_NONE, false, kMfma32 + kDirectStores>(a, st);
    // the eight-wave kernel and its variants
    case kEightWaves: return launch_tile<TEPI_NONE, false, kEightWaves>(a, st);
    case kEightWaves + 2: return launch_tile<TEPI_NONE, false, kEightWaves + 2>(a, st);
    case kEightWaves + 16: return launch_tile<TEPI_NONE, false, kEightWaves + 16>(a, st);
    case kEightWaves + 8192: return launch_tile<TEPI_NONE, false, kEightWaves + 8192>(a, st);
    // gemm_mid_kernel's shapes, no K slices
    case 65536: return launch_mid<TEPI_NONE, false>(a, st, {kMid128, 1});
    case 65538: return launch_mid<TEPI_NONE, false>(a, st, {kMid128Pairs, 1});
    case 65539: return launch_mid<TEPI_NONE, false>(a, st, {kMid128x192, 1});
    case 65540: return launch_mid<TEPI_NONE, false>(a, st, {kMid128x64Pairs, 1});
    case 65541: return launch_mid<TEPI_NONE, false>(a, st, {kMid128x64, 1});
    case 65542: return launch_mid<TEPI_NONE, false>(a, st, {kMid64, 1});
    case 65543: return launch_mid<TEPI_NONE, false>(a, st, {kMid64x128, 1});
    default: return MI_EUNSUPPORTED;
  }
}
