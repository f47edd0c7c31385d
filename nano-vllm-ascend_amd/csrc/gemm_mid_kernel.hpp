#pragma once
// ---------------------------------------------------------------------------
// The same GEMM on 128 x 128 tiles, for shapes whose 256 x 256 tiles cannot fill the chip (64 < M <= ~2048 rows:
// large decode batches, short prompts).  Four waves, each 64 features x 64 tokens (2 x 2 accumulators); one K step of
// the tile is two 16 KiB half-tiles in the layout of gemm_tile_index.hpp (A: local row = tile feature row, B: local
// row = tile token row) in a ring of NST stages.  One barrier per K step: "my pieces of step t have landed" (a COUNTED
// wait: the pieces of the NST - 2 steps behind it may still fly) -> barrier (everybody's have, and everybody is done
// reading step t - 1) -> request step t + NST - 1 into the buffer step t - 1 used -> fragments of step t -> sixteen
// MFMAs.  These shapes have at most a workgroup or two per CU and a K loop of 16-80 steps: with one step of
// prefetch (NST = 2, two workgroups per CU) every step waits out most of a DMA round trip (0.75 us per step
// measured); NST = 4 (128 KiB, one workgroup per CU) keeps three steps in flight.
// Same summation order and epilogues as the large kernel: results are bit-identical.
// SwiGLU: the tile's 128 weight rows are, per wave, 32 gate rows (fragment 0) and the 32 up rows that pair with them.
// ---------------------------------------------------------------------------
// Other shapes (MidShape): fewer features or tokens per tile where 128 x 128 tiles leave CUs without work or are filled with repeated
// rows - the ring then holds more of the shorter K steps, and about as many bytes are on their way.
template <int N, int PER_STEP>
__device__ __forceinline__ void mid_wait(int behind) {  // all but the pieces of the `behind` (<= N) newest K steps have landed
  if constexpr (N == 0) {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  } else {
    if (behind >= N) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N * PER_STEP) : "memory");
    else mid_wait<N - 1, PER_STEP>(behind);
  }
}

template <int EPI, bool BIAS, int NST, class ARGS = TileArgs, class SH = Mid128>
__global__ __launch_bounds__(64 * SH::NW, NST * SH::STAGE <= 81920 ? 2 : 1) void gemm_mid_kernel(const ARGS a) {
  constexpr int WF = SH::WF, WT = SH::WT;
  static_assert(WF == 2 || (EPI != TEPI_SILU && !ARGS::kDual), "a wave holds the gate and the up fragment of its outputs");
  __shared__ __attribute__((aligned(1024))) char lds[NST * SH::STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fw = wave / SH::TW, tw = wave % SH::TW, hi = lane >> 5, l31 = lane & 31;
  const int KT_all = a.K / BK;
  const int KT = EPI == TEPI_PARTIAL ? KT_all / (int)gridDim.y : KT_all;
  const int64_t kbeg_bytes = EPI == TEPI_PARTIAL ? (int64_t)blockIdx.y * KT * (BK * 2) : 0;
  int n0 = ((int)blockIdx.x % a.tiles_f) * SH::F, m0 = ((int)blockIdx.x / a.tiles_f) * SH::T, m_end = a.M;
  int64_t wrow0 = 0;
  if constexpr (EPI == TEPI_ANY) {
    const int ntiles = any_tiles(a);
    if ((int)blockIdx.x >= ntiles) return;  // (the grid is the host's bound on the grouped tiles)
    const AnyTile t = any_tile(a, (int)blockIdx.x, ntiles, SH::T, ARGS::kDual ? SH::F / 2 : SH::F);
    n0 = t.n0, m0 = t.m0, m_end = t.m_end, wrow0 = (int64_t)t.group * a.w_rows;
  }

  // LDS-DMA: wave w moves its share of the 1 KiB pieces (8 local rows each) of the feature rows and of the token rows
  const char* srcA[SH::A_PIECES];
  const char* srcB[SH::B_PIECES];
#pragma unroll
  for (int i = 0; i < SH::A_PIECES; ++i) {
    const int lr = (wave * SH::A_PIECES + i) * 8 + (lane >> 3), c = (lane & 7) ^ swizzle(lr);
    if constexpr (EPI == TEPI_ANY) {
      // two weights: every wave's first fragment holds 32 rows of w, its second the rows of w2 that pair with them
      const bool second = ARGS::kDual && ((lr >> 5) & 1);
      const int rowA = ARGS::kDual ? n0 + (lr >> 6) * 32 + (lr & 31) : n0 + lr;
      srcA[i] = reinterpret_cast<const char*>(second ? a.w2 : a.w) + ((wrow0 + min(rowA, a.N - 1)) * a.K + c * 8) * 2;
    } else {
      const int rowA = mid_weight_row(lr, n0, a.N, EPI == TEPI_SILU);
      srcA[i] = reinterpret_cast<const char*>(a.w) + kbeg_bytes + ((int64_t)min(rowA, a.N - 1) * a.K + c * 8) * 2;
    }
  }
#pragma unroll
  for (int i = 0; i < SH::B_PIECES; ++i) {
    const int lr = (wave * SH::B_PIECES + i) * 8 + (lane >> 3), c = (lane & 7) ^ swizzle(lr);
    int64_t rowB = min(m0 + lr, m_end - 1);
    if constexpr (EPI == TEPI_ANY)
      if (ARGS::kGather) rowB = a.x_rows[rowB];
    srcB[i] = reinterpret_cast<const char*>(a.x) + kbeg_bytes + (rowB * a.ldx + c * 8) * 2;
  }
  auto issue = [&](int kt, int p) __attribute__((always_inline)) {
    char* dst = lds + p * SH::STAGE;
#pragma unroll
    for (int i = 0; i < (SH::A_PIECES > SH::B_PIECES ? SH::A_PIECES : SH::B_PIECES); ++i) {
      if (i < SH::A_PIECES)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(srcA[i < SH::A_PIECES ? i : 0] + (int64_t)kt * (BK * 2)),
                                         (__attribute__((address_space(3))) void*)(dst + (wave * SH::A_PIECES + i) * 1024), 16, 0, 0);
      if (i < SH::B_PIECES)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(srcB[i < SH::B_PIECES ? i : 0] + (int64_t)kt * (BK * 2)),
                                         (__attribute__((address_space(3))) void*)(dst + SH::F * 128 + (wave * SH::B_PIECES + i) * 1024), 16, 0, 0);
    }
  };
  int kx[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    kx[kk] = (l31 >> 3) * 1024 + (l31 & 7) * 128 + ((frag_chunk(kk, hi) ^ swizzle(l31)) << 4);

  f32x16 acc[WF][WT];
#pragma unroll
  for (int f = 0; f < WF; ++f)
#pragma unroll
    for (int b = 0; b < WT; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[f][b][r] = 0.f;

#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if (s < KT) issue(s, s);
  int p = 0, pn = NST - 1;  // ring slots of step kt and of step kt + NST - 1
  for (int kt = 0; kt < KT; ++kt) {
    // requested so far: steps <= kt + NST - 2; the same number of pieces per step and wave, completing in order
    mid_wait<NST - 2, SH::A_PIECES + SH::B_PIECES>(min(KT - 1 - kt, NST - 2));
    __builtin_amdgcn_sched_barrier(0);
    if (kt + NST - 1 < KT) issue(kt + NST - 1, pn);
    const char* sa = lds + p * SH::STAGE + fw * WF * 4096;
    const char* sb = lds + p * SH::STAGE + SH::F * 128 + tw * WT * 4096;
    u32x4 A[WF][4], B[WT][4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
      for (int f = 0; f < WF; ++f) A[f][kk] = *reinterpret_cast<const u32x4*>(sa + f * 4096 + kx[kk]);
#pragma unroll
      for (int b = 0; b < WT; ++b) B[b][kk] = *reinterpret_cast<const u32x4*>(sb + b * 4096 + kx[kk]);
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int f = 0; f < WF; ++f)
#pragma unroll
        for (int b = 0; b < WT; ++b)
          acc[f][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(A[f][kk]), as_frag(B[b][kk]), acc[f][b], 0, 0, 0);
    p = p + 1 == NST ? 0 : p + 1;
    pn = pn + 1 == NST ? 0 : pn + 1;
  }

  // epilogue: lane (hi, l31) holds token (tw WT + b) 32 + l31, features 8 rq + 4 hi + {0..3} of each 32-row fragment
  if constexpr (EPI == TEPI_ANY) {
#pragma unroll
    for (int b = 0; b < WT; ++b) {
      const AnyRow row = any_row(a, m0 + (tw * WT + b) * 32 + l31, m_end);
#pragma unroll
      for (int f = 0; f < (ARGS::kDual ? 1 : WF); ++f)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
          const int col = n0 + (ARGS::kDual ? fw : fw * WF + f) * 32 + 8 * rq + 4 * hi;
          f32x4 v, v2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = acc[f][b][4 * rq + e];
            if (ARGS::kDual) v2[e] = acc[WF - 1][b][4 * rq + e];
          }
          any_store(a, row, col, v, v2);
        }
    }
    return;
  }
  const int n_out = EPI == TEPI_SILU ? a.N >> 1 : a.N;
  const bool wide = n_out % 8 == 0 && a.ldy % 8 == 0;
#pragma unroll
  for (int b = 0; b < WT; ++b) {
    const int tok = m0 + (tw * WT + b) * 32 + l31;
    const bool tok_ok = tok < a.M;
    if (EPI == TEPI_PARTIAL) {
      float* prow = a.part + ((int64_t)blockIdx.y * a.M + min(tok, a.M - 1)) * a.N;
#pragma unroll
      for (int f = 0; f < WF; ++f)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
          const int col = n0 + (fw * WF + f) * 32 + 8 * rq + 4 * hi;
          if (tok_ok && col < a.N)
            *reinterpret_cast<f32x4*>(prow + col) =
                f32x4{acc[f][b][4 * rq], acc[f][b][4 * rq + 1], acc[f][b][4 * rq + 2], acc[f][b][4 * rq + 3]};
        }
      continue;
    }
    uint16_t* yrow = a.y + (int64_t)min(tok, a.M - 1) * a.ldy;
#pragma unroll
    for (int f = 0; f < (EPI == TEPI_SILU ? 1 : WF); ++f) {
      const int col0 = EPI == TEPI_SILU ? (n0 >> 1) + fw * 32 : n0 + (fw * WF + f) * 32;
      u32x2 pk[4];
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const int col = col0 + 8 * rq + 4 * hi;
        float o[4];
        if (EPI == TEPI_SILU) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {  // the roundings and the silu form of the large kernel's epilogue
            const float gb = rbf(acc[0][b][4 * rq + e]);
            const float sb = rbf(gb * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gb * -1.4426950408889634f)));
            o[e] = sb * rbf(acc[WF - 1][b][4 * rq + e]);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = acc[f][b][4 * rq + e];
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
          const auto sx = __builtin_amdgcn_permlane32_swap(pk[2 * p2][0], pk[2 * p2 + 1][0], false, false);
          const auto sy = __builtin_amdgcn_permlane32_swap(pk[2 * p2][1], pk[2 * p2 + 1][1], false, false);
          const int col = col0 + 8 * (2 * p2 + hi);
          if (tok_ok && col < n_out) *reinterpret_cast<u32x4*>(yrow + col) = u32x4{sx[0], sy[0], sx[1], sy[1]};
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
}

