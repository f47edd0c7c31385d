#pragma once
// ---------------------------------------------------------------------------
// The same GEMM on smaller tiles, for shapes whose 256 x 256 tiles cannot fill the chip (large decode batches, prompts of
// some thousand rows).  128 x 128: four waves, each 64 features x 64 tokens (2 x 2 accumulators); one K step of
// the tile is two 16 KiB half-tiles in the layout of gemm_tile_index.hpp (A: local row = tile feature row, B: local
// row = tile token row) in a ring of NST stages.  One barrier per K step: "my pieces of step t + 1 have landed" (a COUNTED wait: the
// pieces of the NST - 2 steps behind it may still fly) and "I have read step t" -> barrier -> step t's matrix instructions, and behind each of
// them two fragment reads of step t + 1 and one request of step t + NST, into the slot of step t.
// What bounds it: with a tile or two per CU nothing else stands beside a wave's own waits, so a step must not have its requests, its reads
// and its matrix instructions one after the other (the reads of a 128 x 128 tile's step take a CU's LDS 512 cycles, its requests the
// address path about as long, its matrix instructions 512).  us per step of 64, 128 x 128 tiles, ring of four: two tiles 0.53 with the three one
// after the other, 0.45 with the reads a step ahead, 0.28 so; 224 tiles 0.54 / 0.46 / 0.40: now the L2s' rate, 32 KiB per tile and step = 17.5
// TB/s (64 x 64: 256 tiles 0.25 -> 0.16, 25 TB/s).  Launches (cold weights): 137 x 4096 x 1024 7.0 -> 6.3 us, 500 x 1024 x 2048 10.3 -> 7.7, 886 x 4096
// x 1024 15.0 -> 13.4, 2450 x 1024 x 3072 31.9 -> 25.5, with SwiGLU 500 x 6144 x 1024 14.7 -> 13.2.
// A ring of two steps still leaves a step's pieces one step's time to arrive (two tiles share the CU then); four (128 KiB, one tile per CU)
// keep three steps in flight.
// Same summation order and epilogues as the large kernel: results are bit-identical.
// SwiGLU: the tile's 128 weight rows are, per wave, 32 gate rows (fragment 0) and the 32 up rows that pair with them.
// ---------------------------------------------------------------------------
// Other shapes (MidShape): fewer features or tokens per tile where 128 x 128 tiles leave CUs without work or are filled with repeated
// rows - the ring then holds more of the shorter K steps, and about as many bytes are on their way.
template <int N, int PER_STEP>
__device__ __forceinline__ void mid_wait(int behind) {  // all but the pieces of the `behind` (<= N) newest K steps have landed
  if constexpr (N == 0) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  } else {
    if (behind >= N) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N * PER_STEP) : "memory");
    else mid_wait<N - 1, PER_STEP>(behind);
  }
}

// one piece: a lane's 16 bytes at byte `off` (its own) + k (the wave's) of the operand to dst + 16 lane
__device__ __forceinline__ void mid_piece(const __amdgpu_buffer_rsrc_t r, char* dst, uint32_t off, uint32_t k) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, off, k, 0, 0);
}
// Block b's tile (its feature tile and its token tile; false: none).  The dispatcher places block b on XCD b % 8 (a speed assumption only): XCD x works on
// feature run x % 2^lf and token run x >> lf, features fastest, so that its L2 fetches 1 / 2^lf of the weights and 2^lf / 8 of the activations.
__device__ __forceinline__ bool mid_tile(uint32_t b, uint32_t tiles_f, uint32_t tiles_t, int lf, uint32_t& f, uint32_t& t) {
  const uint32_t run_f = tiles_f >> lf, n = run_f * tiles_t, each = ((n << lf) + 7) >> 3;
  const uint32_t i = ((b & 7) >> lf) * each + (b >> 3);
  t = i / run_f;  // (one division: each is some 40 dependent instructions in front of the first request)
  f = i - t * run_f + (b & ((1u << lf) - 1)) * run_f;
  return (b >> 3) < each && i < n;
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
  const uint32_t k0 = EPI == TEPI_PARTIAL ? blockIdx.y * (uint32_t)KT * (BK * 2) : 0;  // bytes of a row in front of this slice of K
  int n0 = 0, m0 = 0, m_end = a.M;
  int64_t wrow0 = 0;
  if constexpr (EPI == TEPI_ANY) {
    const int ntiles = any_tiles(a);
    if ((int)blockIdx.x >= ntiles) return;  // (the grid is the host's bound on the grouped tiles)
    const AnyTile t = any_tile(a, (int)blockIdx.x, ntiles, SH::T, ARGS::kDual ? SH::F / 2 : SH::F);
    n0 = t.n0, m0 = t.m0, m_end = t.m_end, wrow0 = (int64_t)t.group * a.w_rows;
  } else {
    uint32_t f, t;
    if (!mid_tile(blockIdx.x, a.tiles_f, a.tiles_t, a.xcd_lf, f, t)) return;
    n0 = f * SH::F, m0 = t * SH::T;
  }

  // LDS-DMA: wave w moves its share of the 1 KiB pieces (8 local rows each) of the feature rows and of the token rows.  A piece's source is a 32-bit
  // offset per lane from the operand's base (the entry points refuse operands beyond 2 GiB) and the K step on the scalar unit.
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.w), 0, 0x80000000u, 0x00020000);
  const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.x), 0, 0x80000000u, 0x00020000);
  const uint16_t* w2 = a.w;
  if constexpr (ARGS::kDual) w2 = a.w2;
  const __amdgpu_buffer_rsrc_t w2_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w2), 0, 0x80000000u, 0x00020000);
  uint32_t offA[SH::A_PIECES], offB[SH::B_PIECES];
#pragma unroll
  for (int i = 0; i < SH::A_PIECES; ++i) {
    const int lr = (wave * SH::A_PIECES + i) * 8 + (lane >> 3), c = (lane & 7) ^ swizzle(lr);
    int64_t rowA = 0;
    if constexpr (EPI == TEPI_ANY)
      // two weights: every wave's first fragment holds 32 rows of w, its second the rows of w2 that pair with them
      rowA = wrow0 + min(ARGS::kDual ? n0 + (lr >> 6) * 32 + (lr & 31) : n0 + lr, a.N - 1);
    else
      rowA = min(mid_weight_row(lr, n0, a.N, EPI == TEPI_SILU), a.N - 1);
    offA[i] = (uint32_t)((rowA * a.K + c * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < SH::B_PIECES; ++i) {
    const int lr = (wave * SH::B_PIECES + i) * 8 + (lane >> 3), c = (lane & 7) ^ swizzle(lr);
    int64_t rowB = min(m0 + lr, m_end - 1);
    if constexpr (EPI == TEPI_ANY)
      if (ARGS::kGather) rowB = a.x_rows[rowB];
    offB[i] = (uint32_t)((rowB * a.ldx + c * 8) * 2);
  }
  constexpr int PIECES = SH::A_PIECES + SH::B_PIECES;
  auto piece = [&](int kt, int p, int i) __attribute__((always_inline)) {  // the i-th of this wave's pieces of step kt, into ring slot p
    const uint32_t k = k0 + (uint32_t)kt * (BK * 2);
    char* const image = lds + p * SH::STAGE;
    if (i < SH::A_PIECES) {
      const int q = wave * SH::A_PIECES + i;
      const uint32_t off = offA[i < SH::A_PIECES ? i : 0];
      if constexpr (EPI == TEPI_ANY && ARGS::kDual)
        if ((q >> 2) & 1) {
          mid_piece(w2_rsrc, image + q * 1024, off, k);
          return;
        }
      mid_piece(w_rsrc, image + q * 1024, off, k);
    } else {
      const int q = wave * SH::B_PIECES + i - SH::A_PIECES;
      mid_piece(x_rsrc, image + SH::F * 128 + q * 1024, offB[i < SH::A_PIECES ? 0 : i - SH::A_PIECES], k);
    }
  };
  auto issue = [&](int kt, int p) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) piece(kt, p, i);
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
  for (int s = 0; s < NST; ++s)
    if (s < KT) issue(s, s);
  struct Frags {
    u32x4 A[WF][4], B[WT][4];
  } fa, fb;
  constexpr int READS = 4 * (WF + WT), MULS = 4 * WF * WT;
  auto read = [&](int p, int i, Frags& f) __attribute__((always_inline)) {  // the i-th fragment of the step in ring slot p, k ascending
    const int kk = i / (WF + WT), r = i % (WF + WT);
    if (r < WF) f.A[r < WF ? r : 0][kk] = *reinterpret_cast<const u32x4*>(lds + p * SH::STAGE + (fw * WF + r) * 4096 + kx[kk]);
    else f.B[r < WF ? 0 : r - WF][kk] = *reinterpret_cast<const u32x4*>(lds + p * SH::STAGE + SH::F * 128 + (tw * WT + r - WF) * 4096 + kx[kk]);
  };
  auto multiply = [&](int i, const Frags& f) __attribute__((always_inline)) {  // the i-th matrix instruction of a step, k ascending
    const int kk = i / (WF * WT), u = i / WT % WF, b = i % WT;
    acc[u][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(f.A[u][kk]), as_frag(f.B[b][kk]), acc[u][b], 0, 0, 0);
  };
  int p = 0;  // ring slot of step kt
  // Step kt, which is not the last one: its fragments are in `cur`; behind its matrix instructions the reads of step kt + 1 into `next` (two each: in
  // front of the first one it would wait for them) and the requests of step kt + NST, one each (all at once they hold the wave up for as long as its
  // matrix instructions take) - REST: near the end, where there may be none.
  auto step = [&](auto rest, int kt, const Frags& cur, Frags& next) __attribute__((always_inline)) {
    constexpr bool REST = decltype(rest)::value;
    // requested so far: steps <= kt + NST - 1; the same number of pieces per step and wave, completing in order
    mid_wait<NST - 2, PIECES>(REST ? min(KT - 2 - kt, NST - 2) : NST - 2);
    __builtin_amdgcn_sched_barrier(0);
    const int free = p;  // (everybody has read step kt)
    p = p + 1 == NST ? 0 : p + 1;
    if (REST && kt + NST < KT) issue(kt + NST, free);
    constexpr int RD = MULS < READS ? (READS + MULS / 2 - 1) / (MULS / 2) : 2, DM = (PIECES + MULS - 1) / MULS;
#pragma unroll
    for (int i = 0; i < MULS; ++i) {
      multiply(i, cur);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
      for (int j = 0; j < RD; ++j)
        if (i * RD + j < READS) {
          read(p, i * RD + j, next);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
      if constexpr (!REST)
#pragma unroll
        for (int j = 0; j < DM; ++j)
          if (i * DM + j < PIECES) {
            piece(kt + NST, free, i * DM + j);
            __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
          }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  mid_wait<NST - 1, PIECES>(min(KT - 1, NST - 1));
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < READS; ++i) read(0, i, fa);
  int kt = 0;
  for (; kt + 1 + NST < KT; kt += 2) {
    step(std::false_type{}, kt, fa, fb);
    step(std::false_type{}, kt + 1, fb, fa);
  }
  for (; kt + 2 < KT; kt += 2) {
    step(std::true_type{}, kt, fa, fb);
    step(std::true_type{}, kt + 1, fb, fa);
  }
  if (kt + 1 < KT) {
    step(std::true_type{}, kt, fa, fb);
#pragma unroll
    for (int i = 0; i < MULS; ++i) multiply(i, fb);
  } else {
#pragma unroll
    for (int i = 0; i < MULS; ++i) multiply(i, fa);
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

