// True 32-bit products on the bf16 matrix instructions.  Included by gemm_any.hip (GemmAnyArgs, finish, group_tile).
#pragma once
#include <cfloat>

namespace mi {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

// Operands are split times 2^24, and sums leave times 2^-48: the last bit of the smallest number, 2^-149, is then above the smallest normal number, so
// that no part of any operand is lost or subnormal, and a sum reaches below what fp32 holds.
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;

// Eight numbers, times kSplitScale, as three bf16 parts, each the nearest to what the parts before it leave: h + m + l exactly (8 + 8 + 8 bits; the
// rests are floats).  (The rests by the two-term dot product, one instruction in place of two: the same time.)
struct SplitParts {
  u32x4 part[3];
};
__device__ __forceinline__ SplitParts split_parts(const f32x4& a, const f32x4& b) {
  SplitParts p;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float u = kSplitScale * (i < 2 ? a[2 * i] : b[2 * i - 4]), v = kSplitScale * (i < 2 ? a[2 * i + 1] : b[2 * i - 3]);
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      p.part[s][i] = pack_bf(u, v);
      u -= lo_bf(p.part[s][i]), v -= hi_bf(p.part[s][i]);
    }
  }
  return p;
}

// 64 x 64 tiles, four waves with 2 x 2 fragments of 16 x 16 each (two weights: of each), K in steps of 32.  A step's operands travel memory -> registers (two
// steps ahead) -> three bf16 parts -> LDS (two images, one barrier a step), each number split once per workgroup; all products of parts but l l on
// v_mfma_f32_16x16x32_bf16, h h in one sum and the seven others, smallest first, in another.  Left out: below 2^-34 of |x w|, so that a sum of one product is
// rounded as fp32 arithmetic rounds it (without m l and l m, which reach 2^-24 together, up to 0.95 of a last bit).  A step of 32 k is rounded
// once into each sum where the fp32 matrix instruction rounds eight times: error against 64 bits (2-norm) 1.9e-7 at K = 1024 and 4.0e-7 at 4096, the fp32
// instruction's (gemm_any_f32_kernel) 5.7e-7 and 1.15e-6.
// What bounds it: the fp32 matrix rate is 1/16 of the bf16 one, so eight products are half of its time; the split (thirteen vector instructions for
// two numbers) and the LDS (24 KB written and 48 KB read per step) take about as long as the products beside them, and the clock falls with the matrix
// pipe's load.  The matrix instructions stand among the next step's split (one tile alone on its CU, of six products, 34.7 -> 27.9 us, 721 x 1024 x 1024).
// us with cold weights, gemm_any_f32_kernel / here: 4096 x 4096 x 4096 1127 / 970-1010, 1500 x 4096 x 2048 237 / 200, 721 x 3072 x 1024 61 / 57; 11324 pairs of
// 32 experts, 1024 -> 2 x 512, 276 / 241.  Steps of four layers without / with it: width 1024, 1327 rows 1840 / 1760, 2831 rows 3237 / 2890; width 2048, 2831 rows
// 12400 / 11210.  128-row tiles were 8 % faster at 4096 x 4096 x 4096 and lose with their fewer tiles below it and with uneven groups (a step of 721
// rows 1311 us, 1337 with 128 x 32 of two weights, 1347 with 48 x 64; all with six products).
// An infinity has no finite rest, a number of 2^104 and more times 2^24 is one, and so may a sum of 2^80 and more be: a wave with an output
// that is not finite sums its outputs once more on the fp32 matrix instruction, and takes from there those that were not finite and no other (an output is a
// function of its own row of x and of the weights).  us, no / one / forty rows with a NaN: 2831 x 1024 x 1024 56 / 69 / 78, 2048 x 2048 x 2048 with two
// weights 233 / 273 / 343 (gemm_any_f32_kernel 69 and 321 whatever the numbers are).
// Rows beyond the group's end and features beyond N are read from the last valid one and not stored.  Needs what gemm_any_f32_kernel needs.
// GROUPS: a workgroup finds its tiles, every gridDim.y-th row tile of all groups.
template <bool DUAL, bool EXT, bool GROUPS>
__global__ __launch_bounds__(256, 2) void gemm_any_split_kernel(GemmAnyArgs a) {
  constexpr int FM = 2, FN = 2, WM = 2, WN = 2, BM = 16 * FM * WM, BN = 16 * FN * WN, BK = 32, ND = DUAL ? 2 : 1;
  constexpr int FRAGS = BM / 16 + ND * BN / 16, PLANE = FRAGS * 1024, STAGE = 3 * PLANE, U = FRAGS / 4;
  __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * BN, KT = a.K / BK;
  const int wm = wave / WN * FM, wn = wave % WN * FN;   // the wave's first fragment of rows, of features
  const int r16 = lane & 15, kg = lane >> 4;
  for (int tile = blockIdx.y;; tile += gridDim.y) {
    int m0 = tile * BM, m_hi = a.M;
    const float *x = a.x, *w = static_cast<const float*>(a.w), *w2 = static_cast<const float*>(a.w2);
    float* y = a.y;
    if constexpr (GROUPS) {
      int g;
      if (!group_tile<BM>(a.group_offsets, a.n_groups, tile, g, m0, m_hi)) return;
      w += (int64_t)g * a.N * a.K;
      if (DUAL) w2 += (int64_t)g * a.N * a.K;
    } else {
      x += (int64_t)blockIdx.z * a.x_batch;
      y += (int64_t)blockIdx.z * a.y_batch;
      if (a.gate) a.gate += (int64_t)blockIdx.z * a.gate_batch;
      w += (int64_t)blockIdx.z * a.N * a.K;
      if (DUAL) w2 += (int64_t)blockIdx.z * a.N * a.K;
    }
    // A wave's u-th fragment of the tile's operands is number 4 u + wave: 16 rows of x, then of w, then of w2; four lanes a row, lane c of them k = 4 c ..
    // and 16 + 4 c .. of the step.  In LDS a part of a fragment is 64 pieces of 16 bytes in the order in which the matrix instruction's lanes
    // take them, the rows XOR-ed with 2 c (eight lanes at a time write to eight different bank groups).
    const float* src[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int f = u * 4 + wave, r = lane >> 2, c = lane & 3;
      if (f < BM / 16) {
        const int m = min(m0 + f * 16 + r, m_hi - 1);
        src[u] = x + (a.x_rows ? a.x_rows[m] : m) * a.ldx + c * 4;
      } else {
        const int q = f - BM / 16, d = q / (BN / 16);
        src[u] = (DUAL && d ? w2 : w) + (int64_t)min(n0 + (q - d * (BN / 16)) * 16 + r, a.N - 1) * a.K + c * 4;
      }
    }
    const int to = wave * 1024 + (lane & 3) * 256 + (((lane >> 2) ^ (2 * (lane & 3))) << 4);
    const int from = kg * 256 + ((r16 ^ (2 * kg)) << 4);
    struct Raw {
      f32x4 v[U][2];
    } ra, rb;
    auto request = [&](int kt, Raw& r) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        r.v[u][0] = *reinterpret_cast<const f32x4*>(src[u] + kt * BK);
        r.v[u][1] = *reinterpret_cast<const f32x4*>(src[u] + kt * BK + 16);
      }
    };
    auto put = [&](const Raw& r, int image) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const SplitParts p = split_parts(r.v[u][0], r.v[u][1]);
#pragma unroll
        for (int s = 0; s < 3; ++s) *reinterpret_cast<u32x4*>(lds + image * STAGE + s * PLANE + u * 4096 + to) = p.part[s];
      }
    };
    f32x4 acc[ND][FM][FN], low[ND][FM][FN];
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[d][i][j] = low[d][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    struct Parts {
      u32x4 x[3][FM], w[3][ND][FN];
    };
    auto read = [&](int image, Parts& p) __attribute__((always_inline)) {
      const char* at = lds + image * STAGE + from;
#pragma unroll
      for (int s = 2; s >= 0; --s) {
#pragma unroll
        for (int i = 0; i < FM; ++i) p.x[s][i] = *reinterpret_cast<const u32x4*>(at + s * PLANE + (wm + i) * 1024);
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int j = 0; j < FN; ++j) p.w[s][d][j] = *reinterpret_cast<const u32x4*>(at + s * PLANE + (BM / 16 + d * (BN / 16) + wn + j) * 1024);
      }
    };
    auto multiply = [&](const Parts& p) __attribute__((always_inline)) {
      const auto all = [&](int sw, int sx, auto& sum) __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int i = 0; i < FM; ++i)
              sum[d][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, p.w[sw][d][j]), __builtin_bit_cast(bf16x8, p.x[sx][i]),
                                                                     sum[d][i][j], 0, 0, 0);
      };
      all(2, 1, low), all(1, 2, low), all(2, 0, low), all(0, 2, low), all(1, 1, low), all(1, 0, low), all(0, 1, low), all(0, 0, acc);
    };
    request(0, ra);
    if (1 < KT) request(1, rb);
    put(ra, 0);  // (behind the barrier of the tile before: it is read)
    if (2 < KT) request(2, ra);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // step kt: its parts from image kt & 1; step kt + 1 (in `next`) into the other image; step kt + 3 asked for
    auto step = [&](auto inside, int kt, Raw& next) __attribute__((always_inline)) {
      Parts p;
      read(kt & 1, p);
      constexpr bool INSIDE = decltype(inside)::value;
      if (INSIDE || kt + 1 < KT) put(next, (kt + 1) & 1);
      if (INSIDE || kt + 3 < KT) request(kt + 3, next);
      multiply(p);
      // reads, some of the split in their shadow, then its rest and its LDS writes among the matrix instructions
      constexpr int MULS = 8 * ND * FM * FN, VALU = U * 52, EACH = MULS / (3 * U);
      __builtin_amdgcn_sched_group_barrier(0x100, 3 * (FM + ND * FN), 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);
#pragma unroll
      for (int i = 0; i < MULS; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (VALU - 16 + MULS - 1) / MULS, 0);
        if (i % EACH == EACH - 1) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    int kt = 0;
    for (; kt + 4 < KT; kt += 2) {
      step(std::true_type{}, kt, rb);
      step(std::true_type{}, kt + 1, ra);
    }
    for (; kt + 1 < KT; kt += 2) {
      step(std::false_type{}, kt, rb);
      step(std::false_type{}, kt + 1, ra);
    }
    if (kt < KT) step(std::false_type{}, kt, rb);
    bool finite = true;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          acc[d][i][j] = (acc[d][i][j] + low[d][i][j]) * kSplitUnscale;
#pragma unroll
          for (int r = 0; r < 4; ++r) finite &= fabsf(acc[d][i][j][r]) <= FLT_MAX;
        }
    if (__builtin_expect(__any(!finite), 0)) {
      // the wave's outputs on the fp32 matrix instruction, k in gemm_any_f32_kernel's order; each that was not finite, and only those, from here
      const float *xr[FM], *wr[ND][FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int m = min(m0 + (wm + i) * 16 + r16, m_hi - 1);
        xr[i] = x + (a.x_rows ? a.x_rows[m] : m) * a.ldx + kg * 4;
      }
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int j = 0; j < FN; ++j) wr[d][j] = (DUAL && d ? w2 : w) + (int64_t)min(n0 + (wn + j) * 16 + r16, a.N - 1) * a.K + kg * 4;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) low[d][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int k = 0; k < a.K; k += BK) {
        f32x4 xf[2][FM], wf[2][ND][FN];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int i = 0; i < FM; ++i) xf[h][i] = *reinterpret_cast<const f32x4*>(xr[i] + k + h * 16);
#pragma unroll
          for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int j = 0; j < FN; ++j) wf[h][d][j] = *reinterpret_cast<const f32x4*>(wr[d][j] + k + h * 16);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int d = 0; d < ND; ++d)
#pragma unroll
              for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                  low[d][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[h][d][j][e], xf[h][i][e], low[d][i][j], 0, 0, 0);
      }
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[d][i][j][r] = fabsf(acc[d][i][j][r]) <= FLT_MAX ? acc[d][i][j][r] : low[d][i][j][r];
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = m0 + (wm + i) * 16 + r16;
      if (m >= m_hi) continue;
      const int64_t yrow = a.y_rows ? a.y_rows[m] : m;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int n = n0 + (wn + j) * 16 + kg * 4;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = n + r < a.N ? finish<DUAL, EXT>(a, m, yrow, n + r, acc[0][i][j][r], acc[ND - 1][i][j][r]) : 0.f;
        float* yp = y + yrow * a.ldy + n;
        if (n + 4 <= a.N && a.ldy % 4 == 0 && dev_aligned16(y)) {
          *reinterpret_cast<float4*>(yp) = float4{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < a.N) yp[r] = v[r];
        }
      }
    }
    if constexpr (!GROUPS) return;
  }
}

}  // namespace mi
