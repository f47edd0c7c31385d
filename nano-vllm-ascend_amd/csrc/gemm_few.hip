// A decode step of a few rows: the projections with the launch in front of them in their operand load.
//
// A step of one row is nothing but launches: 31 us a layer for 31.5 MB of weights (5 us at what the memory delivers), and three of its
// eight launches - two add+RMSNorm and the merge of the attention's context splits - handle a few KiB, 2.3 to 3.6 us each plus the
// boundary.  With few rows those KiB are cheap enough for every workgroup of the NEXT launch to handle for itself:
//
//   gemm_norm_few_kernel   sums the previous projection's fp32 K-slice sums, adds the residual, norms (18 bytes per element and row from
//                          the L2s), multiplies - qkv, and gate_up with SwiGLU
//   gemm_merge_few_kernel  weighs the attention's splits (a wave: its own 64 channels, its head's weights), multiplies - o_proj
//
// The weights are asked for before the operand's arithmetic, which runs under their round trip.  The same arithmetic in the same order as mi_add_rmsnorm_splitk / the merge of mi_paged_attn_decode_fused followed by gemm_skinny_kernel: the same bits, so a row does not
// depend on how many are in the batch.
//
// A step of Qwen3-0.6B (28 layers, captured; keys 128 / 1500), us: all launches | the norms here | the merge too
//   1 row   872 / 912 | 822 / 870 | 747 / 758      2 rows  869 / 946 | 830 / 893 | 762 / 783
//   3 rows  882 / 955 | 841 / 891 | 812 / 828      4 rows  875 / 977 | 817 / 929 | 777 / 837
// Five rows took a second pass over the rows and lost (892 / 1014 | 914 / 1040 | 909 / 1013; 8 rows 900 / 1127 | 916 / 1137 | 956 / 1156):
// every workgroup repeats the norm, and at 18 bytes per element and row the repeats come through each CU's L1.  Hence kFewRows.
// The operand is asked for before the weights: loads come back in order, and behind 12 MB of weights it waits for all of them (1 row
// 760 / 773).
#include "gemm_skinny_kernel.hpp"

namespace mi {

constexpr int kFewRows = 4;

// B fragments of a [rows][64 per wave] bf16 image in LDS, 16-byte chunks XOR-swizzled by the row (rows at one chunk: other bank groups)
__device__ __forceinline__ int few_chunk(int row, int chunk) { return (chunk & ~7) | ((chunk ^ row) & 7); }

// the weights of a wave's K slice of 64, RT row tiles
template <int RT, int WF>
struct FewWeights {
  u32x4 v[RT][WF == 2 ? 1 : 2];
  __device__ __forceinline__ void load(const uint16_t* w, const int (&tile)[RT], int K, int kbeg, int lane) {
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int s = 0; s < (WF == 2 ? 1 : 2); ++s)
        v[t][s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(
            WF == 2 ? w + (((int64_t)tile[t] * (K >> 6) + (kbeg >> 6)) * 1024 + lane * 16) / 2
                    : w + ((int64_t)tile[t] * (K >> 5) + (kbeg >> 5) + s) * 512 + lane * 8));
  }
  __device__ __forceinline__ bf16x8 frag(int t, int s) const {
    if constexpr (WF == 2) {
      const uint32_t lo = v[t][0][2 * s], hi = v[t][0][2 * s + 1];
      const auto f0 = __builtin_amdgcn_cvt_pk_f32_fp8(lo, false), f1 = __builtin_amdgcn_cvt_pk_f32_fp8(lo, true);
      const auto f2 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, false), f3 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, true);
      return as_frag(u32x4{pack_bf(f0[0], f0[1]), pack_bf(f1[0], f1[1]), pack_bf(f2[0], f2[1]), pack_bf(f3[0], f3[1])});
    } else {
      return as_frag(v[t][s]);
    }
  }
};

// WAVES: K / 64; K / 256 waves take a row
template <int WAVES, int PART, int WF, bool SILU>
__global__ __launch_bounds__(WAVES * 64) void gemm_norm_few_kernel(const float* __restrict__ part, const uint16_t* __restrict__ residual,
                                                                   const uint16_t* __restrict__ norm_w, float eps,
                                                                   const uint16_t* __restrict__ w, const float* __restrict__ scale,
                                                                   uint16_t* __restrict__ y, uint16_t* __restrict__ residual_out, int M,
                                                                   int N) {
#pragma clang fp contract(off)  // (the norm's separate roundings; the products are matrix instructions)
  constexpr int K = WAVES * 64, RT = SILU ? 2 : 1, RW = WAVES / kFewRows;
  static_assert(WAVES % kFewRows == 0, "all rows at a time");
  __shared__ __attribute__((aligned(16))) uint16_t xs[kFewRows][K];
  __shared__ __attribute__((aligned(16))) float red[WAVES][RT][64][4];
  __shared__ float row_ss[kFewRows][RW];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int row = wave / RW, vec = (wave % RW) * 64 + lane;  // four columns
  const int lrow = min(row, M - 1);
  f32x4 p[PART];
#pragma unroll
  for (int sp = 0; sp < PART; ++sp) p[sp] = *reinterpret_cast<const f32x4*>(part + ((int64_t)sp * M + lrow) * K + vec * 4);
  const u32x2 rr = *reinterpret_cast<const u32x2*>(residual + (int64_t)lrow * K + vec * 4);
  const u32x2 wr = *reinterpret_cast<const u32x2*>(norm_w + vec * 4);
  __builtin_amdgcn_sched_barrier(0);  // (loads come back in order: the weights behind what is needed first)
  int tile[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) tile[t] = (int)blockIdx.x + t * (N >> 5);
  FewWeights<RT, WF> a;
  a.load(w, tile, K, wave * 64, lane);
  __builtin_amdgcn_sched_barrier(0);

  f32x4 s = p[0];
#pragma unroll
  for (int sp = 1; sp < PART; ++sp) s += p[sp];
  const u32x2 raw = {pack_bf(s[0], s[1]), pack_bf(s[2], s[3])};
  float v[4];
  u32x2 ro;
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    v[2 * j] = lo_bf(raw[j]) + lo_bf(rr[j]);
    v[2 * j + 1] = hi_bf(raw[j]) + hi_bf(rr[j]);
    ro[j] = pack_bf(v[2 * j], v[2 * j + 1]);
    ss += v[2 * j] * v[2 * j];
    ss += v[2 * j + 1] * v[2 * j + 1];
  }
  ss = wave_sum_up(ss);
  if (lane == 0) row_ss[row][wave % RW] = ss;
  __syncthreads();
  float tot = row_ss[row][0];
#pragma unroll
  for (int i = 1; i < RW; ++i) tot += row_ss[row][i];
  const float rs = 1.0f / sqrtf(tot / (float)K + eps);
  u32x2 n;
#pragma unroll
  for (int j = 0; j < 2; ++j) n[j] = pack_bf(rbf(v[2 * j] * rs) * lo_bf(wr[j]), rbf(v[2 * j + 1] * rs) * hi_bf(wr[j]));
  *reinterpret_cast<u32x2*>(&xs[row][few_chunk(row, vec >> 1) * 8 + (vec & 1) * 4]) = n;
  __syncthreads();
  f32x4 acc[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int xrow = min(r, M - 1);  // (columns beyond M: copies, not stored)
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const bf16x8 b = as_frag(*reinterpret_cast<const u32x4*>(&xs[xrow][few_chunk(xrow, wave * 8 + s * 4 + g) * 8]));
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.frag(t, s), b, acc[t], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < RT; ++t) *reinterpret_cast<f32x4*>(red[wave][t][lane]) = acc[t];
  if (blockIdx.x == 0 && row < M) *reinterpret_cast<u32x2*>(residual_out + (int64_t)row * K + vec * 4) = ro;
  __syncthreads();
  if (wave > 0 || r >= M) return;
  f32x4 sum[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    sum[t] = *reinterpret_cast<const f32x4*>(red[0][t][lane]);
#pragma unroll
    for (int i = 1; i < WAVES; ++i) sum[t] += *reinterpret_cast<const f32x4*>(red[i][t][lane]);
    if constexpr (WF == 2) sum[t] *= *reinterpret_cast<const f32x4*>(scale + tile[t] * 16 + 4 * g);
  }
  float o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[i] = sum[0][i];
    if constexpr (SILU) {
      const float gb = rbf(sum[0][i]);
      const float sb = rbf(gb / (1.0f + expf(-gb)));
      o[i] = sb * rbf(sum[RT - 1][i]);
    }
  }
  *reinterpret_cast<u32x2*>(y + (int64_t)r * (SILU ? N >> 1 : N) + blockIdx.x * 16 + 4 * g) = u32x2{pack_bf(o[0], o[1]), pack_bf(o[2], o[3])};
}

// WAVES: K / (64 gridDim.y).  SP, MB: splits and rows, rounded up.  part_o / part_ml: the attention's workspace (16 splits per row, heads of 128)
template <int WAVES, int SP, int WF, int MB>
__global__ __launch_bounds__(WAVES * 64) void gemm_merge_few_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                                    int splits, const uint16_t* __restrict__ w,
                                                                    const float* __restrict__ scale, float* __restrict__ part, int M, int N,
                                                                    int K) {
  __shared__ __attribute__((aligned(16))) uint16_t xs[WAVES][kFewRows][64];
  __shared__ __attribute__((aligned(16))) float red[WAVES][64][4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int kbeg = ((int)blockIdx.y * WAVES + wave) * 64;
  const int heads = K >> 7, head = kbeg >> 7, d = (kbeg & 64) + lane;
  float ov[MB][SP];  // (of splits without keys: whatever is there, not used)
  float2 ml[MB];
#pragma unroll
  for (int row = 0; row < MB; ++row) {
    const int64_t at = ((int64_t)min(row, M - 1) * heads + head) * 16;
    ml[row] = *reinterpret_cast<const float2*>(part_ml + (at + min(lane, splits - 1)) * 2);
#pragma unroll
    for (int s = 0; s < SP; ++s) ov[row][s] = part_o[(at + min(s, splits - 1)) * 128 + d];
  }
  __builtin_amdgcn_sched_barrier(0);  // (loads come back in order: the weights behind what is needed first)
  const int tile[1] = {(int)blockIdx.x};
  FewWeights<1, WF> a;
  a.load(w, tile, K, kbeg, lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int row = 0; row < MB; ++row) {
    const float ms = lane < splits ? ml[row].x : -INFINITY;
    const float mx = wave_max(ms);
    const float e = ms != -INFINITY ? exp2f(ms - mx) : 0.f;
    const float den = wave_sum(e * (lane < splits ? ml[row].y : 0.f));
    float acc = 0.f;
#pragma unroll
    for (int s = 0; s < SP; ++s) {
      const float es = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e), s));  // (lanes from `splits` on: 0)
      if (es != 0.f) acc = fmaf(es, ov[row][s], acc);
    }
    const float inv = den > 0.f ? 1.0f / den : 0.f;
    xs[wave][row][few_chunk(row, lane >> 3) * 8 + (lane & 7)] = f2bf(acc * inv);
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const int xrow = min(r, M - 1);
#pragma unroll
  for (int s = 0; s < 2; ++s)  // (the wave's own image: its LDS operations are in order)
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.frag(0, s), as_frag(*reinterpret_cast<const u32x4*>(&xs[wave][xrow][few_chunk(xrow, s * 4 + g) * 8])),
                                                  acc, 0, 0, 0);
  *reinterpret_cast<f32x4*>(red[wave][lane]) = acc;
  __syncthreads();
  if (wave > 0 || r >= M) return;
  f32x4 sum = *reinterpret_cast<const f32x4*>(red[0][lane]);
#pragma unroll
  for (int i = 1; i < WAVES; ++i) sum += *reinterpret_cast<const f32x4*>(red[i][lane]);
  if constexpr (WF == 2) sum *= *reinterpret_cast<const f32x4*>(scale + tile[0] * 16 + 4 * g);
  *reinterpret_cast<f32x4*>(part + ((int64_t)blockIdx.y * M + r) * N + blockIdx.x * 16 + 4 * g) = sum;
}

}  // namespace mi

using namespace mi;

extern "C" int mi_few_rows_max(void) { return kFewRows; }

extern "C" int mi_gemm_norm_few(const float* partials, int nsplit, const mi_bf16* residual, const mi_bf16* norm_w, float eps, const void* w_packed,
                                const float* scale, mi_bf16* y, mi_bf16* residual_out, int M, int N, int K, int epilogue, mi_stream stream) {
  if (!partials || !residual || !norm_w || !w_packed || !y || !residual_out || residual_out == residual || M < 0 || N <= 0 || K <= 0)
    return MI_EINVAL;
  if (epilogue != 0 && epilogue != 1) return MI_EINVAL;
  if (!aligned16(partials) || !aligned16(residual) || !aligned16(norm_w) || !aligned16(w_packed) || !aligned16(y) || !aligned16(residual_out) ||
      !aligned16(scale))
    return MI_EINVAL;
  const bool silu = epilogue == 1;
  if (M > kFewRows || (K != 512 && K != 768 && K != 1024) || nsplit < 1 || N % (silu ? 32 : 16)) return MI_EUNSUPPORTED;
  if (N / (silu ? 32 : 16) >= 2048) return MI_EUNSUPPORTED;  // (gemm_skinny_kernel sums those in other slices)
  if (M == 0) return MI_OK;
  const dim3 grid(N / (silu ? 32 : 16));
  const auto* wp = static_cast<const uint16_t*>(w_packed);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(K), 0, S(stream), partials, residual, norm_w, eps, wp, scale, y, residual_out, M, N);
    return check_launch();
  };
  auto by_form = [&](auto waves, auto parts) {
    constexpr int W = decltype(waves)::value, P = decltype(parts)::value;
    if (scale) return silu ? go(gemm_norm_few_kernel<W, P, 2, true>) : go(gemm_norm_few_kernel<W, P, 2, false>);
    return silu ? go(gemm_norm_few_kernel<W, P, 1, true>) : go(gemm_norm_few_kernel<W, P, 1, false>);
  };
  using std::integral_constant;
  auto by_parts = [&](auto waves) {
    switch (nsplit) {
      case 2: return by_form(waves, integral_constant<int, 2>{});
      case 4: return by_form(waves, integral_constant<int, 4>{});
      case 8: return by_form(waves, integral_constant<int, 8>{});
      default: return (int)MI_EUNSUPPORTED;
    }
  };
  if (K == 512) return by_parts(integral_constant<int, 8>{});
  if (K == 768) return by_parts(integral_constant<int, 12>{});
  return by_parts(integral_constant<int, 16>{});
}

extern "C" int mi_gemm_merge_few_splitk(const void* workspace, int splits, const void* w_packed, const float* scale, float* partials, int M, int N,
                                        int K, int ksplit, mi_stream stream) {
  if (!workspace || !w_packed || !partials || M < 0 || N <= 0 || K <= 0 || splits < 1 || splits > 16) return MI_EINVAL;
  if (!aligned16(workspace) || !aligned16(w_packed) || !aligned16(partials) || !aligned16(scale)) return MI_EINVAL;
  if (M > kFewRows || N % 16 || K % 128 || ksplit < 1 || ksplit > 16 || K % (64 * ksplit)) return MI_EUNSUPPORTED;
  const int waves = K / (64 * ksplit);
  if ((waves != 4 && waves != 8 && waves != 12 && waves != 16) || (int64_t)N / 16 * ksplit >= 2048) return MI_EUNSUPPORTED;
  if (M == 0) return MI_OK;
  const float* part_o = static_cast<const float*>(workspace);
  const float* part_ml = part_o + (size_t)M * (K / 128) * 16 * 128;
  const auto* wp = static_cast<const uint16_t*>(w_packed);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(N / 16, ksplit), dim3(waves * 64), 0, S(stream), part_o, part_ml, splits, wp, scale, partials, M, N, K);
    return check_launch();
  };
  using std::integral_constant;
  auto by_rows = [&](auto w, auto sp, auto wf) {
    constexpr int W = decltype(w)::value, SP = decltype(sp)::value, WF = decltype(wf)::value;
    return M == 1 ? go(gemm_merge_few_kernel<W, SP, WF, 1>) : M == 2 ? go(gemm_merge_few_kernel<W, SP, WF, 2>) : go(gemm_merge_few_kernel<W, SP, WF, 4>);
  };
  auto by_splits = [&](auto w, auto wf) {
    if (splits <= 4) return by_rows(w, integral_constant<int, 4>{}, wf);
    return splits <= 8 ? by_rows(w, integral_constant<int, 8>{}, wf) : by_rows(w, integral_constant<int, 16>{}, wf);
  };
  auto by_form = [&](auto w) { return scale ? by_splits(w, integral_constant<int, 2>{}) : by_splits(w, integral_constant<int, 1>{}); };
  if (waves == 4) return by_form(integral_constant<int, 4>{});
  if (waves == 8) return by_form(integral_constant<int, 8>{});
  if (waves == 12) return by_form(integral_constant<int, 12>{});
  return by_form(integral_constant<int, 16>{});
}
