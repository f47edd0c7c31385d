// The channel-wise gated delta rule over prompt portions, sixteen rows at a time on the fp32 matrix instruction
// (mi_channel_delta_blocks); short steps walk row by row (seqmix.hip: channel_delta_kernel).
//
//   S <- diag(g_t) S;   u_t = beta_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t
//
// Over a block of rows t = 0..15 behind the state S0, with P_t = g_0 .. g_t and P_jt = g_{j+1} .. g_t (products per key channel, all at
// most 1: nothing is divided by a decay, so nothing can overflow):
//   the decayed state read with k_t:  D_t = (k_t P_t)^T S0,   A_tj = sum_d k_t P_jt k_j  (j < t)
//   read with q_t:                    E_t = (q_t P_t)^T S0,   B_tj = sum_d q_t P_jt k_j  (j <= t)
//   u_t = beta_t (v_t - D_t - sum_j A_tj u_j)   =>   U = T (V - D),  T = (1 + diag(beta) A)^-1 diag(beta)   (16 x 16, lower triangular)
//   O = E + B U,      S <- diag(P_15) S0 + sum_j (k_j P_j15) u_j^T
// blocks_prepare_kernel (a workgroup per block and head, all blocks at once) leaves (k P), (q P), (k P_.15), P_15, B and T of a block as
// one record in MFMA operand order; blocks_walk_kernel (two waves per 16 value columns, S in their registers as MFMA accumulators, which
// are the next block's B operand as they stand) walks a sequence's records.
//
// What bounds it: the longest sequence's chain of blocks - 56 matrix instructions of 32 cycles a wave (128 channels), the LDS reads, sums and
// barriers between them -, and the matrix pipe where two workgroups share a CU, against 0.71 us per ROW of the row-by-row walk (LDS reads,
// cross-lane sums, plain FMAs).
// 8 sequences of 1024 rows, 8 heads, 128 x 128: 809 us row by row, 206 so (one wave for all channels 263).  The error against 64 bits is
// the row-by-row one's or less (rms of the results, 64 .. 1400 rows and decays from 0.05 to 1: 0.87 to 0.98 of it).  A NaN or an
// infinity in a row must not reach the rows in front of it through the zeros above the diagonals of T and B: see causal() below.
#include <type_traits>

#include "seqmix_common.hpp"

namespace mi {

constexpr int kB = 16;                     // rows of a block
constexpr int kStateCols = 32;             // value columns of a block of the state's memory layout (seqmix.hip: kDeltaCols)

// floats of a record, DP = 16 DT key channels: [k P: DP * 16][q P: DP * 16][k P_.15: DP * 16][B: 256][T: 256][P_15: DP], rounded up to
// whole KiB
constexpr int record_floats(int dp) { return (3 * dp * kB + 512 + dp + 255) & ~255; }

// First record of sequence s, whose rows begin at r0: r0 / 16 + s, at least as far from the next sequence's as it has blocks
// (ceil(n / 16) <= (r0 + n) / 16 - r0 / 16 + 1), so that no block has to add up the sequences before it.
__host__ __device__ constexpr int first_record(int r0, int s) { return r0 / kB + s; }

struct BlockArgs {
  const float* qkv;
  int64_t ld;
  int q_off, k_off, v_off;
  const float* beta_pre;   // [rows][H]
  int64_t ld_beta;
  const float* decay_pre;  // [rows][H * D]
  int64_t ld_decay;
  const float* dt_bias;    // [H * D]
  const float* a_log;      // [H]
  const int32_t* cu_q;
  const int32_t* kv_lens;
  const int32_t* slot_ids;
  int n_seqs, H, G, D, Dv;
  float* state;
  float* records;
  float* out;
  int64_t ldo;
};

__device__ __forceinline__ bool finite(float x) { return fabsf(x) < INFINITY; }
// the first of the block's rows whose value in this lane's column is not finite (kB: none)
__device__ __forceinline__ int first_bad(f32x4 b, int kg) {
  int first = kB;
#pragma unroll
  for (int r = 3; r >= 0; --r) first = finite(b[r]) ? first : 4 * kg + r;
  first = min(first, __shfl_xor(first, 16));
  return min(first, __shfl_xor(first, 32));
}
// y = L b of a lower triangular L, operands and result as the walk has them (a lane: rows 4 kg .. + 3 of its column), where the matrix
// instruction's zeros above L's diagonal met a b that is not finite: rows in front of the column's first such row are taken again with
// zeros from it on (their sums do not reach that far), the others stay what they are - the row-by-row walk's is not finite either.
__device__ __forceinline__ f32x4 causal(f32x4 l, f32x4 b, f32x4 y, int kg) {
  const int first = first_bad(b, kg);
  f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < 4; ++r) z = __builtin_amdgcn_mfma_f32_16x16x4f32(l[r], 4 * kg + r < first ? b[r] : 0.f, z, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 4; ++r) y[r] = 4 * kg + r < first ? z[r] : y[r];
  return y;
}
__device__ __forceinline__ f32x4 sum8(const f32x4 (&x)[8]) { return ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7])); }

template <int DT>
__global__ __launch_bounds__(256) void blocks_prepare_kernel(BlockArgs a) {
  constexpr int DP = 16 * DT, LD = DP + 4;   // (rows 16 bytes apart in their banks: sixteen of them are read at one channel group)
  __shared__ __attribute__((aligned(16))) float kk[kB][LD], qq[kB][LD], gg[kB][LD];
  __shared__ float am[kB][kB + 1], bm[kB][kB + 1], gamma[DP], beta[kB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = blockIdx.y;
  // the block's sequence: the last one whose records begin at or before it
  int s = -1;
  for (int i0 = 0; i0 < a.n_seqs; i0 += 64) {
    const int i = i0 + lane;
    const int found = __popcll(__ballot(i < a.n_seqs && first_record(a.cu_q[min(i, a.n_seqs - 1)], i) <= (int)blockIdx.x));
    s += found;
    if (found < 64) break;
  }
  s = __builtin_amdgcn_readfirstlane(s);
  const int r0 = a.cu_q[s] + ((int)blockIdx.x - first_record(a.cu_q[s], s)) * kB, n = min(kB, a.cu_q[s + 1] - r0);
  if (n <= 0) return;  // (a record that no block uses)
  // ---- the rows' q, k and decays; rows beyond the sequence's end change nothing: k = q = 0, g = 1, beta = 0 ----
  const int hq = h / (a.H / a.G);
  const float rate = expf(a.a_log[h]);
  constexpr int RW = kB / 4, C = DP / 64;
  float qv[RW][C], kv[RW][C], gv[RW][C], bv[RW];
#pragma unroll
  for (int i = 0; i < RW; ++i) {   // (every load first, at clamped places: none waits for another)
    const int64_t r = r0 + min(wave * RW + i, n - 1);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int d = min(lane + 64 * c, a.D - 1);
      qv[i][c] = a.qkv[r * a.ld + a.q_off + hq * a.D + d];
      kv[i][c] = a.qkv[r * a.ld + a.k_off + hq * a.D + d];
      gv[i][c] = a.decay_pre[r * a.ld_decay + h * a.D + d];
    }
    bv[i] = a.beta_pre[r * a.ld_beta + h];
  }
  float bias[C];
#pragma unroll
  for (int c = 0; c < C; ++c) bias[c] = a.dt_bias[h * a.D + min(lane + 64 * c, a.D - 1)];
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int t = wave * RW + i;
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const bool ok = t < n && lane + 64 * c < a.D;
      const float q = ok ? qv[i][c] : 0.f, k = ok ? kv[i][c] : 0.f;
      qv[i][c] = q, kv[i][c] = k;
      gg[t][lane + 64 * c] = ok ? expf(-rate * softplus_f(gv[i][c] + bias[c])) : 1.f;
      sq = fmaf(q, q, sq);
      sk = fmaf(k, k, sk);
    }
    const float nq = (1.f / sqrtf((float)a.D)) / sqrtf(wave_sum(sq) + 1e-6f), nk = 1.f / sqrtf(wave_sum(sk) + 1e-6f);
    if (lane == 0) beta[t] = t < n ? sigmoid_f(bv[i]) : 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) qq[t][lane + 64 * c] = qv[i][c] * nq, kk[t][lane + 64 * c] = kv[i][c] * nk;
  }
  __syncthreads();
  // ---- A and B: sixteen lanes per j walk t = 0..15 with p = k_j P_jt (0 before t = j) ----
  {
    const int j = tid >> 4, c = tid & 15;
    float p[DT];
#pragma unroll
    for (int i = 0; i < DT; ++i) p[i] = 0.f;
#pragma unroll 4
    for (int t = 0; t < kB; ++t) {
      float sa = 0.f, sb = 0.f;
#pragma unroll
      for (int i = 0; i < DT; ++i) {
        const float k = kk[t][16 * i + c];
        p[i] = t == j ? k : p[i] * gg[t][16 * i + c];
        sa = fmaf(p[i], k, sa);
        sb = fmaf(p[i], qq[t][16 * i + c], sb);
      }
      sa = xor_sum<8>(xor_sum<4>(xor_sum<2>(xor_sum<1>(sa))));
      sb = xor_sum<8>(xor_sum<4>(xor_sum<2>(xor_sum<1>(sb))));
      if (c == 0) am[t][j] = sa, bm[t][j] = sb;
    }
  }
  __syncthreads();
  // ---- the decayed vectors in place (a thread per channel and direction): kk <- k P, qq <- q P, gg <- k P_.15; T column by column ----
  float* const rec = a.records + ((int64_t)blockIdx.x * a.H + h) * record_floats(DP);
  float* const rec_q = rec + DP * kB;
  float* const rec_k = rec_q + DP * kB;
  float* const rec_b = rec_k + DP * kB;
  // (products of up to sixteen decays in 64 bits, rounded once: the walk applies them to what it has summed over all rows)
  float back[2][kB];
#pragma unroll
  for (int i = 0; i < (2 * DP + 255) / 256; ++i) {
    const int id = tid + 256 * i, d = id < DP ? id : id - DP;
    if (id < 2 * DP) {
      double p = 1.;
      if (id < DP) {
#pragma unroll
        for (int t = 0; t < kB; ++t) {
          p *= gg[t][d];
          qq[t][d] = (float)(qq[t][d] * p);
        }
        gamma[d] = (float)p;
      } else {
#pragma unroll
        for (int t = kB - 1; t >= 0; --t) {
          back[i][t] = (float)(kk[t][d] * p);
          p *= gg[t][d];
        }
        p = 1.;
#pragma unroll
        for (int t = 0; t < kB; ++t) {
          p *= gg[t][d];
          kk[t][d] = (float)(kk[t][d] * p);
        }
      }
    }
  }
  if (tid < kB) {
    const int c = tid;
    float col[kB];
#pragma unroll
    for (int i = 0; i < kB; ++i) {
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) sum = fmaf(am[i][j], col[j], sum);
      col[i] = beta[i] * ((i == c ? 1.f : 0.f) - sum);
    }
#pragma unroll
    for (int i = 0; i < kB; ++i) rec_b[256 + ((c >> 2) * 16 + i) * 4 + (c & 3)] = col[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < (2 * DP + 255) / 256; ++i) {
    const int id = tid + 256 * i;
    if (id >= DP && id < 2 * DP)
#pragma unroll
      for (int t = 0; t < kB; ++t) gg[t][id - DP] = back[i][t];
  }
  __syncthreads();
  // ---- the record, 16 bytes a thread: slot (tile m of 16 channels, lane group g, r) ----
  for (int i = tid; i < DT * 64; i += 256) {
    const int m = i >> 6, kg = (i >> 4) & 3, r = i & 15;
    *reinterpret_cast<float4*>(rec + i * 4) = *reinterpret_cast<const float4*>(&kk[r][16 * m + 4 * kg]);
    *reinterpret_cast<float4*>(rec_q + i * 4) = *reinterpret_cast<const float4*>(&qq[r][16 * m + 4 * kg]);
    *reinterpret_cast<float4*>(rec_k + i * 4) = float4{gg[4 * kg][16 * m + r], gg[4 * kg + 1][16 * m + r], gg[4 * kg + 2][16 * m + r], gg[4 * kg + 3][16 * m + r]};
  }
  if (tid < 64) {
    const int kg = tid >> 4, r = tid & 15;
    *reinterpret_cast<float4*>(rec_b + tid * 4) = float4{bm[r][4 * kg], bm[r][4 * kg + 1], bm[r][4 * kg + 2], bm[r][4 * kg + 3]};
  }
  for (int d = tid; d < DP; d += 256) rec_b[512 + d] = gamma[d];
}

// The rank-th sequence in the order of the rows it brings, the most first: the longest chains begin first and alone.  By one wave for itself, a
// lane for every 64th sequence (up to kOrderedSeqs: read again in every round of the bisection, the numbers of 233 sequences, all but 29 of one row,
// 16 heads of 64 x 128, took a third of the whole call: 679 us, so 455).
constexpr int kOrderedSeqs = 512;
__device__ __forceinline__ int by_length(const int32_t* cu_q, int n_seqs, int rank) {
  const int lane = threadIdx.x & 63;
  int n[kOrderedSeqs / 64], top = 0;
#pragma unroll
  for (int j = 0; j < kOrderedSeqs / 64; ++j) {
    const int i = j * 64 + lane;
    n[j] = i < n_seqs ? cu_q[i + 1] - cu_q[i] : -1;
  }
#pragma unroll
  for (int j = 0; j < kOrderedSeqs / 64; ++j) top = max(top, n[j]);
#pragma unroll
  for (int o = 1; o < 64; o *= 2) top = max(top, __shfl_xor(top, o));
  int lo = 0, hi = __builtin_amdgcn_readfirstlane(top) + 1, behind = 0;   // count(n >= lo) > rank >= count(n >= hi) = behind
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    int c = 0;
#pragma unroll
    for (int j = 0; j < kOrderedSeqs / 64; ++j)
      if (j * 64 < n_seqs) c += __popcll(__ballot(n[j] >= mid));
    if (c > rank) lo = mid;
    else hi = mid, behind = c;
  }
  int k = rank - behind, found = 0;
#pragma unroll
  for (int j = 0; j < kOrderedSeqs / 64; ++j) {
    uint64_t has = __ballot(n[j] == lo);
    const int c = __popcll(has);
    if (k >= 0 && k < c) {
      for (int l = 0; l < k; ++l) has &= has - 1;
      found = j * 64 + __builtin_ctzll(has);
    }
    k -= c;
  }
  return found;
}

// grid: (heads, value columns / (16 CG), sequences) in one, the longest sequences first; two waves take 16 columns, each half of the key channels: what
// one has read of the state meets the other's in LDS, both then have the block's u; the rows' results, which nothing waits for, are put together
// beside the next block's products.  Two records with the rows' values behind each, by LDS-DMA a block ahead, its pieces between the products; in
// front of a group's matrix instructions stand the LDS reads of the next one.  us, before (one wave for all channels, 64 columns a workgroup,
// sequences in order) / so: 11 sequences, 8112 rows, 8 heads of 128 x 128 219 / 158 (sequences in order 201; 64 columns, eight waves in step 215); 728
// rows of 16 sequences 58 / 39.  Of the whole call's time before, drawn steps of 1 .. 500 sequences: 128 channels 0.68 .. 1.02, 64 0.67 .. 1.06 (the most
// where equal sequences filled the CUs once with 64 columns each and now do twice, with 32), 200 and 256 0.61 .. 1.00.
// 64 channels: four workgroups per CU (with a ring of three records and two per CU, 13 sequences of 1752 rows, 16 heads of 64 x 128 677 / 767 us,
// 26 of 840, 8 heads 322 / 363; so 718 and 338) - 128 registers, hence E's products behind D's sum.
// CG: groups of 16 columns of a workgroup.  256 channels leave room for one workgroup per CU: 32 columns were twice the records for
// sequences of a row or two (69 sequences of up to 130 rows, 16 heads of 256 x 256 421 / 520 us; so 414), 64 where there are more than the chip holds.
template <int DT, int CG = 2>
__global__ __launch_bounds__(128 * CG, DT == 4 ? 4 : CG == 4 || DT == 8 ? 2 : 1) void blocks_walk_kernel(BlockArgs a) {
  constexpr int DP = 16 * DT, HT = DT / 2, KT = HT < 4 ? HT : 4, REC = record_floats(DP), PIECES = REC / 256, PP = (PIECES + 2 * CG - 1) / (2 * CG);
  constexpr int IMG = REC * 4 + CG * 1024;
  constexpr bool FOUR = DT == 4;   // workgroups per CU
  __shared__ __attribute__((aligned(1024))) char lds[2 * IMG + 3 * CG * 1024];   // (behind the ring: all waves' D, half of the waves' E)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const int cg = wave % CG, half = wave / CG;   // 16 columns, HT tiles of 16 key channels
  // heads, their columns (one XCD's, where the heads are a multiple of eight: they share the records), sequences
  const int zs = (a.Dv + 16 * CG - 1) / (16 * CG), hz = (int)blockIdx.x % (a.H * zs), h = hz % a.H, col = hz / a.H * (16 * CG) + cg * 16 + r16;
  const int rank = (int)blockIdx.x / (a.H * zs), s = a.n_seqs <= kOrderedSeqs ? by_length(a.cu_q, a.n_seqs, rank) : rank;
  const int r0 = a.cu_q[s], n = a.cu_q[s + 1] - r0;
  if (n == 0) return;
  const int nb = (n + kB - 1) / kB;
  const char* const recs = reinterpret_cast<const char*>(a.records + ((int64_t)first_record(r0, s) * a.H + h) * REC);
  const int64_t rec_stride = (int64_t)a.H * REC * 4;
  const float* vp[2];   // the next block's rows 4 kg + 2 half + i at this lane's column
#pragma unroll
  for (int i = 0; i < 2; ++i)
    vp[i] = a.qkv + (int64_t)(r0 + min(4 * kg + 2 * half + i, n - 1)) * a.ld + a.v_off + (int64_t)h * a.Dv + min(col, a.Dv - 1);
  // PP + 2 requests, whatever the block (beyond the end: the last one's again; rows beyond the end: the last row's)
  auto piece = [&](int b, int st, int i) __attribute__((always_inline)) {
    const int p = min(wave * PP + i, PIECES - 1);
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(recs + min(b, nb - 1) * rec_stride + p * 1024 + (uint32_t)(lane * 16)),
                                     (__attribute__((address_space(3))) void*)(lds + st * IMG + p * 1024), 16, 0, 0);
  };
  auto values = [&](int b, int st) __attribute__((always_inline)) {
    char* const to = lds + st * IMG;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)vp[i],
                                       (__attribute__((address_space(3))) void*)(to + REC * 4 + cg * 1024 + (2 * half + i) * 256), 4, 0, 0);
    const int left = n - 1 - (b + 1) * kB;   // rows behind the next block's first
    if (left >= kB - 1) {
#pragma unroll
      for (int i = 0; i < 2; ++i) vp[i] += (int64_t)kB * a.ld;
    } else if (left >= 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i) vp[i] += (int64_t)(kB + min(4 * kg + 2 * half + i, left) - (4 * kg + 2 * half + i)) * a.ld;
    }
  };
  // the state: S[m][r] = key channel 16 (half HT + m) + 4 kg + r of this lane's column; in memory as the row-by-row kernels keep it
  const int cb = col / kStateCols, cbs = (a.Dv + kStateCols - 1) / kStateCols, cc = col % kStateCols;
  const bool has_state = cb < cbs, has_col = col < a.Dv;
  float* const st = a.state + (((int64_t)a.slot_ids[s] * a.H + h) * cbs + cb) * (DP * kStateCols) + half * HT * (16 * kStateCols);
  f32x4 S[HT];
#pragma unroll
  for (int m = 0; m < HT; ++m) S[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (has_state && a.kv_lens[s] > n) {
#pragma unroll
    for (int m = 0; m < HT; ++m) {
#pragma unroll
      for (int r = 0; r < 4; ++r) S[m][r] = st[(4 * m + r) * (4 * kStateCols) + cc * 4 + kg];
    }
  }
  const uint32_t x_mine = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)(lds + 2 * IMG) + wave * 1024 + lane * 16;
  const uint32_t x_other = half ? x_mine - CG * 1024 : x_mine + CG * 1024, x_e = x_mine + (half ? CG : 2 * CG) * 1024;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  float* op = a.out + (int64_t)(r0 + 4 * kg) * a.ldo + (int64_t)h * a.Dv + col;   // (formed beyond the columns, not used there)
  auto store = [&](int b) __attribute__((always_inline)) {
    if (b * kB + kB <= n) {
      if (has_col)
#pragma unroll
        for (int r = 0; r < 4; ++r) op[r * a.ldo] = o[r];
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (has_col && b * kB + 4 * kg + r < n) op[r * a.ldo] = o[r];
    }
    op += (int64_t)kB * a.ldo;
  };
#pragma unroll
  for (int q = 0; q < PP; ++q) piece(0, 0, q);
  values(0, 0);
  f32x4 e_own = {}, x = {}, w = {}, u = {};
  // block b's rows, when the halves' sums of E have met (in the next block, beside its products)
  auto finish = [&](int b) __attribute__((always_inline)) {
    f32x4 e_other;
    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(e_other) : "v"(x_e) : "memory");
    e_other += e_own;
    o = e_other + x;
    float zero = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) zero = fmaf(o[r], 0.f, zero);
    // (the state has what is not finite either way; the whole wave takes the branch)
    if (__builtin_expect(__any(zero != 0.f), 0)) {
      const char* const at = recs + b * rec_stride + 3 * DP * kB * 4 + lane * 16;
      const f32x4 x2 = causal(*reinterpret_cast<const f32x4*>(at), causal(*reinterpret_cast<const f32x4*>(at + 1024), w, u, kg), x, kg);
      o = e_other + x2;
    }
    store(b);
  };
  int cur = 0;
  for (int b = 0; b < nb; ++b) {
    // record b has landed; everybody is done with record b - 1: its place is free
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (b > 0 && half == 0) finish(b - 1);   // (the other half's products keep the matrix pipe busy)
    const char* const img = lds + cur * IMG;
    cur ^= 1;
    const char* const rec = img + lane * 16 + half * HT * 1024;
    const char* const rec_q = rec + DP * kB * 4;
    const char* const rec_k = rec_q + DP * kB * 4;
    const char* const rec_b = img + lane * 16 + 3 * DP * kB * 4;
    const char* const gam = rec_b - lane * 16 + 2048 + kg * 16 + half * HT * 64;   // P_15 of this lane's channels 16 m + 4 kg ..
    auto vec = [](const char* p) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(p); };
    f32x4 d[8], e[8];   // (eight chains: each is an eighth as long, and so is its rounding)
#pragma unroll
    for (int r = 0; r < 8; ++r) d[r] = e[r] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 mine, pf[2][2], qf[2][2], gf[2][2], kf[2][4], tf = vec(rec_b + 1024), bf = vec(rec_b);
#pragma unroll
    for (int r = 0; r < 4; ++r) u[r] = *reinterpret_cast<const float*>(img + REC * 4 + cg * 1024 + r * 256 + lane * 4);
    auto read_q = [&](int c) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        pf[c & 1][i] = vec(rec + (2 * c + i) * 1024);
        qf[c & 1][i] = vec(rec_q + (2 * c + i) * 1024);
        gf[c & 1][i] = vec(gam + (2 * c + i) * 64);
      }
    };
    auto read_k = [&](int c) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < KT; ++i) kf[c & 1][i] = vec(rec_k + (KT * c + i) * 1024);
    };
    read_q(0);
#pragma unroll
    for (int c = 0; c < HT / 2; ++c) {
      if (c + 1 < HT / 2) read_q(c + 1);
      else read_k(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          f32x4 &dx = d[4 * i + r], &ex = e[4 * i + r];
          dx = __builtin_amdgcn_mfma_f32_16x16x4f32(pf[c & 1][i][r], S[2 * c + i][r], dx, 0, 0, 0);
          if constexpr (!FOUR) ex = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[c & 1][i][r], S[2 * c + i][r], ex, 0, 0, 0);
          // the next record, a piece behind every few products (in front of them all the CU's requests took 700 cycles)
          constexpr int EVERY = HT * 4 / PP;
          static_assert(EVERY > 0, "every piece has its place");
          const int at = (c * 2 + i) * 4 + r;
          if (at % EVERY == EVERY - 1 && at / EVERY < PP) {
            piece(b + 1, cur, at / EVERY);
            __builtin_amdgcn_sched_barrier(0);
          }
          if (at == HT * 4 - 1) {
            values(b + 1, cur);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      if constexpr (FOUR) {   // (E behind D: a set of chains less in registers)
        mine = sum8(d);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) e[4 * i + r] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[0][i][r], S[i][r], e[4 * i + r], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) S[2 * c + i] *= gf[c & 1][i];
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) u[r] = has_col && b * kB + 4 * kg + r < n ? u[r] : 0.f;
    if constexpr (!FOUR) mine = sum8(d);
    f32x4 other;
    asm volatile("ds_write_b128 %0, %1" ::"v"(x_mine), "v"(mine) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (read below, and written again only behind the next block's barrier)
    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(other) : "v"(x_other) : "memory");
    w = u - (mine + other);
    u = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) u = __builtin_amdgcn_mfma_f32_16x16x4f32(tf[r], w[r], u, 0, 0, 0);
#pragma unroll
    for (int c = 0; c < HT / KT; ++c) {
      if (c + 1 < HT / KT) read_k(c + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 4; ++r)   // (r outside i: a tile's four products wait for each other)
#pragma unroll
        for (int i = 0; i < KT; ++i) S[KT * c + i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c & 1][i][r], u[r], S[KT * c + i], 0, 0, 0);
    }
    e_own = sum8(e);
    if (half) {   // (read behind the next block's barrier, and written again behind its second)
      asm volatile("ds_write_b128 %0, %1" ::"v"(x_e), "v"(e_own) : "memory");
    } else {
      x = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) x = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[r], u[r], x, 0, 0, 0);
    }
  }
  // (the requests beyond the end land before the workgroup's LDS is given away)
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if (half == 0) finish(nb - 1);
  if (!has_state) return;
#pragma unroll
  for (int m = 0; m < HT; ++m) {
#pragma unroll
    for (int r = 0; r < 4; ++r) st[(4 * m + r) * (4 * kStateCols) + cc * 4 + kg] = S[m][r];
  }
}

// ---------------------------------------------------------------------------
// Linear attention with a decayed state (mi_linear_attention's recurrence, S <- diag(g_t) S + k_t v_t^T, o_t = S^T q_t) in the same blocks:
//   O = (q_t P_t)^T S0 + B V,   B_tj = sum_d q_t P_jt k_j  (j <= t),      S <- diag(P_15) S0 + sum_j (k_j P_j15) v_j^T
// FORGET: g_t per channel from the f rows, k = 1 - g; else one decay per head.  A record: [q P: DP * 16][k P_.15: DP * 16][B: 512][P_15: 2 DP],
// B and P_15 as high and low parts: a row behind quick decays is little more than its own products, and the state meets the same P_15
// block after block where a head has one decay.
//
// What bounds it: the row-by-row walk reads q, k (and g) of every row for every value column from LDS, 0.38 - 0.42 us a row; here 72 matrix
// instructions (128 channels) are 1.0 us per sixteen rows, with the LDS reads and sums between them 2.3.  8 sequences of 1024 rows, 16
// heads of 128 x 128: a decay per head 399 us row by row, 205 so (preparation 68); per channel 458, 235 (109).  rms error against 64
// bits, row by row = 1 (128 and 300 rows; D 64, 128, 256; means of six inputs): forget gates 0.82 - 0.86, decays of 1 - 2^-5 and slower 0.64 - 0.87,
// one decay of 0.3 to 0.8 0.81 - 0.87, of 0.95 0.79 - 0.90.  (B's products of q and k summed over the lanes in 32 bits: 1.01 - 1.08 for decays up to
// 0.7, whose rows are little else, and 1 to 4 % less time; the lanes' few products each are.)
// ---------------------------------------------------------------------------
constexpr int lin_record_floats(int dp) { return (2 * dp * kB + 512 + 2 * dp + 255) & ~255; }

struct LinearArgs {
  const float* proj;
  int64_t ld;
  int q_off, k_off, v_off;
  bool q_silu, k_silu, v_silu;
  const float* decay;     // [H]
  const float* f_bias;    // [H * D]
  const float* lower;     // [H * D]
  const int32_t* cu_q;
  const int32_t* kv_lens;
  const int32_t* slot_ids;
  int n_seqs, H, D, Dv;
  float* state;
  float* records;
  float* out;
  int64_t ldo;
};

template <int O>   // v + the value of lane ^ O, without the LDS crossbar
__device__ __forceinline__ double xor_sum64(double v) {
  return v + __hiloint2double(__float_as_int(xor_get<O>(__int_as_float(__double2hiint(v)))), __float_as_int(xor_get<O>(__int_as_float(__double2loint(v)))));
}

__device__ __forceinline__ float silu_if(bool on, float z) { return on ? z / (1.f + expf(-z)) : z; }

template <int DT, bool FORGET>
__global__ __launch_bounds__(256) void linear_prepare_kernel(LinearArgs a) {
  constexpr int DP = 16 * DT, LD = DP + 4;   // (as blocks_prepare_kernel)
  __shared__ __attribute__((aligned(16))) float kk[kB][LD], qq[kB][LD], gg[FORGET ? kB : 1][LD];
  __shared__ float bm[kB][kB + 1], bl[kB][kB + 1], gamma[DP], gamma_low[DP];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = blockIdx.y;
  int s = -1;   // the block's sequence: the last one whose records begin at or before it
  for (int i0 = 0; i0 < a.n_seqs; i0 += 64) {
    const int i = i0 + lane;
    const int found = __popcll(__ballot(i < a.n_seqs && first_record(a.cu_q[min(i, a.n_seqs - 1)], i) <= (int)blockIdx.x));
    s += found;
    if (found < 64) break;
  }
  s = __builtin_amdgcn_readfirstlane(s);
  const int r0 = a.cu_q[s] + ((int)blockIdx.x - first_record(a.cu_q[s], s)) * kB, n = min(kB, a.cu_q[s + 1] - r0);
  if (n <= 0) return;  // (a record that no block uses)
  // rows beyond the sequence's end and channels beyond D change nothing: q = k = 0, g = 1
  constexpr int RW = kB / 4, C = DP / 64;
  float qv[RW][C], kv[RW][C];
#pragma unroll
  for (int i = 0; i < RW; ++i) {   // (every load first, at clamped places: none waits for another)
    const float* p = a.proj + (int64_t)(r0 + min(wave * RW + i, n - 1)) * a.ld + h * a.D;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int d = min(lane + 64 * c, a.D - 1);
      qv[i][c] = p[a.q_off + d];
      kv[i][c] = p[a.k_off + d];
    }
  }
  const float head_decay = FORGET ? 1.f : a.decay[h];
  float lo[C], fb[C];
  if constexpr (FORGET) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int d = h * a.D + min(lane + 64 * c, a.D - 1);
      lo[c] = a.lower[d], fb[c] = a.f_bias[d];
    }
  }
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int t = wave * RW + i;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const bool ok = t < n && lane + 64 * c < a.D;
      qq[t][lane + 64 * c] = ok ? silu_if(a.q_silu, qv[i][c]) : 0.f;
      if constexpr (FORGET) {
        const float f = lo[c] + (1.f - lo[c]) * sigmoid_f(kv[i][c] + fb[c]);
        gg[t][lane + 64 * c] = ok ? f : 1.f;
        kk[t][lane + 64 * c] = ok ? 1.f - f : 0.f;
      } else {
        kk[t][lane + 64 * c] = ok ? silu_if(a.k_silu, kv[i][c]) : 0.f;
      }
    }
  }
  __syncthreads();
  // ---- B: sixteen lanes per j walk t = 0..15, four channels at a time, with p = k_j P_jt (0 before t = j); one decay per head: with k_j,
  // and the sum times the decay's power ----
  {
    const int j = tid >> 4, c = (tid & 15) * 4;
    using T = std::conditional_t<FORGET, double, float>;
    T p[C][4];
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const f32x4 k = *reinterpret_cast<const f32x4*>(&kk[j][64 * i + c]);
#pragma unroll
      for (int e = 0; e < 4; ++e) p[i][e] = k[e];
    }
    double power = 1.;   // of the head's decay, t - j
#pragma unroll 4
    for (int t = 0; t < kB; ++t) {
      T sum[4] = {0, 0, 0, 0};
      const bool decays = t > j;
      if (!FORGET && decays) power *= head_decay;
#pragma unroll
      for (int i = 0; i < C; ++i) {
        const f32x4 q = *reinterpret_cast<const f32x4*>(&qq[t][64 * i + c]);
        if constexpr (FORGET) {
          const f32x4 g = *reinterpret_cast<const f32x4*>(&gg[t][64 * i + c]);
#pragma unroll
          for (int e = 0; e < 4; ++e) p[i][e] = decays ? p[i][e] * g[e] : p[i][e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] += p[i][e] * q[e];
      }
      const double b = xor_sum64<8>(xor_sum64<4>(xor_sum64<2>(xor_sum64<1>(((double)sum[0] + sum[1]) + ((double)sum[2] + sum[3])))));
      const double bp = t < j ? 0. : FORGET ? b : b * power;
      if (c == 0) bm[t][j] = (float)bp, bl[t][j] = (float)(bp - (float)bp);
    }
  }
  __syncthreads();
  // ---- the decayed vectors in place, a thread per channel and direction (products of up to sixteen decays in 64 bits, rounded once: the
  // walk applies them to what it has summed over all rows) ----
#pragma unroll
  for (int i = 0; i < (2 * DP + 255) / 256; ++i) {
    const int id = tid + 256 * i, d = id < DP ? id : id - DP;
    if (id >= 2 * DP) break;
    double p = 1.;
    if (id < DP) {
#pragma unroll
      for (int t = 0; t < kB; ++t) {
        if (FORGET) p *= gg[FORGET ? t : 0][d];
        else if (t < n) p *= head_decay;
        qq[t][d] = (float)(qq[t][d] * p);
      }
      gamma[d] = (float)p;
      gamma_low[d] = (float)(p - gamma[d]);
    } else {
#pragma unroll
      for (int t = kB - 1; t >= 0; --t) {
        kk[t][d] = (float)(kk[t][d] * p);
        if (FORGET) p *= gg[FORGET ? t : 0][d];
        else if (t < n) p *= head_decay;
      }
    }
  }
  __syncthreads();
  // ---- the record, 16 bytes a thread: slot (tile m of 16 channels, lane group g, r) ----
  float* const rec_q = a.records + ((int64_t)blockIdx.x * a.H + h) * lin_record_floats(DP);
  float* const rec_k = rec_q + DP * kB;
  float* const rec_b = rec_k + DP * kB;
  for (int i = tid; i < DT * 64; i += 256) {
    const int m = i >> 6, kg = (i >> 4) & 3, r = i & 15;
    *reinterpret_cast<float4*>(rec_q + i * 4) = *reinterpret_cast<const float4*>(&qq[r][16 * m + 4 * kg]);
    *reinterpret_cast<float4*>(rec_k + i * 4) = float4{kk[4 * kg][16 * m + r], kk[4 * kg + 1][16 * m + r], kk[4 * kg + 2][16 * m + r], kk[4 * kg + 3][16 * m + r]};
  }
  if (tid < 64) {
    const int kg = tid >> 4, r = tid & 15;
    *reinterpret_cast<float4*>(rec_b + tid * 4) = float4{bm[r][4 * kg], bm[r][4 * kg + 1], bm[r][4 * kg + 2], bm[r][4 * kg + 3]};
    *reinterpret_cast<float4*>(rec_b + 256 + tid * 4) = float4{bl[r][4 * kg], bl[r][4 * kg + 1], bl[r][4 * kg + 2], bl[r][4 * kg + 3]};
  }
  for (int d = tid; d < DP; d += 256) rec_b[512 + d] = gamma[d], rec_b[512 + DP + d] = gamma_low[d];
}

// grid: (sequences, heads, value columns / 64); a wave takes 16 columns, its S as blocks_walk_kernel's.  Ring of three records by LDS-DMA
// two blocks ahead, with the rows' values behind each.
template <int DT>
__global__ __launch_bounds__(256, 1) void linear_walk_kernel(LinearArgs a) {
  constexpr int DP = 16 * DT, REC = lin_record_floats(DP), PIECES = REC / 256, PP = (PIECES + 3) / 4, IMG = REC * 4 + 4096;
  static_assert(3 * IMG <= 163840, "three records");
  __shared__ __attribute__((aligned(1024))) char lds[3 * IMG];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const int s = blockIdx.x, h = blockIdx.y, col = blockIdx.z * 64 + wave * 16 + r16;
  const int r0 = a.cu_q[s], n = a.cu_q[s + 1] - r0;
  if (n == 0) return;
  const int nb = (n + kB - 1) / kB;
  const char* const recs = reinterpret_cast<const char*>(a.records + ((int64_t)first_record(r0, s) * a.H + h) * REC);
  const int64_t rec_stride = (int64_t)a.H * REC * 4;
  const float* vp[4];   // the next block's rows 4 kg + r at this lane's column
#pragma unroll
  for (int r = 0; r < 4; ++r)
    vp[r] = a.proj + (int64_t)(r0 + min(4 * kg + r, n - 1)) * a.ld + a.v_off + (int64_t)h * a.Dv + min(col, a.Dv - 1);
  // PP + 4 requests, whatever the block (beyond the end: the last one's again; rows beyond the end: the last row's)
  auto issue = [&](int b, int st) __attribute__((always_inline)) {
    const int bb = min(b, nb - 1);
    char* const to = lds + st * IMG;
#pragma unroll
    for (int i = 0; i < PP; ++i) {
      const int p = min(wave * PP + i, PIECES - 1);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(recs + bb * rec_stride + p * 1024 + (uint32_t)(lane * 16)),
                                       (__attribute__((address_space(3))) void*)(to + p * 1024), 16, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)vp[r],
                                       (__attribute__((address_space(3))) void*)(to + REC * 4 + wave * 1024 + r * 256), 4, 0, 0);
    const int left = n - 1 - (b + 1) * kB;   // rows behind the next block's first
    if (left >= kB - 1) {
#pragma unroll
      for (int r = 0; r < 4; ++r) vp[r] += (int64_t)kB * a.ld;
    } else if (left >= 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) vp[r] += (int64_t)(kB + min(4 * kg + r, left) - (4 * kg + r)) * a.ld;
    }
  };
  // the state: S[m][r] = key channel 16 m + 4 kg + r of this lane's column; in memory four channels of a column together (as the
  // row-by-row kernel keeps it)
  const int cb = col / kStateCols, cbs = (a.Dv + kStateCols - 1) / kStateCols, cc = col % kStateCols;
  const bool has_state = cb < cbs, has_col = col < a.Dv;
  float* const st = a.state + (((int64_t)a.slot_ids[s] * a.H + h) * cbs + cb) * (DP * kStateCols) + (kg * kStateCols + cc) * 4;
  f32x4 S[DT];
#pragma unroll
  for (int m = 0; m < DT; ++m) {
    S[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (has_state && a.kv_lens[s] > n) S[m] = *reinterpret_cast<const f32x4*>(st + m * (16 * kStateCols));
  }
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  float* op = a.out + (int64_t)(r0 + 4 * kg) * a.ldo + (int64_t)h * a.Dv + col;   // (formed beyond the columns, not used there)
  auto store = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (has_col && b * kB + 4 * kg + r < n) op[r * a.ldo] = o[r];
    op += (int64_t)kB * a.ldo;
  };
#pragma unroll
  for (int i = 0; i < 2; ++i) issue(i, i);
  int cur = 0;
  for (int b = 0; b < nb; ++b) {
    // record b has landed (record b + 1's requests may be out); everybody is done with record b - 1: its place is free
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PP + 4) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (b > 0) store(b - 1);   // (here, not behind the block: the wait above would have to see them home)
    issue(b + 2, cur == 0 ? 2 : cur - 1);
    const char* const img = lds + cur * IMG;
    cur = cur == 2 ? 0 : cur + 1;
    const char* const rec_q = img + lane * 16;
    const char* const rec_k = rec_q + DP * kB * 4;
    const char* const rec_b = rec_k + DP * kB * 4;
    const char* const gam = rec_b - lane * 16 + 2048 + kg * 16;   // P_15 of this lane's channels 16 m + 4 kg ..
    auto vec = [](const char* p) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(p); };
    f32x4 e[8];   // (eight chains: each is an eighth as long, and so is its rounding)
#pragma unroll
    for (int r = 0; r < 8; ++r) e[r] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 qf[2][2], gf[2][2], gl[2][2], kf[2][2], v, bf = vec(rec_b);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = *reinterpret_cast<const float*>(img + REC * 4 + wave * 1024 + r * 256 + lane * 4);
    auto read = [&](int c) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        qf[c & 1][i] = vec(rec_q + (2 * c + i) * 1024);
        kf[c & 1][i] = vec(rec_k + (2 * c + i) * 1024);
        gf[c & 1][i] = vec(gam + (2 * c + i) * 64);
        gl[c & 1][i] = vec(gam + DP * 4 + (2 * c + i) * 64);
      }
    };
    read(0);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = has_col && b * kB + 4 * kg + r < n ? v[r] : 0.f;
    if (a.v_silu)   // (silu(0) = 0)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = silu_if(true, v[r]);
#pragma unroll
    for (int c = 0; c < DT / 2; ++c) {
      if (c + 1 < DT / 2) read(c + 1);
      // a pair of tiles: read with the decayed queries, then decayed and the rows added
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          f32x4& ex = e[4 * i + r];
          ex = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[c & 1][i][r], S[2 * c + i][r], ex, 0, 0, 0);
        }
      // (the rows are summed from zero and meet the state once: sixteen roundings of their size, one of the state's)
      f32x4 rows[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int r = 0; r < 4; ++r)   // (r outside i: a tile's four products wait for each other)
#pragma unroll
        for (int i = 0; i < 2; ++i) rows[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c & 1][i][r], v[r], rows[i], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[2 * c + i][r] = fmaf(gf[c & 1][i][r], S[2 * c + i][r], fmaf(gl[c & 1][i][r], S[2 * c + i][r], rows[i][r]));
    }
    const f32x4 low = vec(rec_b + 1024);
    f32x4 state4[4], rows4[4];   // (what is left of the sums is added in 64 bits: it rounds once)
#pragma unroll
    for (int r = 0; r < 4; ++r) state4[r] = e[r] + e[r + 4];
    auto add_up = [&](f32x4 b4) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        rows4[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(low[r], b4[r], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        rows4[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[r], b4[r], rows4[r], 0, 0, 0);
      }
      f32x4 y;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        y[i] = (float)((((double)state4[0][i] + state4[1][i]) + ((double)state4[2][i] + state4[3][i])) +
                       (((double)rows4[0][i] + rows4[1][i]) + ((double)rows4[2][i] + rows4[3][i])));
      return y;
    };
    o = add_up(v);
    float zero = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) zero = fmaf(o[r], 0.f, zero);
    // (the state has what is not finite either way; the whole wave takes the branch)
    if (__builtin_expect(__any(zero != 0.f), 0)) {   // rows in front of the column's first value that is not finite: see causal()
      const int first = first_bad(v, kg);
      f32x4 front;
#pragma unroll
      for (int r = 0; r < 4; ++r) front[r] = 4 * kg + r < first ? v[r] : 0.f;
      const f32x4 y = add_up(front);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = 4 * kg + r < first ? y[r] : o[r];
    }
  }
  store(nb - 1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the requests beyond the end land before the workgroup's LDS is given away)
  if (!has_state) return;
#pragma unroll
  for (int m = 0; m < DT; ++m) *reinterpret_cast<f32x4*>(st + m * (16 * kStateCols)) = S[m];
}

static int tiles_of(int D) { return D <= 64 ? 4 : D <= 128 ? 8 : D <= 256 ? 16 : 0; }

}  // namespace mi

using namespace mi;

// Where the block form is used: a sequence's chain of blocks is 1.9 us per 16 rows against 0.71 us a row, but every sequence, also one
// that brings a single row, costs a record and a workgroup per 32 columns.  us from cold inputs, rows / blocks, 8 heads of 128 x 128: one sequence of 16 rows
// 35 / 35, of 32 46 / 37; 32 sequences of 16 rows 46 / 52, of 32 64 / 62; 64 of 16 69 / 75; 32 rows beside 31 single ones 50 / 46, 64 beside 127 96 / 107, 96
// beside 127 124 / 108, 128 beside 255 174 / 193, 160 beside 255 201 / 193; 256 sequences of 2 rows 69 / 186 (4 heads of 64 x 128, 16 of 128 x 128
// and 8 of 256 x 256: none slower beyond the line).
extern "C" int64_t mi_channel_delta_blocks_elems(int n_rows, int n_seqs, int max_rows, int H, int D) {
  const int dt = tiles_of(D);
  if (n_rows < 0 || n_seqs < 1 || H < 1 || D < 1 || dt == 0) return -1;
  if (max_rows < 32 + n_seqs / 2) return 0;
  return ((int64_t)n_rows / kB + n_seqs) * H * record_floats(16 * dt);
}

extern "C" int mi_channel_delta_blocks(const float* qkv, int64_t ld, int q_off, int k_off, int v_off, const float* beta_pre,
                                       int64_t ld_beta, const float* decay_pre, int64_t ld_decay, const float* dt_bias,
                                       const float* a_log, const float* gate_pre, int64_t ld_gate, const float* norm_w, float* state,
                                       const int32_t* cu_q, const int32_t* kv_lens, const int32_t* slot_ids, int n_seqs, int n_rows,
                                       int H, int G, int D, int Dv, float eps, float* workspace, int64_t ws_elems, float* out,
                                       int64_t ldo, mi_stream stream) {
  if (!qkv || !beta_pre || !decay_pre || !dt_bias || !a_log || !gate_pre || !norm_w || !state || !cu_q || !kv_lens || !slot_ids || !out ||
      !workspace || n_seqs < 1 || n_rows < 0 || H < 1 || G < 1 || H % G || D < 1 || Dv < 1)
    return MI_EINVAL;
  const int dt = tiles_of(D);
  if (dt == 0 || H > 65535 || Dv > 65535) return MI_EUNSUPPORTED;
  if (n_rows == 0) return MI_OK;
  if (!aligned16(workspace) || ws_elems < ((int64_t)n_rows / kB + n_seqs) * H * record_floats(16 * dt)) return MI_EWORKSPACE;
  const BlockArgs a{qkv, ld, q_off, k_off, v_off, beta_pre, ld_beta, decay_pre, ld_decay, dt_bias, a_log, cu_q, kv_lens, slot_ids,
                    n_seqs, H, G, D, Dv, state, workspace, out, ldo};
  const auto walks = [&](int cg) { return (int64_t)n_seqs * H * ((Dv + 16 * cg - 1) / (16 * cg)); };   // (32 columns: a block of the state's layout)
  if (walks(2) > 0x7fffffff) return MI_EUNSUPPORTED;
  const dim3 prep(n_rows / kB + n_seqs, H);
  const auto launch = [&](auto prepare, auto walk_kernel, int cg) -> int {
    hipLaunchKernelGGL(prepare, prep, dim3(256), 0, S(stream), a);
    if (check_launch() != MI_OK) return MI_ELAUNCH;
    hipLaunchKernelGGL(walk_kernel, dim3((unsigned)walks(cg)), dim3(128 * cg), 0, S(stream), a);
    return check_launch();
  };
  // (256 channels: a CU holds one workgroup; where 32 columns each would be more than that, 64)
  const int rc = dt == 4             ? launch(blocks_prepare_kernel<4>, blocks_walk_kernel<4>, 2)
                 : dt == 8           ? launch(blocks_prepare_kernel<8>, blocks_walk_kernel<8>, 2)
                 : walks(2) <= 256   ? launch(blocks_prepare_kernel<16>, blocks_walk_kernel<16>, 2)
                                     : launch(blocks_prepare_kernel<16>, blocks_walk_kernel<16, 4>, 4);
  return rc != MI_OK ? rc : launch_head_norm(out, ldo, gate_pre, ld_gate, norm_w, n_rows, H, Dv, eps, S(stream));
}

// Where linear attention takes the block form.  us, rows / blocks, a decay per head (per channel), 16 heads of 128 x 128: one sequence of 64 rows
// 20 / 21 (23 / 23), of 128 38 / 32 (43 / 33), 1024 275 / 185; 8 of 100 49 / 42; 32 of 32 53 / 55 (59 / 62), of 64 109 / 85; 64 rows beside 31
// single ones 83 / 66; 8 heads: 8 of 100 34 / 35.
extern "C" int64_t mi_linear_attention_blocks_elems(int n_rows, int n_seqs, int max_rows, int H, int D) {
  const int dt = tiles_of(D);
  if (n_rows < 0 || n_seqs < 1 || H < 1 || D < 1 || dt == 0) return -1;
  if (max_rows < (n_seqs < 16 ? 96 : 48 + n_seqs / 2)) return 0;
  return ((int64_t)n_rows / kB + n_seqs) * H * lin_record_floats(16 * dt);
}

namespace mi {
int launch_linear_blocks(const float* proj, int64_t ld, int q_off, int k_off, int v_off, int q_act, int k_act, int v_act, int decay_kind,
                         const float* decay, const float* f_bias, const float* lower, float* state, const int32_t* cu_q,
                         const int32_t* kv_lens, const int32_t* slot_ids, int n_seqs, int n_rows, int H, int D, int Dv, float* workspace,
                         int64_t ws_elems, float* out, int64_t ldo, hipStream_t st) {
  const int dt = tiles_of(D);
  if (dt == 0 || H > 65535 || Dv > 65535 || !aligned16(state)) return MI_EUNSUPPORTED;
  if (!aligned16(workspace) || ws_elems < ((int64_t)n_rows / kB + n_seqs) * H * lin_record_floats(16 * dt)) return MI_EWORKSPACE;
  const LinearArgs a{proj, ld, q_off, k_off, v_off, q_act == MI_ACT_SILU, k_act == MI_ACT_SILU, v_act == MI_ACT_SILU, decay, f_bias, lower, cu_q,
                     kv_lens, slot_ids, n_seqs, H, D, Dv, state, workspace, out, ldo};
  const dim3 prep(n_rows / kB + n_seqs, H), walk(n_seqs, H, (Dv + 63) / 64);   // (64 columns hold whole blocks of the state's layout)
  const auto launch = [&](auto prepare, auto walk_kernel) -> int {
    hipLaunchKernelGGL(prepare, prep, dim3(256), 0, st, a);
    if (check_launch() != MI_OK) return MI_ELAUNCH;
    hipLaunchKernelGGL(walk_kernel, walk, dim3(256), 0, st, a);
    return check_launch();
  };
  if (decay_kind == MI_DECAY_FORGET)
    return dt == 4   ? launch(linear_prepare_kernel<4, true>, linear_walk_kernel<4>)
           : dt == 8 ? launch(linear_prepare_kernel<8, true>, linear_walk_kernel<8>)
                     : launch(linear_prepare_kernel<16, true>, linear_walk_kernel<16>);
  return dt == 4   ? launch(linear_prepare_kernel<4, false>, linear_walk_kernel<4>)
         : dt == 8 ? launch(linear_prepare_kernel<8, false>, linear_walk_kernel<8>)
                   : launch(linear_prepare_kernel<16, false>, linear_walk_kernel<16>);
}
}  // namespace mi
