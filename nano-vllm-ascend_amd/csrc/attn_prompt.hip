// Attention of prompt portions over paged K / V rows for fp32 queries (mi_swa_attention, mi_paged_attention_*): causal within a
// window / chunk / kept first keys, distance bias, sink, capped scores, separate key and value head sizes, gate.
//
// A workgroup takes 128 columns - a column is a (step row, query head) - of one sequence and one key/value head: with H / G
// query heads to a key/value head, 128 / (H / G) consecutive rows of the sequence.  Its eight waves own 16 columns each and
// walk the same keys, 32 at a time: a step's K and V rows go from memory to LDS once for all 128 columns (LDS-DMA into a ring of
// NST images, NST - 1 steps in flight, one barrier per step), as stored, a row's 16-byte chunks XOR-swizzled by its number.
//   scores   S^T = K Q^T: keys on the MFMA's row axis, the columns on its column axis.
//            bf16 cache: v_mfma_f32_16x16x32_bf16 with q as bf16 hi + lo (products exact, 16 mantissa bits of q);
//            fp32 cache: v_mfma_f32_16x16x4_f32.
//   softmax  scale, bias, cap, mask, running reference point and sum per column in fp32 on the accumulators; a lane holds the keys
//            4 kg + {0..3} of the step's two 16-key tiles for its column.
//   output   O^T += V^T P^T with the contraction slots in the order the scores lie in the registers, so a weight never leaves
//            its lane.  bf16 cache: weights as hi + lo pairs, V^T by the transposing LDS read (four keys at a lane's channel); fp32
//            cache: V element by element.  Values that are the leading channels of the key rows (latent attention) are read from
//            the K image: nothing is loaded for them.
//
// What bounds it: memory latency per step where a walk is short (a window), the matrix and LDS pipes (64 matrix instructions and 32
// KiB of fragments per 16 columns and 32 keys at 256 channels) where it is long.  The kernels it replaces - a wave per 16
// columns with K and V from L2 by every wave and V in 4-byte gathers; over fp32 rows plain FMA chains - waited for memory.
// Measured: see launch_prompt_attention.
//
// Keys that a column does not see weigh 0 in its products, and 0 times a NaN or an infinity among their values is NaN: a column whose
// result is not finite is taken again without them (attend_column; the look at the results costs 0.6 us of a launch).
#include "attn_bias.hpp"

namespace mi {

constexpr int kCols = 128, kKeys = 32, kPromptThreads = 512, kWaves = 8;
constexpr float kLog2e = 1.44269504088896340736f;
typedef short s16x4 __attribute__((ext_vector_type(4)));

// One column by one wave, keys it does not see left out instead of weighed with 0: for columns that the matrix instructions gave
// something that is not finite, because a key of their step that they do not see has a NaN or an infinity among its values.
template <typename TC>
__device__ __forceinline__ void attend_column(const float* q, const TC* k_cache, const TC* v_cache, const int32_t* table, int pos, int h, int H,
                                              int G, int D, int Dv, int block_size, int window, float scale, const AttnBias& bias, int64_t ldv,
                                              const float* gate, float* out) {
  const int lane = threadIdx.x & 63, g = h / (H / G), Gv = bias.value_heads, gv = h / (H / Gv), bs_shift = block_shift(block_size);
  const int lo = first_key(bias, pos, window), gap = kept_gap(bias, lo);
  const HeadBias hb = head_bias(bias, h, H);
  float m = -INFINITY, l = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};   // (Dv <= 256)
  for (int j0 = gap; j0 <= pos; j0 += 64) {
    const int j = key_at<true>(j0 + lane, lo, gap);
    float sc = -INFINITY;
    if (j <= pos) {
      const TC* kr = k_cache + (int64_t)cache_row(table, j, G, g, block_size, bs_shift) * D;
      float dot = 0.f;
#pragma unroll 1
      for (int d = 0; d < D; ++d) dot = fmaf(q[d], ld_f<TC>(kr + d), dot);
      sc = capped(bias, dot * scale - dist_bias(hb, pos - j));
    }
    const float m_new = fmaxf(m, wave_max(sc));
    const float mref = m_new == -INFINITY ? 0.f : m_new;
    const float p = j <= pos ? expf(sc - mref) : 0.f, corr = expf(m - mref);
    l = l * corr + wave_sum(p);
    m = m_new;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] *= corr;
    const int n = min(64, pos - j0 + 1);
#pragma unroll 1
    for (int jj = 0; jj < n; ++jj) {
      const float pj = __shfl(p, jj);
      const TC* vr = v_cache + (int64_t)cache_row(table, key_at<true>(j0 + jj, lo, gap), Gv, gv, block_size, bs_shift) * ldv;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (lane + 64 * i < Dv) acc[i] = fmaf(pj, ld_f<TC>(vr + lane + 64 * i), acc[i]);
    }
  }
  const float inv = 1.f / with_sink(bias, h, m, l);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int d = lane + 64 * i;
    if (d < Dv) out[d] = acc[i] * inv * (gate ? sigmoid_f(gate[d]) : 1.f);
  }
}

// The rank-th tile (of R rows) in the order of the positions their last rows have, the largest first - the longest walks first, whatever
// sequences they belong to: workgroups are dispatched in this order, and where there are more than the chip holds the short ones fill
// the gaps (with sequence after sequence the last sequence's longest walks began when half of the chip was idle).  By one wave for itself, a
// lane a sequence: bisection for the position that rank tiles lie behind.  table: {rows, rows in front of them} of more than 64 sequences in
// LDS (from memory in every round of the bisection, 3 loads per 64 sequences: us, sequence after sequence / so / now: 100 sequences of 1 row behind 600
// and one of 300, 16 heads of 64 on fp32 pages 215 / 262 / 219, 300 and one of 600 752 / 897 / 770).  us, sequence after sequence / this order:
// 8 x 1024 rows, 16 heads over one 256-channel row (1024 workgroups, one per CU) 271 / 210; 11 prompts, 8112 rows, 8 / 4 heads x 128, window
// 512: 95 / 89.
constexpr int kOrderedSeqs = 4096;   // (the smallest ring's 32 KiB)
__device__ __forceinline__ bool tile_by_end(const int32_t* cu_q, const int32_t* kv_lens, const int2* table, int n_seqs, int R, int rank, int& s,
                                            int& first) {
  const int lane = threadIdx.x & 63;
  int n = 0, past = 0;
  auto look = [&](int i) __attribute__((always_inline)) {
    n = past = 0;
    if (i >= n_seqs) return;
    if (table) {
      n = table[i].x, past = table[i].y;
    } else {
      n = cu_q[i + 1] - cu_q[i], past = kv_lens[i] - n;
    }
  };
  const int r_shift = block_shift(R);   // (a division is half of a round of the bisection)
  auto by_rows = [&](int rows) __attribute__((always_inline)) { return r_shift >= 0 ? rows >> r_shift : rows / R; };
  // tiles whose last row's position is at least p, among the lane's sequence
  auto from = [&](int p) __attribute__((always_inline)) {
    const int nt = by_rows(n + R - 1);
    return nt - (past + n - 1 < p ? nt : min(by_rows(max(p - past, 0)), max(nt - 1, 0)));
  };
  auto over_all = [&](auto&& f) __attribute__((always_inline)) {  // (sums below 2^24: exact)
    int c = 0;
    for (int i = lane; i < n_seqs + lane; i += 64) {
      if (table) look(i);
      c += f();
    }
    return (int)wave_sum((float)c);
  };
  look(lane);
  int top = -1;
  for (int i = lane; i < n_seqs + lane; i += 64) {
    if (table) look(i);
    if (n > 0) top = max(top, past + n - 1);
  }
  const int last = (int)wave_max((float)top);   // (rounded beyond 2^24: hi only has to lie behind every position)
  int lo = 0, hi = last + 1 + (last >> 23), behind = 0;
  if (rank >= over_all([&] { return from(0); })) return false;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1, c = over_all([&] { return from(mid); });
    if (c > rank) lo = mid;
    else hi = mid, behind = c;
  }
  int k = rank - behind;
  for (int i0 = 0; i0 < n_seqs; i0 += 64) {
    look(i0 + lane);
    const int end = past + n - 1;
    uint64_t has = __ballot(n > 0 && (lo == end || (lo >= past && lo < end && (lo - past + 1) % R == 0)));
    const int c = __builtin_popcountll(has);
    if (k < c) {
      for (; k > 0; --k) has &= has - 1;
      const int at = __builtin_ctzll(has);
      s = i0 + at;
      first = cu_q[s] + (lo - __builtin_amdgcn_readlane(past, at)) / R * R;
      return true;
    }
    k -= c;
  }
  return false;
}

// up to 32 DKM key and 16 DVM value channels; smaller heads are zero-padded to that in the images: a branch per fragment would put
// every fragment's LDS latency behind the one before.  VIK: the values are the leading channels of the key rows.  PAGED16: pages
// of a multiple of 16 rows.  V4: value rows that start on 4 bytes only (bf16, an even stride), requested in 4-byte pieces.
// TWO: registers for two workgroups per CU (128; four of them spilled).
template <typename TC, int DKM, int DVM, int NST, bool VIK, bool PAGED16, bool V4 = false, bool TWO = false>
__global__ __launch_bounds__(kPromptThreads, TWO ? 4 : 2) void prompt_attention_kernel(
    const float* __restrict__ q, int64_t ldq, const TC* __restrict__ k_cache, const TC* __restrict__ v_cache,
    const int32_t* __restrict__ block_tables, int table_cols, const int32_t* __restrict__ cu_q,
    const int32_t* __restrict__ kv_lens, int n_seqs, int H, int G, int D, int Dv, int block_size, int window, float scale,
    AttnBias bias, int64_t ldv, const float* __restrict__ gate, int64_t ldg, float* __restrict__ out, int64_t ldo, bool longest_first) {
  constexpr bool BF = sizeof(TC) == 2;
  constexpr int VEC = 16 / (int)sizeof(TC);                 // channels of a 16-byte chunk
  constexpr int KROW = DKM * 32 * (int)sizeof(TC);          // bytes of a row in the image
  constexpr int VROW = VIK ? KROW : DVM * 16 * (int)sizeof(TC);
  constexpr int KB = kKeys * KROW, VB = VIK ? 0 : kKeys * VROW, STAGE = KB + VB;
  // LDS-DMA instructions of 1 KiB; PP per wave, all of one operand and of one half (16 keys) of the step
  constexpr int KP = KB / 1024, VP = VB / 1024, PP = (KP + VP + kWaves - 1) / kWaves <= 2 ? (KP + VP + kWaves - 1) / kWaves
                                                     : (KP + VP <= 32 ? 4 : 8);
  static_assert(!V4 || (BF && !VIK), "see above");
  static_assert(KP / 2 % PP == 0 && VP / 2 % PP == 0 && KP + VP <= PP * kWaves && (NST & (NST - 1)) == 0, "see above");
  static_assert(NST * STAGE >= kOrderedSeqs * 8, "the order's table");
  __shared__ __attribute__((aligned(1024))) char lds[NST * STAGE];
  // the chunk that lies at position p of row r is p ^ swizzle(r): sixteen rows at one chunk (a K fragment) and four or eight
  // rows at neighbouring chunks (a V fragment) fall into different banks
  auto swizzle = [](int r, int row_bytes) __attribute__((always_inline)) {
    if (!BF) return r & 15;
    return row_bytes == 128 ? (r >> 1) & 7 : ((r & 7) << 1) | ((r >> 3) & 1);
  };
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = blockIdx.y, hpg = H / G;
  const int Gv = bias.value_heads, gv = g / (G / Gv);
  const int h0 = blockIdx.z * kCols, nh = min(hpg - h0, kCols);   // heads of this kv head that the workgroup takes
  const int R = kCols / nh;                                       // rows of a tile
  int s = 0, first, nr;
  if (longest_first) {
    int2* const table = n_seqs > 64 ? reinterpret_cast<int2*>(lds) : nullptr;
    if (table) {
      for (int i = tid; i < n_seqs; i += kPromptThreads) {
        const int n = cu_q[i + 1] - cu_q[i];
        table[i] = int2{n, kv_lens[i] - n};
      }
      __syncthreads();
    }
    const bool found = tile_by_end(cu_q, kv_lens, table, n_seqs, R, (int)blockIdx.x, s, first);
    if (table) __syncthreads();   // (the ring's images lie there next)
    if (!found) return;  // (the grid is the host's bound)
    nr = min(R, cu_q[s + 1] - first);
  } else {
    // ---- the tile: sequences in order, a sequence's last rows (the longest walks) first ----
    int t = blockIdx.x, nt = 0;
    for (; s < n_seqs; ++s) {
      nt = (cu_q[s + 1] - cu_q[s] + R - 1) / R;
      if (t < nt) break;
      t -= nt;
    }
    if (s == n_seqs) return;  // (the grid is the host's bound)
    first = cu_q[s] + (nt - 1 - t) * R, nr = min(R, cu_q[s + 1] - first);
  }
  const int pos0 = kv_lens[s] - (cu_q[s + 1] - cu_q[s]) + (first - cu_q[s]);
  const int32_t* table = block_tables + (int64_t)s * table_cols;
  const int bs_shift = block_shift(block_size);
  // the walk: steps of 32 keys that start at multiples of 32 - the kept first keys that lie before the window, then the window
  const int lo_key = first_key(bias, pos0, window), hi_key = pos0 + nr - 1;
  const int kept_end = (min(bias.kept, lo_key) + kKeys - 1) & ~(kKeys - 1);
  const int win0 = max(lo_key & ~(kKeys - 1), kept_end);
  const int n_steps = kept_end / kKeys + (hi_key >= win0 ? (hi_key - win0) / kKeys + 1 : 0);
  auto next_step = [&](int u) { return u + kKeys == kept_end ? win0 : u + kKeys; };

  // ---- loading: a wave's pieces; a lane's row and chunk of each ----
  const int p0 = min(wave * PP, KP + VP - PP);   // (waves beyond the pieces repeat the last ones: the same bytes)
  const bool is_v = !VIK && p0 >= KP;
  const int first_row = (is_v ? p0 - KP : p0) * 1024 / (is_v ? VROW : KROW), half = first_row >> 4;
  const int heads = is_v ? Gv : G, head = is_v ? gv : g, ldr = is_v ? (int)ldv : D;
  const TC* const cache = is_v ? v_cache : k_cache;
  int prow[PP], pchan[PP], poff[PP];
  bool pok[PP];
#pragma unroll
  for (int i = 0; i < PP; ++i) {
    const int rb = is_v ? VROW : KROW, at = (is_v ? p0 - KP + i : p0 + i) * 1024 + lane * 16;
    prow[i] = at / rb;
    pchan[i] = ((at % rb / 16) ^ swizzle(prow[i], rb)) * VEC;
    pok[i] = pchan[i] < (is_v ? Dv : D);   // (chunks of the zero padding are not loaded)
    poff[i] = (prow[i] - 16 * half) * ldr + pchan[i];
  }
  if (D < 32 * DKM || (!VIK && Dv < 16 * DVM)) {
    for (int i = tid * 16; i < NST * STAGE; i += kPromptThreads * 16) *reinterpret_cast<u32x4*>(lds + i) = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();
  }
  // PAGED16: sixteen keys from a multiple of sixteen on lie in one page: one look-up per step for a wave, one step ahead.
  // Rows from the last key on repeat it (their weights are 0: no kernel reads a cache row its sequence has not written).
  int pg = 0;
  auto half_key = [&](int u) __attribute__((always_inline)) { return min(u + 16 * half, hi_key & ~15); };
  auto blk_of = [&](int key) __attribute__((always_inline)) { return bs_shift >= 0 ? key >> bs_shift : key / block_size; };
  auto look_up = [&](int u) __attribute__((always_inline)) {
    if (PAGED16) pg = table[blk_of(half_key(u))];
  };
  auto issue = [&](int u, int slot) __attribute__((always_inline)) {
    char* const dst = lds + slot * STAGE + p0 * 1024;
    auto dma = [&](const TC* src, int i) __attribute__((always_inline)) {
      if (pok[i])
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)(dst + i * 1024), 16, 0, 0);
    };
    const int k0 = half_key(u);   // (PAGED16)
    const TC* base = cache + ((int64_t)((uint32_t)pg * heads + head) * block_size + (k0 - blk_of(k0) * block_size)) * ldr;
    auto row_at = [&](int r) __attribute__((always_inline)) {   // row r of the step
      const int key = min(u + r, hi_key);
      return PAGED16 ? base + (key - k0) * ldr : cache + (int64_t)cache_row(table, key, heads, head, block_size, bs_shift) * ldr;
    };
    if (V4 && is_v) {
#pragma unroll
      for (int i = 0; i < PP * 4; ++i) {
        // (channels of the zero padding repeat the last ones, which nothing reads: a request without a lane, half a row beyond a head's
        // channels, would be branched over, and the waits below count on every one)
        const int at = (p0 - KP) * 1024 + i * 256 + lane * 4, r = at / VROW, c = ((at % VROW / 16) ^ swizzle(r, VROW)) * VEC + (at & 15) / 2;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(row_at(r) + min(c, Dv - 2)),
                                         (__attribute__((address_space(3))) void*)(dst + i * 256), 4, 0, 0);
      }
    } else if (PAGED16 && u + kKeys - 1 <= hi_key) {
#pragma unroll
      for (int i = 0; i < PP; ++i) dma(base + poff[i], i);
    } else {
#pragma unroll
      for (int i = 0; i < PP; ++i) dma(row_at(prow[i]) + pchan[i], i);
    }
  };

  // ---- computing: this lane's column ----
  const int r16 = lane & 15, kg = lane >> 4;
  const int col = wave * 16 + r16, crow = col / nh, ch = g * hpg + h0 + (col - crow * nh);
  const bool live = crow < nr;
  const int my_pos = pos0 + min(crow, nr - 1);
  const int my_lo = first_key(bias, my_pos, window);
  const int w_first = wave * 16 / nh, w_last = min((wave * 16 + 15) / nh, nr - 1);
  const bool w_live = w_first < nr;
  const int w_lo = first_key(bias, pos0 + min(w_first, nr - 1), window), w_hi = pos0 + w_last;
  // steps all of whose keys every one of the wave's columns sees: from w_in0 on, up to the wave's first row
  const int w_in0 = first_key(bias, pos0 + w_last, window), w_in1 = (wave * 16 + 15) / nh < nr ? pos0 + w_first : -1;
  const HeadBias hb = head_bias(bias, ch, H);
  constexpr int QK = BF ? DKM : 2 * DKM;                    // K fragments of a 16-key tile
  const int dk = BF ? D / 32 : D / 16, dvt = Dv / 16;
  bf16x8 qh[BF ? QK : 1], ql[BF ? QK : 1];
  f32x4 qf[BF ? 1 : QK];
  {
    const float* qp = q + (int64_t)(first + (live ? crow : 0)) * ldq + ch * D;
    const bool vec = (ldq % 4 == 0) && ((reinterpret_cast<uintptr_t>(q) & 15u) == 0);
    auto q4 = [&](int d) __attribute__((always_inline)) {
      if (!live) return f32x4{0.f, 0.f, 0.f, 0.f};
      if (vec) return *reinterpret_cast<const f32x4*>(qp + d);
      return f32x4{qp[d], qp[d + 1], qp[d + 2], qp[d + 3]};
    };
#pragma unroll
    for (int ks = 0; ks < QK; ++ks) {
      if constexpr (BF) {
        const f32x4 a = ks < dk ? q4(ks * 32 + kg * 8) : f32x4{0.f, 0.f, 0.f, 0.f};
        const f32x4 b = ks < dk ? q4(ks * 32 + kg * 8 + 4) : f32x4{0.f, 0.f, 0.f, 0.f};
        qh[ks] = as_frag(u32x4{pack_bf(a[0], a[1]), pack_bf(a[2], a[3]), pack_bf(b[0], b[1]), pack_bf(b[2], b[3])});
        ql[ks] = as_frag(u32x4{pack_bf(a[0] - rbf(a[0]), a[1] - rbf(a[1])), pack_bf(a[2] - rbf(a[2]), a[3] - rbf(a[3])),
                               pack_bf(b[0] - rbf(b[0]), b[1] - rbf(b[1])), pack_bf(b[2] - rbf(b[2]), b[3] - rbf(b[3]))});
      } else {
        qf[ks] = ks < dk ? q4(ks * 16 + kg * 4) : f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
  }
  // fragment addresses inside an image: K fragment ks of tile tt at kslot[ks & 3] + (ks >> 2) * 256 + tt * 16 rows; V (bf16): this
  // lane's 8 bytes of key row 4 kg + (r16 >> 2) at vslot ^ 32 (f & 7), + (f >> 3) * 256; V (fp32): key row 4 kg + e
  int kslot[4], vslot[BF ? 1 : 4];
#pragma unroll
  for (int i = 0; i < 4; ++i) kslot[i] = r16 * KROW + (((i * 4 + kg) ^ swizzle(r16, KROW)) << 4);
  if constexpr (BF) {
    const int r = 4 * kg + (r16 >> 2);
    vslot[0] = (VIK ? 0 : KB) + r * VROW + ((((r16 & 3) >> 1) ^ swizzle(r, VROW)) << 4) + (r16 & 1) * 8;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      vslot[e] = (VIK ? 0 : KB) + (4 * kg + e) * VROW + (((r16 >> 2) ^ swizzle(4 * kg + e, VROW)) << 4) + (r16 & 3) * 4;
  }
  float m = live ? -INFINITY : 0.f, l = 0.f;   // (a column without a row: all its weights are 0, and none of them asks for another point)
  f32x4 oacc[DVM];
#pragma unroll
  for (int f = 0; f < DVM; ++f) oacc[f] = f32x4{0.f, 0.f, 0.f, 0.f};

  int u0 = kept_end > 0 ? 0 : win0, ui = u0;   // the step that is computed, the next one to be requested
  look_up(ui);
#pragma unroll
  for (int i = 0; i < NST - 1; ++i)
    if (i < n_steps) {
      issue(ui, i);
      ui = next_step(ui);
      look_up(ui);
    }
  for (int k = 0; k < n_steps; ++k, u0 = next_step(u0)) {
    const int behind = min(n_steps - 1 - k, NST - 2);   // steps requested behind this one: their pieces may still fly
    if (V4 && is_v && NST > 2 && behind == 2) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(8 * PP) : "memory");
    else if (V4 && is_v && NST > 2 && behind == 1) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(4 * PP) : "memory");
    else if (NST > 2 && behind == 2) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * PP) : "memory");
    else if (NST > 2 && behind == 1) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PP) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (k + NST - 1 < n_steps) {   // (into the image everybody finished reading before the barrier)
      issue(ui, (k + NST - 1) & (NST - 1));
      ui = next_step(ui);
      look_up(ui);
    }
    // (waves whose rows see none of this step's keys only load)
    if (!(w_live && u0 <= w_hi && (u0 < bias.kept || u0 + kKeys > w_lo))) continue;
    const char* kb = lds + (k & (NST - 1)) * STAGE;
    // q's hi and lo parts have sums of their own: four independent chains
    f32x4 sacc[2], slow[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) sacc[tt] = f32x4{0.f, 0.f, 0.f, 0.f}, slow[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < QK; ++ks)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const u32x4 kv = *reinterpret_cast<const u32x4*>(kb + kslot[ks & 3] + (ks >> 2) * 256 + tt * 16 * KROW);
        if constexpr (BF) {
          sacc[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(kv), qh[ks], sacc[tt], 0, 0, 0);
          slow[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(kv), ql[ks], slow[tt], 0, 0, 0);
        } else {
          const f32x4 kf = __builtin_bit_cast(f32x4, kv);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            f32x4& s4 = e & 1 ? slow[tt] : sacc[tt];
            s4 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[e], qf[ks][e], s4, 0, 0, 0);
          }
        }
      }
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) sacc[tt] += slow[tt];
    // scores in units of ln 2: the weights are powers of two of them, m is their maximum
    float sc[8];
    const float d0 = (float)(my_pos - u0 - kg * 4);   // distance of the lane's first key; its others: 1, 2, 3 and 16..19 less
    // the bias kind is the same for the whole launch: a branch every wave takes the same way, so that the logarithms
    // are not evaluated (and thrown away) where the bias is linear or absent
    if (bias.kind == MI_BIAS_NONE && bias.softcap <= 0.f) {
#pragma unroll
      for (int e = 0; e < 8; ++e) sc[e] = sacc[e >> 2][e & 3] * (scale * kLog2e);
    } else if (bias.kind == MI_BIAS_SLOPE && bias.softcap <= 0.f) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        sc[e] = fmaf(sacc[e >> 2][e & 3], scale * kLog2e, -(hb.a * kLog2e) * (d0 - (float)((e >> 2) * 16 + (e & 3))));
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float dist = d0 - (float)((e >> 2) * 16 + (e & 3));
        float v = sacc[e >> 2][e & 3] * scale;
        if (bias.kind != MI_BIAS_NONE) v -= hb.log ? hb.a * log1pf(hb.b * fmaxf(dist, 0.f)) : hb.a * dist;
        sc[e] = capped(bias, v) * kLog2e;
      }
    }
    if (u0 < w_in0 || u0 + kKeys - 1 > w_in1) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int key = u0 + kg * 4 + (e >> 2) * 16 + (e & 3);
        const bool vis = live && key <= my_pos && (key >= my_lo || key < bias.kept);
        sc[e] = vis ? sc[e] : -INFINITY;
      }
    }
    // No maximum in the common case: a lane's eight weights against the current reference point add up to at most 2^8 while none of them is
    // larger (until a column has seen a key its point is -inf, the sum is not finite and the comparison fails).  Weights of up to 2^8 are held as
    // hi + lo, and in fp32, as those below 1 are.  (The maximum, its exchange and the rescaling were a third of a step's vector instructions.)
    float pv[8];
    auto weigh = [&](float ref) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < 8; ++e) pv[e] = __builtin_amdgcn_exp2f(sc[e] - ref);
      return ((pv[0] + pv[1]) + (pv[2] + pv[3])) + ((pv[4] + pv[5]) + (pv[6] + pv[7]));
    };
    float psum = weigh(m);
    if (__any(!(psum <= 256.f))) {
      float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
      mx = xor_max<32>(xor_max<16>(mx));
      const float m_new = fmaxf(m, mx);
      const float mref = m_new == -INFINITY ? 0.f : m_new;   // (a column that has seen nothing yet: its weights are 2^-inf = 0)
      const float corr = __builtin_amdgcn_exp2f(m - mref);
      psum = weigh(mref);
      l *= corr;
      m = m_new;
#pragma unroll
      for (int f = 0; f < DVM; ++f) oacc[f] *= corr;
    }
    l += psum;   // (the lane's share)
    if constexpr (BF) {
      u32x4 hi, lo;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        hi[i] = pack_bf(pv[2 * i], pv[2 * i + 1]);
        lo[i] = pack_bf(pv[2 * i] - lo_bf(hi[i]), pv[2 * i + 1] - hi_bf(hi[i]));
      }
      const bf16x8 ph = as_frag(hi), pl = as_frag(lo);
#pragma unroll
      for (int f = 0; f < DVM; ++f) {
        char* p = const_cast<char*>(kb) + (vslot[0] ^ (32 * (f & 7))) + (f >> 3) * 256;
        const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
        const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p + 16 * VROW));
        const u32x2 a2 = __builtin_bit_cast(u32x2, a), b2 = __builtin_bit_cast(u32x2, b);
        const bf16x8 vf = as_frag(u32x4{a2[0], a2[1], b2[0], b2[1]});
        oacc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, ph, oacc[f], 0, 0, 0);
        oacc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pl, oacc[f], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int f = 0; f < DVM; ++f)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float v = *reinterpret_cast<const float*>(kb + (vslot[e & 3] ^ (64 * (f & 3))) + (f >> 2) * 256 + (e >> 2) * 16 * VROW);
          oacc[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, pv[e], oacc[f], 0, 0, 0);
        }
    }
  }

  // the lane holds channels 16 f + 4 kg + {0..3} of its column
  l = xor_sum<32>(xor_sum<16>(l));
  const float inv = 1.f / (bias.sink ? l + __builtin_amdgcn_exp2f(bias.sink[ch] * kLog2e - m) : l);
  const int64_t row = first + crow;
  float* op = out + row * ldo + (int64_t)ch * Dv + kg * 4;
  const float* gp = gate ? gate + row * ldg + (int64_t)ch * Dv + kg * 4 : nullptr;
  const bool ovec = (ldo % 4 == 0) && ((reinterpret_cast<uintptr_t>(out) & 15u) == 0);
  const bool gvec = gate && (ldg % 4 == 0) && ((reinterpret_cast<uintptr_t>(gate) & 15u) == 0);
  f32x4 zero = {0.f, 0.f, 0.f, 0.f};   // (zero times the results: NaN where one of them is not finite)
#pragma unroll
  for (int f = 0; f < DVM; ++f) {
    if (live && f < dvt) {
      f32x4 o = oacc[f] * inv;
#pragma unroll
      for (int e = 0; e < 4; ++e) zero[e] = fmaf(oacc[f][e], 0.f, zero[e]);
      if (gate) {
        const f32x4 z = gvec ? *reinterpret_cast<const f32x4*>(gp + f * 16) : f32x4{gp[f * 16], gp[f * 16 + 1], gp[f * 16 + 2], gp[f * 16 + 3]};
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] *= sigmoid_f(z[e]);
      }
      if (ovec) {
        *reinterpret_cast<f32x4*>(op + f * 16) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) op[f * 16 + e] = o[e];
      }
    }
  }
  const float odd = (zero[0] + zero[1]) + (zero[2] + zero[3]);
  uint64_t todo = __ballot(live && odd != 0.f);
  if (__builtin_expect(todo == 0, 1)) return;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");   // (the columns above are home before they are written again)
  __builtin_amdgcn_wave_barrier();
  while (todo) {
    const int r = __builtin_ctzll(todo) & 15, cr = (wave * 16 + r) / nh, c_ch = g * hpg + h0 + (wave * 16 + r - cr * nh);
    todo &= ~(0x0001000100010001ull << r);   // (a column's four lanes)
    const int64_t at = first + cr;
    attend_column<TC>(q + at * ldq + (int64_t)c_ch * D, k_cache, v_cache, table, pos0 + cr, c_ch, H, G, D, Dv, block_size, window, scale, bias, ldv,
                      gate ? gate + at * ldg + (int64_t)c_ch * Dv : nullptr, out + at * ldo + (int64_t)c_ch * Dv);
  }
}

int launch_prompt_attention(const float* q, int64_t ldq, const void* k_cache, const void* v_cache, bool bf16, const int32_t* bt,
                            int cols, const int32_t* cu_q, const int32_t* kv_lens, int n_seqs, int rows, int H, int G, int D,
                            int Dv, int block_size, int window, float scale, const AttnBias& bias, int64_t ldv,
                            const float* gate, int64_t ldg, float* out, int64_t ldo, hipStream_t st) {
  const int vec = bf16 ? 8 : 4;
  if (D % (bf16 ? 32 : 16) || Dv % 16 || D > 256 || Dv > 256 || ldv % (bf16 ? 2 : vec) || !aligned16(k_cache) || !aligned16(v_cache) || G > 65535)
    return MI_EUNSUPPORTED;
  const int hpg = H / G, heads = hpg < kCols ? hpg : kCols, R = kCols / heads;
  const int64_t tiles = rows / R + n_seqs;
  if (tiles > 0x7fffffff || (hpg + kCols - 1) / kCols > 65535) return MI_EUNSUPPORTED;
  const dim3 grid((unsigned)tiles, G, (hpg + kCols - 1) / kCols);
  // Where there are more workgroups than the chip holds.  (Looking for the order takes 1 to 2 us of a workgroup, which like walks do not give back; unlike
  // ones do, also of sequences of a tile or less: us, sequence after sequence / longest first, 8 / 4 heads of 128, 361 sequences of 1 .. 63 rows behind 16
  // .. 1498 317 / 264, 16 / 8 heads of 64 on fp32 pages, 241 of 1 .. 339 574 / 466; 24 x 72 rows, 16 heads on as many 27.6 / 28.3.)
  const bool longest_first = tiles * G * grid.z > 512 && tiles < 1 << 24 && n_seqs <= kOrderedSeqs;   // (its sums are exact below 2^24)
  // us, the kernels before / this one: 8 x 1024 rows, 16 heads over one 256-channel row (values inside it) 917 / 271; 11 prompts,
  // 8112 rows, 8 / 4 heads x 128, window 512: 189 / 96; fp32 pages, 733 rows of 16 sequences behind up to 700: 760 / 83.  With K
  // and V through registers into the image (V transposed on the way): 345, 104, 86.
  const bool vik = k_cache == v_cache && bias.value_heads == G && ldv == D && Dv <= D;
  const bool paged16 = block_size % 16 == 0;
  // fp32 heads of more than 128 channels and a few dozen keys: 256 channels' padding and a ring of two cost more than the plain kernel's FMA
  // chains until the walk is longer (us, that one / here: 8 / 4 heads x 160, 40 rows 23 / 34, 100 rows 46 / 57, 200 rows faster here; 16
  // heads over one row of 256 channels 27 / 37, 100 rows 52 / 48; up to 32 keys are one step here: x 256, 30 rows 37 / 24)
  const int64_t keys = (int64_t)cols * block_size;   // (at most so many for any sequence)
  if (!bf16 && (D > 128 || Dv > 128) && keys > 32 && keys <= (vik ? 64 : 128) && rows > 32 * (int64_t)n_seqs) return MI_EUNSUPPORTED;
  // ... and of at most 32 channels, padded to 64, where there are too few tiles for the chip (8 / 4 heads x 32: 1 x 400 rows 36 / 40, 1 x 1600 140 /
  // 151; 4 x 1000 rows 171 / 115; x 16: 4 x 400 31 / 40, 4 x 1600 217 / 242)
  if (!bf16 && D <= 32 && Dv <= 32 && keys > 32 && tiles * G * grid.z <= (D <= 16 && Dv <= 16 ? 420 : 108)) return MI_EUNSUPPORTED;
  // fp32 heads of up to 64 channels: two workgroups per CU where the matrix pipe would wait for the one, but not where a few hundred uneven
  // walks would meet on some CUs and leave others idle, and not where one per CU is all there is (us, one / two, the rule's numbers in
  // brackets: 60 x 3 rows behind 500, 16 / 8 heads [496, alike] 86 / 57, 100 x 1 behind 600 and 300 rows, 8 / 4 [428, alike] 103 / 79, 13 x 225
  // (16 / 8) [464, alike] 56 / 42, 1 x 4539
  // (16 / 8) [568] 762 / 670, 16 x 1600 (16 / 8) [3328] 995 / 920; 12 x 481 (6 / 1) [286] 60 / 84, 1 x 7500 (6 / 1) [358] 690 / 819,
  // (8 / 4) [472] 900 / 1000, 14 up to 1370 (6 / 1) [537] 138 / 167; 30 x 30 behind 100 (32 / 4) [344, at least 224] 27 / 36; up to 256: 3 to 6 % more)
  const int64_t wgs = tiles * G * grid.z, least = std::max<int64_t>(rows / R, n_seqs) * G * grid.z;
  // (a tile per sequence, short prompts, or walks of the window's length)
  const bool alike = rows <= (int64_t)n_seqs * std::max(R, 256) || keys >= 2 * (int64_t)window;
  const bool two = !bf16 && (wgs > 540 || (least > 256 && alike));
#define MI_PROMPT(TC, DKM, DVM, NST, ...)                                                                                  \
  hipLaunchKernelGGL((prompt_attention_kernel<TC, DKM, DVM, NST, __VA_ARGS__>), grid, dim3(kPromptThreads), 0, st, q, ldq,    \
                     static_cast<const TC*>(k_cache), static_cast<const TC*>(v_cache), bt, cols, cu_q, kv_lens, n_seqs, H, G, D, Dv, \
                     block_size, window, scale, bias, ldv, gate, ldg, out, ldo, longest_first)
  // (WIDE: stages of the ring at 256 channels of keys and of values.  Pages of 24 rows, 400 rows of 4 sequences, 8 / 4 heads, us, the kernels
  // before / 256 channels for every head / by head size: fp32 x 64 72 / 177 / 43, x 128 144 / 183 / 79; bf16 x 64 46 / 46 / 21.)
#define MI_PROMPT_SIZES(TC, PAGED16, WIDE)                                   \
  do {                                                                       \
    if (two && D <= 64 && Dv <= 64) MI_PROMPT(TC, 2, 4, 4, false, PAGED16, false, sizeof(TC) == 4); \
    else if (D <= 64 && Dv <= 64) MI_PROMPT(TC, 2, 4, 4, false, PAGED16);    \
    else if (D <= 64 && Dv <= 128) MI_PROMPT(TC, 2, 8, 4, false, PAGED16);   \
    else if (D <= 128 && Dv <= 128) MI_PROMPT(TC, 4, 8, 4, false, PAGED16);  \
    else if (vik) MI_PROMPT(TC, 8, 16, 4, true, PAGED16);                    \
    else MI_PROMPT(TC, 8, 16, WIDE, false, PAGED16);                         \
  } while (0)
  if (bf16 && ldv % vec) {
    // value rows on 4 bytes (us, the kernel before / element by element / so: 8 x 1024 rows, 8 / 4 heads x 128, window 512 199 / 2440 / 85;
    // 4 x 1024 rows, 16 heads over one of 256 channels 428 / 3580 / 224; 4 x 300 rows, 8 / 4 heads x 64 and 48 34 / 165 / 18)
    if (!paged16) MI_PROMPT(uint16_t, 8, 16, 4, false, false, true);
    else if (D <= 64 && Dv <= 64) MI_PROMPT(uint16_t, 2, 4, 4, false, true, true);
    else if (D <= 128 && Dv <= 128) MI_PROMPT(uint16_t, 4, 8, 4, false, true, true);
    else MI_PROMPT(uint16_t, 8, 16, 4, false, true, true);
  } else if (bf16) {
    if (paged16) MI_PROMPT_SIZES(uint16_t, true, 4);
    else MI_PROMPT_SIZES(uint16_t, false, 4);
  } else {
    if (paged16) MI_PROMPT_SIZES(float, true, 2);
    else MI_PROMPT_SIZES(float, false, 2);
  }
#undef MI_PROMPT_SIZES
#undef MI_PROMPT
  return check_launch();
}

}  // namespace mi
