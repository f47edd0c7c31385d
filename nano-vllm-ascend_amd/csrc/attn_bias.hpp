// Bias, mask and paged addressing that the fp32-query attention kernels share (seqmix.hip, attn_prompt.hip).
#pragma once
#include "seqmix_common.hpp"

namespace mi {

// Distance bias of a score, taken off it: kind MI_BIAS_SLOPE: 2^(-8 (h + 1) / H) * dist (p1 == nullptr) or p1[h] * dist;
// MI_BIAS_LOG: p1[h] * ln(1 + p2[h] * dist); MI_BIAS_NONE: nothing.  ldv: elements between two tokens' value rows (Dv,
// or the key row's length when the values are the leading channels of the key rows of the same cache).
// sink != nullptr: a row's softmax normalises by sum_j exp(s_j) + exp(sink[h]): the extra term is a learned per-head
// logit taken as it is (the score scale does not touch it) that only soaks up weight - nothing is added to the output
// for it.
// softcap > 0: the scaled, biased score s becomes softcap * tanh(s / softcap) before the mask and the softmax.
// value_heads: the value cache has this many heads (a divisor of the key heads G; query head h reads value head
// h / (H / value_heads)) - fewer, wider value heads than key heads let every query head weigh the values of SEVERAL
// key/value heads at once (value rows holding the heads side by side), which is what mixing the heads' softmax weights
// afterwards needs.
// chunk > 0: position i sees the keys of its own chunk only (floor(i / chunk) = floor(j / chunk), positions counted from
// the sequence's start); with the window: both hold.
// kept > 0: the first `kept` keys of a sequence stay visible from everywhere behind them, whatever window and chunk say.
struct AttnBias {
  int kind;
  const float* p1;
  const float* p2;
  const float* sink;
  float softcap;
  int value_heads;
  int chunk;
  int kept;
};
// the oldest key position `pos` sees
__device__ __forceinline__ int first_key(const AttnBias& bias, int pos, int window) {
  int lo = max(0, pos - window + 1);
  if (bias.chunk > 0) lo = max(lo, pos - pos % bias.chunk);
  return lo;
}
// Kept keys lie away from the window: a walk over the keys counts u from lo - min(kept, lo) on, the u below lo stand for
// the kept keys that are older than lo (gap = lo - min(kept, lo) further down), the others for themselves - one run of
// numbers without holes, so that kept and window keys share the rounds of 32 / 64.  lo: the oldest key of the walk's first
// row by window and chunk.
__device__ __forceinline__ int kept_gap(const AttnBias& bias, int lo) { return lo - min(bias.kept, lo); }
template <bool KEEP>
__device__ __forceinline__ int key_at(int u, int lo, int gap) { return KEEP && u < lo ? u - gap : u; }
__device__ __forceinline__ float capped(const AttnBias& bias, float s) {
  return bias.softcap > 0.f ? bias.softcap * tanhf(s / bias.softcap) : s;
}
// the denominator of a finished row: its keys' sum l (relative to the running maximum m) plus the head's sink
__device__ __forceinline__ float with_sink(const AttnBias& bias, int h, float m, float l) {
  return bias.sink ? l + expf(bias.sink[h] - m) : l;
}
struct HeadBias {
  float a, b;
  bool log;
};
__device__ __forceinline__ HeadBias head_bias(const AttnBias& bias, int h, int H) {
  HeadBias r{0.f, 0.f, bias.kind == MI_BIAS_LOG};
  if (bias.kind == MI_BIAS_SLOPE) r.a = bias.p1 ? bias.p1[h] : exp2f(-8.f * (float)(h + 1) / (float)H);
  else if (bias.kind == MI_BIAS_LOG) r.a = bias.p1[h], r.b = bias.p2[h];
  return r;
}
__device__ __forceinline__ float dist_bias(const HeadBias& hb, int dist) {
  return hb.log ? hb.a * log1pf(hb.b * (float)dist) : hb.a * (float)dist;
}

// Row of a token in a paged cache [blocks][kv heads][block_size][.]: (table[key / block_size] * G + g) * block_size +
// key % block_size, in 32-bit arithmetic (rows of a cache are far fewer than 2^32; the byte offset is formed from it with
// one 32 x 32 -> 64-bit multiply-add), the division a shift when block_size is a power of two (bs_shift >= 0).
__device__ __forceinline__ int block_shift(int block_size) {
  return (block_size & (block_size - 1)) == 0 ? __builtin_ctz((unsigned)block_size) : -1;
}
__device__ __forceinline__ uint32_t cache_row(const int32_t* table, int key, int G, int g, int block_size, int bs_shift) {
  const int blk = bs_shift >= 0 ? key >> bs_shift : key / block_size;
  const int off = bs_shift >= 0 ? key & (block_size - 1) : key - blk * block_size;
  return ((uint32_t)table[blk] * (uint32_t)G + (uint32_t)g) * (uint32_t)block_size + (uint32_t)off;
}

// Prompt portions over paged K / V rows (attn_prompt.hip): MI_EUNSUPPORTED for head sizes or alignments it does not take.
int launch_prompt_attention(const float* q, int64_t ldq, const void* k_cache, const void* v_cache, bool bf16, const int32_t* bt,
                            int cols, const int32_t* cu_q, const int32_t* kv_lens, int n_seqs, int rows, int H, int G, int D,
                            int Dv, int block_size, int window, float scale, const AttnBias& bias, int64_t ldv,
                            const float* gate, int64_t ldg, float* out, int64_t ldo, hipStream_t st);

}  // namespace mi
