// Device helpers shared by the sequence-mixer kernels (seqmix.hip, stream_delta.hip).
#pragma once
#include "mi_common.hpp"

namespace mi {

__device__ __forceinline__ float sigmoid_f(float z) { return 1.f / (1.f + expf(-z)); }
__device__ __forceinline__ float softplus_f(float z) { return z > 20.f ? z : log1pf(expf(z)); }

template <typename T>
__device__ __forceinline__ float ld_f(const T* p);
template <>
__device__ __forceinline__ float ld_f<float>(const float* p) { return *p; }
template <>
__device__ __forceinline__ float ld_f<uint16_t>(const uint16_t* p) { return bf2f(*p); }
template <typename T>
__device__ __forceinline__ void st_f(T* p, float v);
template <>
__device__ __forceinline__ void st_f<float>(float* p, float v) { *p = v; }
template <>
__device__ __forceinline__ void st_f<uint16_t>(uint16_t* p, float v) { *p = f2bf(v); }

// sum over a 256-thread workgroup; every thread gets the result.  red: 4 floats of LDS per concurrent reduction.
__device__ __forceinline__ float block_sum256(float v, float* red) {
  v = wave_sum(v);
  __syncthreads();  // (red may still be read from the previous reduction)
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// the sequence a step row belongs to (n_seqs is small: a linear walk, identical on every lane)
__device__ __forceinline__ int seq_of_row(const int32_t* cu_q, int n_seqs, int row) {
  int s = 0;
  while (s + 1 < n_seqs && row >= cu_q[s + 1]) ++s;
  return s;
}

// Read-out norm of the recurrences (seqmix.hip), in place: every head's Dv channels to unit rms, times norm_w [Dv], times sigmoid(gate)
// with a gate.
int launch_head_norm(float* out, int64_t ldo, const float* gate_pre, int64_t ld_gate, const float* norm_w, int n_rows, int H, int Dv,
                     float eps, hipStream_t st);

// mi_linear_attention's recurrence sixteen rows at a time (delta_blocks.hip): out [rows][H * Dv] before the read-out's norm.  MI_EUNSUPPORTED
// for what the blocks do not take.
int launch_linear_blocks(const float* proj, int64_t ld, int q_off, int k_off, int v_off, int q_act, int k_act, int v_act, int decay_kind,
                         const float* decay, const float* f_bias, const float* lower, float* state, const int32_t* cu_q,
                         const int32_t* kv_lens, const int32_t* slot_ids, int n_seqs, int n_rows, int H, int D, int Dv, float* workspace,
                         int64_t ws_elems, float* out, int64_t ldo, hipStream_t st);

}  // namespace mi
