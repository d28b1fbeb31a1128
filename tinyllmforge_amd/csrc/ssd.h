// Arguments and helpers shared by the kernels of the state-space layer (ssd.hip, ssd_groups.hip).
#pragma once
#include "elem.h"

namespace tlf {

constexpr int kSsdMaxN = 512, kSsdMaxP = 512, kSC = 64;   // kSC: tokens per chunk

struct SsdArgs {
  const void *proj;        // [n, ld]
  Partials part;           // decode: or its partial sums
  int64_t ld;
  const void *conv, *conv_bias;              // [taps, channels], [channels]
  const void *dt_bias, *A_log, *D;           // [H]
  void *ring;              // [slots, taps, channels]
  float *state;            // [slots, H, N, P]
  const int32_t *state_slots;                // per sequence
  int32_t num_slots;
  const int64_t *positions;                  // per row
  const int32_t *row_seq, *cu_q, *starts;
  void *xbc;               // [rows, channels] activated
  float *dt, *decay;       // [rows, H]: step size, log2 of the decay
  void *out;               // [n, ldo]
  int64_t ldo;
  int32_t rows, H, P, N, G, taps, inner, channels;
  int32_t first_seq, seqs, first_row, segs, slices;
  int32_t begun;           // ssd_groups.hip: what the first pass goes through of a sequence, in 1/65536
  float *seg_state, *seg_decay;              // [seqs, segs, H, N, P], [seqs, segs, H]
};

template <typename T>
__device__ __forceinline__ float ssd_step(const SsdArgs &a, float raw, int h) {
  return softplus_f32(raw + Elem<T>::ld(static_cast<const T *>(a.dt_bias) + h));
}
template <typename T>
__device__ __forceinline__ float ssd_log2_decay(const SsdArgs &a, float dt, int h) {
  return -expf(Elem<T>::ld(static_cast<const T *>(a.A_log) + h)) * dt * 1.4426950408889634f;
}

// 32-bit rows: the library's exponential; bf16 rows: the hardware's, far more exact than the rounding that follows.
template <typename T>
__device__ __forceinline__ float ssd_silu(float z) {
  if constexpr (sizeof(T) == 4) return silu_f32(z);
  return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}

// Inclusive sum over the wave's 64 lanes, on the vector ALU.
template <int CTRL, int ROWS>
__device__ __forceinline__ float ssd_dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ float ssd_wave_scan(float v) {
  v = ssd_dpp_add<0x111, 0xf>(v);      // row_shr 1, 2, 4, 8: within rows of 16 lanes
  v = ssd_dpp_add<0x112, 0xf>(v);
  v = ssd_dpp_add<0x114, 0xf>(v);
  v = ssd_dpp_add<0x118, 0xf>(v);
  v = ssd_dpp_add<0x142, 0xa>(v);      // row_bcast 15 into rows 1 and 3
  return ssd_dpp_add<0x143, 0xc>(v);   // row_bcast 31 into rows 2 and 3
}

// ssd_groups.hip
int ssd_groups_segments(int H, int P, int N, int G, int seqs, int max_tokens, int dtype);   // 0: not for these sizes
int launch_ssd_groups(SsdArgs a, int max_tokens, hipStream_t stream);

}  // namespace tlf
