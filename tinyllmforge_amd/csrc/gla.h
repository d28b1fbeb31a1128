// Arguments shared by the kernels of gated linear attention (gla.hip, gla_blocks.hip).
#pragma once
#include "elem.h"

namespace tlf {

constexpr int kGlaMaxDk = 256, kGlaMaxDv = 512, kGlaMaxR = 256;

struct GlaArgs {
  const void *proj;        // [n, ld]
  Partials part;           // decode: or its partial sums
  int64_t ld;
  const void *a2;          // [H * dk, R]
  const void *a2_bias;     // [H * dk]
  const void *norm_w;      // [dv]
  float *state;            // [slots, H, dk, dv]
  const int32_t *state_slots;
  int32_t num_slots;
  const int64_t *positions;   // decode: [rows]
  void *out;               // [n, ldo]
  int64_t ldo;
  int32_t rows, H, dk, dv, R;
  float inv_tau, q_scale, eps;
  // portions
  const int32_t *chunk_tok, *chunk_len;   // [chunks]: first row of the chunk in the step, tokens in it
  const int32_t *cu_chunks;               // [seqs + 1]
  const int32_t *starts;                  // [seqs]: tokens before this step, 0: the state starts at zero
  int32_t chunks, seqs;
  // workspace.  One record per (chunk, head): Qd, Kd, A, decays, 64 floats of padding (records a power of two apart
  // would fall into few sets of the L2); o: [chunks, H, 16, dv]
  float *rec, *o;
  int32_t vec;                            // bf16 projection rows may be read 8 bytes at a time, key dim a full row
  int32_t segs;                           // segments per sequence
  float *seg_state, *seg_dec;             // [seqs, segs, H, dk, dv], [seqs, segs, H, DKP]; of stretches (gla_blocks.hip): [2, units, H, ..], [units, H, ..]
  int32_t units;                          // stretches of all sequences' blocks, 0: whole sequences
  int32_t seq0;                           // sequences of the call before the first of these
};

// log2 of sigmoid(z)^(1/tau) = -(max(-z, 0) log2 e + log2(1 + e)) / tau with e = 2^(-|z| log2 e).  log2(1 + e) keeps its
// relative accuracy for small e: the rounding of u = 1 + e is undone by the factor e / (u - 1).
__device__ __forceinline__ float log2_alpha(float z, float inv_tau) {
  const float kL2e = 1.4426950408889634f;
  const float e = __builtin_amdgcn_exp2f(-fabsf(z) * kL2e);
  const float u = 1.0f + e, d = u - 1.0f;
  const float l = d == 0.f ? e * kL2e : __builtin_amdgcn_logf(u) * e * __builtin_amdgcn_rcpf(d);
  return -fmaf(fmaxf(-z, 0.f), kL2e, l) * inv_tau;
}

// Prompt portions in blocks of 32 tokens (gla_blocks.hip): what it takes, its workspace, the launches.
bool gla_blocks_take(const GlaArgs &a, int32_t dtype, int chunk_segs);     // chunk_segs: segments the chunks would have
bool gla_blocks_sizes(int32_t key_dim, int32_t value_dim);
size_t gla_blocks_workspace_bytes(int32_t chunks, int32_t num_seqs, int32_t heads, int32_t key_dim, int32_t value_dim);
int launch_gla_blocks(GlaArgs &a, int first_seq, int longest, void *workspace, hipStream_t stream);

}  // namespace tlf
