// Geometry shared by the kernels of windowed attention with pooled blocks (pooled_attn.hip, pooled_prefill.hip).
//
// A query at position i sees the tokens j with 0 <= i - j < size and one mean key / mean value for every block of
// `pool` consecutive tokens that lies wholly before that window.  Token rows live in the paged K/V cache; the means
// live in a second paged cache with the same page numbers: a page of `bs` tokens owns C = ceil(bs / pool) mean rows,
// and a block's row is in the page of its last token.
#pragma once
#include "elem.h"

namespace tlf {

struct PooledCache {
  const void *k, *v;    // [pages, bs, G, Dp]
  const void *pk, *pv;  // [pages, C, G, Dp]
  const int32_t *bt;    // block tables, one row per sequence
  int64_t bt_stride;
  int32_t bs, pool, C, size;
  int32_t G, D, Dp;     // KV heads, head dimension, padded head dimension (a multiple of 32; pads hold zeros)
  int64_t pages;
  int32_t bs_shift;     // log2 of bs, -1 if it is no power of two
};
inline void pooled_cache_finish(PooledCache &c) {
  c.C = (c.bs + c.pool - 1) / c.pool;
  c.bs_shift = (c.bs & (c.bs - 1)) == 0 ? __builtin_ctz(c.bs) : -1;
}
__device__ __forceinline__ int page_of(const PooledCache &c, int j) { return c.bs_shift >= 0 ? j >> c.bs_shift : j / c.bs; }

// Blocks visible to position i.
__device__ __forceinline__ int pooled_visible(int i, int size, int pool) {
  const int past = i - size + 1;
  return past > 0 ? past / pool : 0;
}
// Cache row (units of G * Dp elements) of token j and of block b; an unmapped page reads row 0 (never visible).
__device__ __forceinline__ int64_t token_row(const PooledCache &c, const int32_t *bt, int j) {
  const int pg = page_of(c, j);
  const int64_t page = bt[pg];
  const bool ok = page >= 0 && page < c.pages;
  return ok ? page * c.bs + (j - pg * c.bs) : 0;
}
__device__ __forceinline__ int64_t block_row(const PooledCache &c, const int32_t *bt, int b) {
  const int pg = page_of(c, b * c.pool + c.pool - 1);
  const int64_t page = bt[pg];
  const bool ok = page >= 0 && page < c.pages;
  return ok ? page * c.C + (b - (pg * c.bs) / c.pool) : 0;
}

// Mean of the rows of block b, one KV head, written to the pooled cache: work item t of 2 * Dp / 8 (K chunks, then V).
template <typename T>
__device__ __forceinline__ void pool_block_chunk(const PooledCache &c, const int32_t *bt, int b, int kvh, int t) {
  const int nch = c.Dp / 8;
  const bool is_v = t >= nch;
  const int ch = is_v ? t - nch : t;
  const T *src = static_cast<const T *>(is_v ? c.v : c.k) + kvh * c.Dp + ch * 8;
  const int64_t rs = static_cast<int64_t>(c.G) * c.Dp;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int r = 0; r < c.pool; ++r) {
    float f[8];
    Elem<T>::ld8(src + token_row(c, bt, b * c.pool + r) * rs, f);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += f[e];
  }
  const float inv = 1.0f / static_cast<float>(c.pool);
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] *= inv;
  T *dst = static_cast<T *>(const_cast<void *>(is_v ? c.pv : c.pk)) + kvh * c.Dp + ch * 8;
  Elem<T>::st8(dst + block_row(c, bt, b) * rs, acc);
}

// Unnormalised attention weight sigmoid(score), argument in units of log 2 with the sign already flipped.
__device__ __forceinline__ float sigmoid_neg_log2(float neg_score_log2) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(neg_score_log2));
}
constexpr float kLog2e = 1.4426950408889634f;

int pooled_cache_check(const PooledCache &c, int32_t dtype);

// What turns rows of a bf16 projection [q heads | k heads | a gate value per q head] into queries, keys and values.
struct PooledProj {
  const unsigned short *rows;   // [n, ld]
  int64_t ld;
  const unsigned short *q_bias, *k_bias;     // NULL: none
  const int64_t *positions;
  const float *cos_sin;         // [max_pos, rot_dims]: cos of the pairs, then sin
  int32_t max_pos, rot_dims;
  float eps;
};
// Whether rows are read eight values at a time.
inline bool pooled_proj_takes(const PooledProj &p, int32_t head_dim) {
  return head_dim % 8 == 0 && head_dim <= 128 && p.rot_dims % 8 == 0 && p.ld % 8 == 0 && aligned16(p.rows) && aligned16(p.q_bias) && aligned16(p.k_bias) &&
         aligned16(p.cos_sin);
}
// Keys, values and pooled rows of portions (pooled_attn.hip); of p, what keys are made from.
int launch_pooled_kv(const PooledCache &c, const PooledProj &p, const int32_t *slots, const int32_t *cu_q, const int32_t *starts, int first_seq, int num_seqs,
                     int max_tokens, int H, hipStream_t stream);
// The pairs of dimensions 8 ch .. 8 ch + 7 turned, each product rounded as in rows that are prepared on their own: a token's key has the same bits
// whichever way its step was cut.
__device__ __forceinline__ void pooled_rotate(float (&x)[8], const float4 &co, const float4 &si) {
  const float cv[4] = {co.x, co.y, co.z, co.w}, sv[4] = {si.x, si.y, si.z, si.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float u = x[2 * e], v = x[2 * e + 1];
    x[2 * e] = __fmul_rn(u, cv[e]) - __fmul_rn(v, sv[e]);
    x[2 * e + 1] = __fmul_rn(v, cv[e]) + __fmul_rn(u, sv[e]);
  }
}
__device__ __forceinline__ void pooled_angles(const PooledProj &p, int64_t pos, int ch, float4 &co, float4 &si) {
  co = make_float4(1.f, 1.f, 1.f, 1.f);
  si = make_float4(0.f, 0.f, 0.f, 0.f);
  if (pos >= 0 && pos < p.max_pos && ch * 8 < p.rot_dims) {
    const float *cs = p.cos_sin + pos * p.rot_dims + ch * 4;
    co = *reinterpret_cast<const float4 *>(cs);
    si = *reinterpret_cast<const float4 *>(cs + p.rot_dims / 2);
  }
}

}  // namespace tlf
