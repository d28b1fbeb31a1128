// Sigmoid attention over a window plus pooled blocks for prompt portions, bf16, on the matrix cores (geometry in
// pooled_attn.h).
//
// A workgroup owns one sequence, one KV head and a tile of query rows; the (row, head) pairs of the KV head's query
// heads are flattened into 128 units, 32 per wave (64 and 16 beyond 128 dimensions).  It walks the pooled rows its last query sees and then the
// tokens from its first query's window on; the loop is prompt_core.h's:
//   P = sigmoid(S * scale + bias)  fp32, masked on the pooled tiles and on those that a window's or the diagonal's edge cuts
// The weights are not normalised: no maximum, no rescaling, no second pass.  Bound by the vector ALU: two quarter-rate operations
// per score.  Eight prompts of 1061 to 2048 tokens, 32 heads of 128 on 8 KV heads, window 1024: layer 372 us with the stages of a tile
// one after the other (and the staging registers, which the compiler had put in LDS), 296 with three stages side by side, 286 - 293 in
// prompt_core.h's.
//
// Where rows of the projection can be read eight values at a time, queries and gates are made from them here, by the one workgroup that reads them
// (PROJ): 12240 tokens write and read 200 MB less, and a layer has two launches in place of three.  All bits are those of rows prepared on their own.
// Eight prompts as above 296 -> 266 us: under the profiler, least times, preparing took 54, pooling 13 and this 238; now keys, values and means
// take 22 (pooled_attn.hip: pooled_kv_kernel) and this 258: rows that come from memory instead of the caches, the norm, biases and rotation.  Three
// of the 30 are pages by scalar loads.  One prompt of up to 320 tokens 30 -> 22.  With the scale in the queries before they are rounded, and 2^-bias
// as a factor, a score takes an instruction less, 262 for 266; but results then are not those of prepared rows, and such a factor leaves the range of
// fp32 at a bias of -89.
#include "pooled_attn.h"
#include "prompt_core.h"
#include "prompt_tiles.h"

namespace tlf {

constexpr int kTK = 64;   // keys per tile

struct PooledPrefillArgs {
  PooledCache c;
  const unsigned short *q;     // [rows, H, Dp]
  const unsigned short *bias;  // [H]
  const float *gate;           // [rows, H]
  PooledProj proj;             // or what both are made from
  const int32_t *cu_q, *starts;
  unsigned short *out;
  int64_t ldo;
  int32_t H, group, hpp, passes;   // query heads, per KV head, per pass
  int32_t bq, first_seq;           // query rows per workgroup
  PromptTiles tiles;
  float scale_log2;
};

__device__ __forceinline__ int pooled_tile_row(int t) {
  return (t & 32) | ((t & 4) << 2) | ((t & 24) >> 1) | (t & 3);
}
__device__ __forceinline__ shortx4 pooled_read_tr16(const unsigned short *p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((shortx4 __attribute__((address_space(3))) *)(p));
}

template <int DC, int CT>
__device__ __forceinline__ void pooled_finish(const PooledPrefillArgs &p, const floatx4 (&acc)[CT][2 * DC], const bool (&uok)[CT], const int (&uoff)[CT], int g) {
  const PooledCache &c = p.c;
  const bool vec = (c.D & 3) == 0 && (p.ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 7) == 0;
#pragma unroll
  for (int k = 0; k < CT; ++k) {
    if (!uok[k]) continue;
    const float gt = p.gate[uoff[k]];
    const int row = uoff[k] / p.H, head = uoff[k] - row * p.H;
    unsigned short *o = p.out + static_cast<int64_t>(row) * p.ldo + static_cast<int64_t>(head) * c.D;
#pragma unroll
    for (int d = 0; d < 2 * DC; ++d) {
      const int col = d * 16 + g * 4;
      const uint2 v = make_uint2(pack_bf16x2(acc[k][d][0] * gt, acc[k][d][1] * gt), pack_bf16x2(acc[k][d][2] * gt, acc[k][d][3] * gt));
      if (vec) {
        if (col < c.D) *reinterpret_cast<uint2 *>(o + col) = v;
      } else {
        const unsigned int e[2] = {v.x, v.y};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (col + r < c.D) o[col + r] = static_cast<unsigned short>(e[r / 2] >> (16 * (r & 1)));
      }
    }
  }
}

template <int DC, bool PROJ>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void pooled_prefill_kernel(const PooledPrefillArgs p) {
  using Core = PromptCore<DC, DC>;
  __shared__ __attribute__((aligned(1024))) unsigned char Ks[2][Core::KB], Vs[2][Core::VB];
  int sq, plane, xt;
  if (!prompt_tile(p.tiles, prompt_block(blockIdx.x, blockIdx.y), sq, plane, xt)) return;
  const PooledCache &c = p.c;
  const int seq = p.first_seq + sq, kvh = plane / p.passes, pass = plane % p.passes;
  const int q0 = p.cu_q[seq], lq = p.cu_q[seq + 1] - q0, start = p.starts[seq];
  const int row0 = xt * p.bq;
  if (row0 >= lq) return;
  const int32_t *bt = c.bt + seq * c.bt_stride;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
  const int nh = min(p.hpp, p.group - pass * p.hpp);         // heads of this pass
  const int last_row = min(row0 + p.bq, lq) - 1;
  const int i_first = start + row0, i_last = start + last_row;

  Core core;
  core.start(TLF_DL_LDSADDR(Ks), TLF_DL_LDSADDR(Vs), tid);

  const int u = core.wave * 32 + n, r = row0 + u / p.hpp, hh = u % p.hpp;
  const bool uok = u < p.bq * p.hpp && r <= last_row && hh < nh;
  const int head = kvh * p.group + pass * p.hpp + (hh < nh ? hh : 0), row = uok ? r : row0;
  const int upos = start + row, unb = pooled_visible(upos, c.size, c.pool);
  const int64_t unit = static_cast<int64_t>(q0 + row) * p.H + head;
  const float pb = -kLog2e * bf16_bits_to_float(p.bias[head]), nscale = -p.scale_log2;
  const unsigned short *qp = PROJ ? p.proj.rows + static_cast<int64_t>(q0 + row) * p.proj.ld + head * c.D : p.q + unit * Core::DP;
  const int64_t pos = PROJ ? p.proj.positions[q0 + row] : 0;
  uint4 raw[2 * DC];                                         // of this lane's pieces of 8, every other one of the row
#pragma unroll
  for (int kc = 0; kc < 2 * DC; ++kc) raw[kc] = *reinterpret_cast<const uint4 *>(qp + (PROJ ? min(kc * 16 + g * 8, c.D - 8) : kc * 16 + g * 8));

  const int nb = pooled_visible(i_last, c.size, c.pool);
  const int ptiles = (nb + kTK - 1) / kTK;
  const int w0 = max(0, i_first - c.size + 1) / kTK * kTK;
  const int tiles = ptiles + (i_last - w0) / kTK + 1;
  const int64_t rs = static_cast<int64_t>(c.G) * Core::DP;
  const unsigned short *kc_ = static_cast<const unsigned short *>(c.k) + kvh * Core::DP;
  const unsigned short *vc_ = static_cast<const unsigned short *>(c.v) + kvh * Core::DP;
  const unsigned short *pk_ = static_cast<const unsigned short *>(c.pk) + kvh * Core::DP;
  const unsigned short *pv_ = static_cast<const unsigned short *>(c.pv) + kvh * Core::DP;

  unsigned int koff[DC], voff[DC];                           // this lane's pieces in a tile of tokens
#pragma unroll
  for (int i = 0; i < DC; ++i) {
    int at, piece;
    core.k_piece(i, lane, at, piece);
    koff[i] = static_cast<unsigned int>(at * static_cast<int>(rs) * 2 + piece * 16);
    core.v_piece(i, lane, at, piece);
    voff[i] = static_cast<unsigned int>(at * static_cast<int>(rs) * 2 + piece * 16);
  }
  // 64 tokens from a multiple of 64 on lie in one page, looked up a tile ahead by a scalar load: a vector load is waited for with the copies before it
  auto page_index = [&](int t) __attribute__((always_inline)) { return page_of(c, w0 + max(0, min(t, tiles - 1) - ptiles) * kTK); };
  int page_next = load_uniform(bt + page_index(0));
  auto copy = [&](int t, auto part) __attribute__((always_inline)) {
    if (part.lead && t < ptiles) {                           // rows of one page's blocks, then the next page's
#pragma unroll
      for (int i = 0; i < DC; ++i) {
        int at, piece;
        core.k_piece(i, lane, at, piece);
        prompt_copy_at(pk_ + block_row(c, bt, min(t * kTK + at, nb - 1)) * rs + piece * 8, core.k_place(t, i));
        core.v_piece(i, lane, at, piece);
        prompt_copy_at(pv_ + block_row(c, bt, min(t * kTK + at, nb - 1)) * rs + piece * 8, core.v_place(t, i));
      }
      return;
    }
    const int j = w0 + (t - ptiles) * kTK;                   // rows past the last query are masked
    const int64_t from = (page_next >= 0 && page_next < c.pages ? static_cast<int64_t>(page_next) * c.bs + (j - page_of(c, j) * c.bs) : 0) * rs;
    page_next = load_uniform(bt + page_index(t + 1));
#pragma unroll
    for (int i = 0; i < DC; ++i) prompt_copy(koff[i], kc_ + from, core.k_place(t, i));
#pragma unroll
    for (int i = 0; i < DC; ++i) prompt_copy(voff[i], vc_ + from, core.v_place(t, i));
  };
  if constexpr (PROJ) {
    float4 co[2 * DC], si[2 * DC];
#pragma unroll
    for (int kc = 0; kc < 2 * DC; ++kc) pooled_angles(p.proj, pos, kc * 2 + g, co[kc], si[kc]);
    copy(0, PromptPart<true, true>{});
    float x[2 * DC][8], ss[8];                               // sums of squares added up as 16 lanes with a piece each add them
#pragma unroll
    for (int kc = 0; kc < 8; ++kc) ss[kc] = 0.f;
#pragma unroll
    for (int kc = 0; kc < 2 * DC; ++kc) {
      const int col = kc * 16 + g * 8;
      unpack8(raw[kc], x[kc]);
      if (p.proj.q_bias) {
        float b[8];
        unpack8(*reinterpret_cast<const uint4 *>(p.proj.q_bias + head * c.D + min(col, c.D - 8)), b);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[kc][e] += b[e];
      }
      pooled_rotate(x[kc], co[kc], si[kc]);
      if (col >= c.D) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[kc][e] = 0.f;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) ss[kc] = fmaf(x[kc][e], x[kc][e], ss[kc]);
      ss[kc] = prompt_unit_sum(ss[kc]);
    }
    const float sum = ((ss[0] + ss[1]) + (ss[2] + ss[3])) + ((ss[4] + ss[5]) + (ss[6] + ss[7]));
    const float inv = 1.0f / sqrtf(sum / static_cast<float>(c.D) + p.proj.eps);
#pragma unroll
    for (int kc = 0; kc < 2 * DC; ++kc) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[kc][e] *= inv;
      raw[kc] = pack8(x[kc]);
    }
  } else {
    copy(0, PromptPart<true, true>{});
  }
#pragma unroll
  for (int kc = 0; kc < 2 * DC; ++kc) core.qf[kc] = __builtin_bit_cast(bf16x8, raw[kc]);
  // tiles between the window's edge and the diagonal hide nothing from anyone
  const int last = i_last - w0 + ptiles * kTK, edge0 = i_first - c.size + 1 - w0 + ptiles * kTK;      // of the keys in the window, counted as tiles are
  const int edge = i_last - c.size >= w0 ? (i_last - c.size - w0) / kTK + 1 : 0;
  core.template walk<true, false>(
      tiles, 0, tiles, ptiles + edge, min(tiles, ptiles + max(0, (i_first + 1 - w0) / kTK)), copy,
      [&](int t, int hf, auto part) __attribute__((always_inline)) {
        const int at = t * kTK + hf * 32;
        if (part.lead && t < ptiles) return at < nb;
        return at <= last && (!part.lead || at + 31 >= edge0);
      },
      []() __attribute__((always_inline)) { return Core::all(0.f); },
      [&](int t, int hf, const typename Core::Scores &s, typename Core::Weights &w, auto part) __attribute__((always_inline)) {
        float e[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) e[j] = sigmoid_neg_log2(fmaf(s[j], nscale, pb));
        if (part.mask) {
          const bool pooled = part.lead && t < ptiles;       // workgroup uniform
          const int key = t * kTK + hf * 32 + (pooled ? 0 : w0 - ptiles * kTK) + g * 8;
          const int lo = part.lead && !pooled ? upos - c.size + 1 : 0, hi = (pooled ? unb : upos + 1) - key;
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const int at = (j & 8) * 2 + (j & 7);
            e[j] = at < hi && (!part.lead || at >= lo - key) ? e[j] : 0.f;
          }
        }
        Core::split(e, w);
      });

  if (!uok) return;
  const float gt = PROJ ? sigmoid_f32(bf16_bits_to_float(p.proj.rows[static_cast<int64_t>(q0 + row) * p.proj.ld + static_cast<int64_t>(p.H + c.G) * c.D + head])) : p.gate[unit];
  unsigned short *o = p.out + static_cast<int64_t>(q0 + row) * p.ldo + static_cast<int64_t>(head) * c.D;
  const uintptr_t to = reinterpret_cast<uintptr_t>(p.out);
  core.store(o, c.D, (c.D & 3) == 0 && (p.ldo & 3) == 0 && (to & 7) == 0, (c.D & 7) == 0 && (p.ldo & 7) == 0 && (to & 15) == 0, g,
             [&](int, float (&f)[4]) __attribute__((always_inline)) {
#pragma unroll
               for (int x = 0; x < 4; ++x) f[x] *= gt;
             });
}

// Heads beyond 128: the stages of a tile one after the other, staged through registers, one tile in LDS at a time.
template <int DC, int CT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void pooled_prefill_wide_kernel(const PooledPrefillArgs p) {
  constexpr int DP = DC * 32, NCH = DC * 4;
  __shared__ __attribute__((aligned(16))) unsigned short Ks[kTK][DP + 8], Vs[kTK][DP + 16];
  int sq, plane, xt;
  if (!prompt_tile(p.tiles, prompt_block(blockIdx.x, blockIdx.y), sq, plane, xt)) return;
  const PooledCache &c = p.c;
  const int seq = p.first_seq + sq, kvh = plane / p.passes, pass = plane % p.passes;
  const int q0 = p.cu_q[seq], lq = p.cu_q[seq + 1] - q0, start = p.starts[seq];
  const int row0 = xt * p.bq;
  if (row0 >= lq) return;
  const int32_t *bt = c.bt + seq * c.bt_stride;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int nh = min(p.hpp, p.group - pass * p.hpp);         // heads of this pass
  const int last_row = min(row0 + p.bq, lq) - 1;
  const int i_first = start + row0, i_last = start + last_row;

  int upos[CT], unb[CT], uoff[CT];
  bool uok[CT];
  float pb[CT];
  bf16x8 qf[CT][DC];
#pragma unroll
  for (int k = 0; k < CT; ++k) {
    const int u = wave * CT * 16 + k * 16 + n;
    const int r = row0 + u / p.hpp, hh = u % p.hpp;
    uok[k] = u < p.bq * p.hpp && r <= last_row && hh < nh;
    const int head = kvh * p.group + pass * p.hpp + (hh < nh ? hh : 0);
    const int row = uok[k] ? r : row0;
    upos[k] = start + row;
    unb[k] = pooled_visible(upos[k], c.size, c.pool);
    uoff[k] = (q0 + row) * p.H + head;
    pb[k] = -kLog2e * bf16_bits_to_float(p.bias[head]);
    const unsigned short *qp = p.q + static_cast<int64_t>(uoff[k]) * DP + g * 8;
#pragma unroll
    for (int kc = 0; kc < DC; ++kc) {
      Pack16 t;
      t.u = *reinterpret_cast<const uint4 *>(qp + kc * 32);
      qf[k][kc] = t.v;
    }
  }
  const float nscale = -p.scale_log2;

  const int nb = pooled_visible(i_last, c.size, c.pool), nb_first = pooled_visible(i_first, c.size, c.pool);
  const int ptiles = (nb + kTK - 1) / kTK;
  const int w0 = max(0, i_first - c.size + 1) / kTK * kTK;
  const int tiles = ptiles + (i_last - w0) / kTK + 1;
  const int64_t rs = static_cast<int64_t>(c.G) * DP;
  const unsigned short *kc_ = static_cast<const unsigned short *>(c.k) + kvh * DP;
  const unsigned short *vc_ = static_cast<const unsigned short *>(c.v) + kvh * DP;
  const unsigned short *pk_ = static_cast<const unsigned short *>(c.pk) + kvh * DP;
  const unsigned short *pv_ = static_cast<const unsigned short *>(c.pv) + kvh * DP;

  uint4 kreg[DC], vreg[DC];
#pragma unroll
  for (int i = 0; i < DC; ++i) kreg[i] = vreg[i] = make_uint4(0, 0, 0, 0);   // keeps the arrays in registers: without it the compiler puts them in LDS
  auto load_tile = [&](int t) __attribute__((always_inline)) {
    if (t < ptiles) {
#pragma unroll
      for (int i = 0; i < DC; ++i) {
        const int item = tid + i * 256, r = item / NCH, ch = item % NCH;
        const int64_t o = block_row(c, bt, min(t * kTK + r, nb - 1)) * rs + ch * 8;
        kreg[i] = *reinterpret_cast<const uint4 *>(pk_ + o);
        vreg[i] = *reinterpret_cast<const uint4 *>(pv_ + o);
      }
    } else {
      // 64 tokens from a multiple of 64 on lie in one page; rows past the last query are masked
      const int j0 = w0 + (t - ptiles) * kTK;
      const int64_t base = token_row(c, bt, j0) * rs;
#pragma unroll
      for (int i = 0; i < DC; ++i) {
        const int item = tid + i * 256, r = item / NCH, ch = item % NCH;
        const int64_t o = base + r * rs + ch * 8;
        kreg[i] = *reinterpret_cast<const uint4 *>(kc_ + o);
        vreg[i] = *reinterpret_cast<const uint4 *>(vc_ + o);
      }
    }
  };
  auto store_tile = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < DC; ++i) {
      const int item = tid + i * 256, r = item / NCH, ch = item % NCH;
      *reinterpret_cast<uint4 *>(&Ks[pooled_tile_row(r)][ch * 8]) = kreg[i];
      *reinterpret_cast<uint4 *>(&Vs[r][ch * 8]) = vreg[i];
    }
  };

  floatx4 acc[CT][2 * DC];
#pragma unroll
  for (int k = 0; k < CT; ++k)
#pragma unroll
    for (int d = 0; d < 2 * DC; ++d) acc[k][d] = floatx4{0.f, 0.f, 0.f, 0.f};

  load_tile(0);
  store_tile();
  lds_barrier();
  for (int t = 0; t < tiles; ++t) {
    const bool more = t + 1 < tiles;
    if (more) load_tile(t + 1);
    const bool pooled = t < ptiles;
    const int k0 = pooled ? t * kTK : w0 + (t - ptiles) * kTK;
    const bool need_mask = pooled ? k0 + kTK > nb_first : (k0 + kTK - 1 > i_first || k0 <= i_last - c.size);
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      floatx4 s0[CT], s1[CT];
#pragma unroll
      for (int k = 0; k < CT; ++k) s0[k] = s1[k] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < DC; ++kc) {
        Pack16 a0, a1;
        a0.u = *reinterpret_cast<const uint4 *>(&Ks[hf * 32 + n][kc * 32 + g * 8]);
        a1.u = *reinterpret_cast<const uint4 *>(&Ks[hf * 32 + n + 16][kc * 32 + g * 8]);
#pragma unroll
        for (int k = 0; k < CT; ++k) {
          s0[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0.v, qf[k][kc], s0[k], 0, 0, 0);
          s1[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1.v, qf[k][kc], s1[k], 0, 0, 0);
        }
      }
      // lane (n, g) of column tile k holds keys k0 + hf * 32 + g * 8 + j
      uint4 ph[CT], pl[CT];
#pragma unroll
      for (int k = 0; k < CT; ++k) {
        float w[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j] = sigmoid_neg_log2(fmaf(j < 4 ? s0[k][j & 3] : s1[k][j & 3], nscale, pb[k]));
        if (need_mask) {  // workgroup uniform
          const int key = k0 + hf * 32 + g * 8;
          const int lo = pooled ? 0 : upos[k] - c.size + 1, hi = pooled ? unb[k] : upos[k] + 1;
#pragma unroll
          for (int j = 0; j < 8; ++j) w[j] = key + j >= lo && key + j < hi ? w[j] : 0.f;
        }
        unsigned int h[4], l[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) weight_pairs(w[2 * j], w[2 * j + 1], h[j], l[j]);
        ph[k] = make_uint4(h[0], h[1], h[2], h[3]);
        pl[k] = make_uint4(l[0], l[1], l[2], l[3]);
      }
      const int vt = hf * 32 + g * 8 + (n >> 2);
#pragma unroll
      for (int d = 0; d < 2 * DC; ++d) {
        const shortx4 v0 = pooled_read_tr16(&Vs[vt][d * 16 + (n & 3) * 4]);
        const shortx4 v1 = pooled_read_tr16(&Vs[vt + 4][d * 16 + (n & 3) * 4]);
        const bf16x8 vb = __builtin_bit_cast(bf16x8, make_uint4(__builtin_bit_cast(uint2, v0).x, __builtin_bit_cast(uint2, v0).y,
                                                               __builtin_bit_cast(uint2, v1).x, __builtin_bit_cast(uint2, v1).y));
#pragma unroll
        for (int k = 0; k < CT; ++k) {
          acc[k][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb, __builtin_bit_cast(bf16x8, ph[k]), acc[k][d], 0, 0, 0);
          acc[k][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb, __builtin_bit_cast(bf16x8, pl[k]), acc[k][d], 0, 0, 0);
        }
      }
    }
    lds_barrier();
    if (more) {
      store_tile();
      lds_barrier();
    }
  }

  pooled_finish<DC, CT>(p, acc, uok, uoff, g);
}

namespace {
int launch_pooled_prefill(PooledPrefillArgs &a, int num_seqs, int max_tokens, hipStream_t s) {
  const PooledCache &c = a.c;
  const int dc = c.Dp / 32, ct = dc <= 4 ? 2 : 1, units = 64 * ct;
  a.group = a.H / c.G;
  a.hpp = a.group < units ? a.group : units;
  a.passes = (a.group + a.hpp - 1) / a.hpp;
  a.bq = units / a.hpp;
  const int blocks = prompt_tiles_make(a.tiles, (max_tokens + a.bq - 1) / a.bq, c.G * a.passes, num_seqs);
  const dim3 grid = prompt_grid<dim3>(blocks);
  if (!blocks) return TLF_E_SHAPE;
#define TLF_POOLED(DC)                                                                             \
  do {                                                                                             \
    if (a.proj.rows) TLF_LAUNCH((pooled_prefill_kernel<DC, true>), grid, dim3(256), 0, s, a);      \
    else TLF_LAUNCH((pooled_prefill_kernel<DC, false>), grid, dim3(256), 0, s, a);                 \
  } while (0)
  switch (dc) {
    case 1: TLF_POOLED(1); break;
    case 2: TLF_POOLED(2); break;
    case 3: TLF_POOLED(3); break;
    case 4: TLF_POOLED(4); break;
    case 5: TLF_LAUNCH((pooled_prefill_wide_kernel<5, 1>), grid, dim3(256), 0, s, a); break;
    case 6: TLF_LAUNCH((pooled_prefill_wide_kernel<6, 1>), grid, dim3(256), 0, s, a); break;
    case 7: TLF_LAUNCH((pooled_prefill_wide_kernel<7, 1>), grid, dim3(256), 0, s, a); break;
    default: TLF_LAUNCH((pooled_prefill_wide_kernel<8, 1>), grid, dim3(256), 0, s, a); break;
  }
#undef TLF_POOLED
  return launch_status();
}
}  // namespace

}  // namespace tlf

extern "C" int tlf_pooled_attn_prefill(const void *q, const void *score_bias, const float *gate, const void *k_cache,
                                       const void *v_cache, const void *pk_cache, const void *pv_cache,
                                       const int32_t *block_tables, int64_t bt_stride, const int32_t *cu_seqlens_q,
                                       const int32_t *seq_starts, int32_t first_seq, int32_t num_seqs,
                                       int32_t max_tokens, void *out, int64_t out_stride, int32_t num_q_heads,
                                       int32_t num_kv_heads, int32_t head_dim, int32_t block_size, int32_t pool,
                                       int32_t window, int64_t num_pages, float scale, void *stream) {
  using namespace tlf;
  if (num_seqs < 0 || max_tokens < 0 || first_seq < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads)
    return TLF_E_SHAPE;
  if (out_stride < static_cast<int64_t>(num_q_heads) * head_dim) return TLF_E_SHAPE;
  if (num_seqs == 0 || max_tokens == 0) return TLF_OK;
  PooledCache c{k_cache, v_cache, pk_cache, pv_cache, block_tables, bt_stride, block_size, pool, 0, window,
                num_kv_heads, head_dim, (head_dim + 31) / 32 * 32, num_pages, -1};
  if (int rc = pooled_cache_check(c, TLF_DT_BF16)) return rc;
  if (!q || !score_bias || !gate || !cu_seqlens_q || !seq_starts || !out) return TLF_E_NULL;
  if (!aligned16(q)) return TLF_E_ALIGN;
  pooled_cache_finish(c);
  PooledPrefillArgs a{c, static_cast<const unsigned short *>(q), static_cast<const unsigned short *>(score_bias), gate, {},
                      cu_seqlens_q, seq_starts, static_cast<unsigned short *>(out), out_stride, num_q_heads,
                      0, 0, 0, 0, first_seq, {}, scale * kLog2e};
  return launch_pooled_prefill(a, num_seqs, max_tokens, static_cast<hipStream_t>(stream));
}

extern "C" int tlf_pooled_attn_portions(const void *proj, int64_t proj_stride, const void *q_bias, const void *k_bias, const int64_t *positions,
                                        const float *cos_sin, int32_t max_pos, int32_t rot_dims, const int32_t *slot_mapping, const void *score_bias,
                                        void *k_cache, void *v_cache, void *pk_cache, void *pv_cache, const int32_t *block_tables, int64_t bt_stride,
                                        const int32_t *cu_seqlens_q, const int32_t *seq_starts, int32_t first_seq, int32_t num_seqs, int32_t max_tokens,
                                        void *out, int64_t out_stride, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
                                        int32_t pool, int32_t window, int64_t num_pages, float scale, float eps, void *stream) {
  using namespace tlf;
  if (num_seqs < 0 || num_seqs > 65535 || max_tokens < 0 || first_seq < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads)
    return TLF_E_SHAPE;
  if (out_stride < static_cast<int64_t>(num_q_heads) * head_dim) return TLF_E_SHAPE;
  if (num_seqs == 0 || max_tokens == 0) return TLF_OK;
  PooledCache c{k_cache, v_cache, pk_cache, pv_cache, block_tables, bt_stride, block_size, pool, 0, window,
                num_kv_heads, head_dim, (head_dim + 31) / 32 * 32, num_pages, -1};
  if (int rc = pooled_cache_check(c, TLF_DT_BF16)) return rc;
  if (rot_dims < 0 || rot_dims % 2 || rot_dims > head_dim) return TLF_E_SHAPE;
  if (proj_stride < static_cast<int64_t>(num_q_heads + num_kv_heads) * head_dim + num_q_heads) return TLF_E_SHAPE;
  if (!proj || !positions || (rot_dims && !cos_sin) || !slot_mapping || !score_bias || !cu_seqlens_q || !seq_starts || !out) return TLF_E_NULL;
  pooled_cache_finish(c);
  const PooledProj p{static_cast<const unsigned short *>(proj), proj_stride, static_cast<const unsigned short *>(q_bias),
                     static_cast<const unsigned short *>(k_bias), positions, cos_sin, max_pos, rot_dims, eps};
  if (!pooled_proj_takes(p, head_dim)) return TLF_E_UNSUPPORTED;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (int rc = launch_pooled_kv(c, p, slot_mapping, cu_seqlens_q, seq_starts, first_seq, num_seqs, max_tokens, num_q_heads, s)) return rc;
  PooledPrefillArgs a{c, nullptr, static_cast<const unsigned short *>(score_bias), nullptr, p,
                      cu_seqlens_q, seq_starts, static_cast<unsigned short *>(out), out_stride, num_q_heads,
                      0, 0, 0, 0, first_seq, {}, scale * kLog2e};
  return launch_pooled_prefill(a, num_seqs, max_tokens, s);
}
