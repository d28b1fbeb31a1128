// Latent attention of long prompt portions, bf16, on the matrix cores, from keys and values expanded per head (geometry in
// latent_attn.h): row r of `expanded` holds the keys' own parts of all heads and then the values, the rotated key part
// shared by the heads is read from the gathered cache rows.
//
// A workgroup owns one portion, one head and 128 query rows, 32 per wave, and walks the keys its window covers; the loop is
// prompt_core.h's:
//   P = 2^(S * scale - m)         fp32; m follows a row's maximum only when that has grown by more than 8 (a factor of 256,
//                                 which the fp32 sums and the bf16 pair hold), so the accumulators are rarely rescaled.  Whether any
//                                 has grown is asked lane by lane; maxima of rows are only formed when one has, and all rows of the wave
//                                 follow theirs then: a largest weight of 1 is not rounded
// 16 heads of 96 and 64 dimensions, eight prompts of 1061 to 2048 tokens: layer 189 us with the stages of a tile one after the other and
// a window of 1024, 171 with three stages side by side, 162 so; three waves per SIMD fit the registers (160 to 165 with two, 160 with three).
#include "latent_attn.h"
#include "prompt_core.h"
#include "prompt_tiles.h"

namespace tlf {

constexpr int kPK = kPromptKeys;      // keys per tile

struct LatentPrefillArgs {
  LatentShape s;
  const unsigned short *q;          // [rows, H, Dq]
  const unsigned short *expanded;   // [kv rows, lde]: H * Da, then H * Va
  const unsigned short *latents;    // [kv rows, Lp]
  const int32_t *cu_q, *starts, *kv_off;
  const float *gate;                // [rows, H] or NULL
  unsigned short *out;              // [rows, ldo]
  int64_t lde, ldo;
  PromptTiles tiles;
  int32_t first_seq, window, by_heads;
  float scale_log2;                 // positive; the sign (or zero) of the scale goes into q
  unsigned int q_keep, q_flip;
};

// Portions of one row tile: the heads take the place of row tiles, so that a sequence's rows, of which every head has a part, are read and
// written by one XCD, one sequence after the other (64 portions of 128 tokens: layer, 16 heads 81 -> 78 us, 12 heads 80 -> 69).
__device__ __forceinline__ bool latent_tile(const LatentPrefillArgs &p, int &sq, int &h, int &xt) {
  if (!prompt_tile(p.tiles, prompt_block(blockIdx.x, blockIdx.y), sq, h, xt)) return false;
  if (p.by_heads) {
    h = xt;
    xt = 0;
  }
  return true;
}

template <int VC, int CT>
__device__ __forceinline__ void latent_finish(const LatentPrefillArgs &p, const floatx4 (&acc)[CT][2 * VC], const float (&l)[CT], const bool (&uok)[CT],
                                              const int (&upos)[CT], int q0, int start, int h, int g) {
  const LatentShape &s = p.s;
  const bool vec = (s.vdim & 3) == 0 && (p.ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 7) == 0;
#pragma unroll
  for (int k = 0; k < CT; ++k) {
    const float den = sum_lanes_16_32_48(l[k]);
    if (!uok[k]) continue;
    float inv = 1.0f / den;                                  // a row sees itself: den > 0
    if (p.gate) inv *= p.gate[static_cast<int64_t>(q0 + upos[k] - start) * s.H + h];
    unsigned short *o = p.out + static_cast<int64_t>(q0 + upos[k] - start) * p.ldo + static_cast<int64_t>(h) * s.vdim;
#pragma unroll
    for (int d = 0; d < 2 * VC; ++d) {
      const int col = d * 16 + g * 4;
      const uint2 v = make_uint2(pack_bf16x2(acc[k][d][0] * inv, acc[k][d][1] * inv), pack_bf16x2(acc[k][d][2] * inv, acc[k][d][3] * inv));
      if (vec) {
        if (col < s.vdim) *reinterpret_cast<uint2 *>(o + col) = v;
      } else {
        const unsigned int e[2] = {v.x, v.y};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (col + r < s.vdim) o[col + r] = static_cast<unsigned short>(e[r / 2] >> (16 * (r & 1)));
      }
    }
  }
}

// DC, VC: query / key and value dimensions in units of 32 (rounded up to what is instantiated)
template <int DC, int VC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DC + VC <= 5 ? 3 : 2))) void latent_prefill_kernel(const LatentPrefillArgs p) {
  using Core = PromptCore<DC, VC>;
  __shared__ __attribute__((aligned(1024))) unsigned char Ks[2][Core::KB], Vs[2][Core::VB];
  int sq, h, xt;
  if (!latent_tile(p, sq, h, xt)) return;
  const LatentShape &s = p.s;
  const int seq = p.first_seq + sq;
  const int q0 = p.cu_q[seq], lq = p.cu_q[seq + 1] - q0, start = p.starts[seq];
  const int row0 = xt * 128;
  if (row0 >= lq) return;
  const int kv0 = p.kv_off[sq], kv_n = p.kv_off[sq + 1] - kv0;
  const int kbase = max(0, start - p.window + 1);            // position of the portion's first dense row
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
  const int last_row = min(row0 + 128, lq) - 1;
  const int i_first = start + row0, i_last = start + last_row;
  Core core;
  core.start(TLF_DL_LDSADDR(Ks), TLF_DL_LDSADDR(Vs), tid);
  const int wave_first = i_first + core.wave * 32, wave_last = min(wave_first + 31, i_last);

  const int r = row0 + core.wave * 32 + n, row = min(r, last_row), upos = start + row;
  const bool uok = r <= last_row;
  const unsigned short *qp = p.q + (static_cast<int64_t>(q0 + row) * s.H + h) * s.Dq + g * 8;
#pragma unroll
  for (int kc = 0; kc < 2 * DC; ++kc) {
    Pack16 t;
    t.u = kc * 16 < s.Dq ? *reinterpret_cast<const uint4 *>(qp + kc * 16) : make_uint4(0, 0, 0, 0);
    t.u = make_uint4((t.u.x & p.q_keep) ^ p.q_flip, (t.u.y & p.q_keep) ^ p.q_flip, (t.u.z & p.q_keep) ^ p.q_flip, (t.u.w & p.q_keep) ^ p.q_flip);
    core.qf[kc] = t.v;
  }

  // This lane's pieces of a tile's rows: their places in the row 0 of the portion's dense rows, their rows in the tile.  A piece of K
  // is of the own part or of the rotated one; the pads of a row meet zeros of the queries and repeat its first piece.
  const unsigned char *kat[DC];
  int krow[DC], vrow[VC];
  unsigned int kstep[DC], vat[VC];
  const unsigned short *own = p.expanded + static_cast<int64_t>(kv0) * p.lde, *turned = p.latents + static_cast<int64_t>(kv0) * s.Lp + s.Ra - s.Da;
  const unsigned int ostep = static_cast<unsigned int>(p.lde * 2), tstep = static_cast<unsigned int>(s.Lp * 2);
#pragma unroll
  for (int i = 0; i < DC; ++i) {
    int piece;
    core.k_piece(i, lane, krow[i], piece);
    const int d = piece * 8 < s.Da + s.Ta ? piece * 8 : 0;
    kat[i] = reinterpret_cast<const unsigned char *>(d < s.Da ? own + h * s.Da + d : turned + d);
    kstep[i] = d < s.Da ? ostep : tstep;
  }
#pragma unroll
  for (int i = 0; i < VC; ++i) {
    int piece;
    core.v_piece(i, lane, vrow[i], piece);
    vat[i] = piece * 8 < s.Va ? piece * 16 : 0;
  }
  const int w0 = max(0, i_first - p.window + 1);             // >= kbase
  const int tiles = (i_last - w0) / kPK + 1;
  auto copy = [&](int t, auto) __attribute__((always_inline)) {
    const int r0 = w0 - kbase + t * kPK;                     // its own row is below kv_n
#pragma unroll
    for (int i = 0; i < DC; ++i)
      prompt_copy_at(kat[i] + static_cast<uint64_t>(kstep[i]) * static_cast<unsigned int>(min(r0 + krow[i], kv_n - 1)), core.k_place(t, i));
    const unsigned short *base = own + static_cast<int64_t>(r0) * p.lde + s.H * s.Da + h * s.Va;
#pragma unroll
    for (int i = 0; i < VC; ++i)
      prompt_copy(ostep * static_cast<unsigned int>(min(vrow[i], kv_n - 1 - r0)) + vat[i], base, core.v_place(t, i));
  };

  float m = -INFINITY, l = 0.f;                              // no key yet
  // tiles between the window's edge and the diagonal hide nothing from any of the wave's rows
  const int to = max(0, wave_last - w0) / kPK + 1;
  const int edge = wave_last - p.window >= w0 ? (wave_last - p.window - w0) / kPK + 1 : 0;
  copy(0, PromptPart<true, true>{});
  core.template walk<true, true>(
      tiles, min(max(0, wave_first - p.window + 1 - w0) / kPK, to - 1), to, edge, min(tiles, max(0, (wave_first + 1 - w0) / kPK)), copy,
      [&](int t, int hf, auto) __attribute__((always_inline)) { return t * kPK + hf * 32 <= wave_last - w0; }, []() __attribute__((always_inline)) { return Core::all(0.f); },
      [&](int t, int hf, typename Core::Scores &sc, typename Core::Weights &w, auto part) __attribute__((always_inline)) {
        if (part.mask) {
          const int seen = upos - (w0 + t * kPK + hf * 32 + g * 8), hidden = seen - p.window;
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const int at = (j & 8) * 2 + (j & 7);
            sc[j] = at <= seen && (!part.lead || at > hidden) ? sc[j] : -INFINITY;
          }
        }
        const float x = Core::largest(sc) * p.scale_log2;
        if (__any(x > m + 8.f)) {                            // sums and accumulators to the new maximum
          const float most = fmaxf(m, prompt_unit_max(x));
          const float back = most == m ? 1.f : __builtin_amdgcn_exp2f(m - most);
          m = most;
          l *= back;
          core.rescale(back);
        }
        const float ms = m == -INFINITY ? 0.f : m;
        float e[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) e[j] = __builtin_amdgcn_exp2f(sc[j] * p.scale_log2 - ms);
        l += Core::sum(e);
        Core::split(e, w);
      });

  const float den = prompt_unit_sum(l);
  if (!uok) return;
  float inv = 1.0f / den;                                    // a row sees itself: den > 0
  if (p.gate) inv *= p.gate[static_cast<int64_t>(q0 + row) * s.H + h];
  unsigned short *o = p.out + static_cast<int64_t>(q0 + row) * p.ldo + static_cast<int64_t>(h) * s.vdim;
  const uintptr_t at = reinterpret_cast<uintptr_t>(p.out);
  core.store(o, s.vdim, (s.vdim & 3) == 0 && (p.ldo & 3) == 0 && (at & 7) == 0, (s.vdim & 7) == 0 && (p.ldo & 7) == 0 && (at & 15) == 0, g,
             [&](int, float (&f)[4]) __attribute__((always_inline)) {
#pragma unroll
               for (int i = 0; i < 4; ++i) f[i] *= inv;
             });
}

__device__ __forceinline__ int prefill_tile_row(int t) { return (t & 32) | ((t & 4) << 2) | ((t & 24) >> 1) | (t & 3); }
__device__ __forceinline__ shortx4 prefill_read_tr16(const unsigned short *p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((shortx4 __attribute__((address_space(3))) *)(p));
}

// Queries beyond 128: the stages of a tile one after the other, a tile staged through registers, one in LDS at a time.  The shared loop
// does not fit the registers with two units per lane, and with one the reads of K and V out of LDS bound it (192 and 128 dimensions,
// 32 heads, eight prompts of 1061 to 2048 tokens: layer 585 us, 687 with the shared loop and spills, 615 with one unit per lane).
template <int DC, int VC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void latent_prefill_wide_kernel(const LatentPrefillArgs p) {
  constexpr int CT = 2, kPQ = 64 * CT, DP = DC * 32, VP = VC * 32;
  __shared__ __attribute__((aligned(16))) unsigned short Ks[kPK][DP + 8], Vs[kPK][VP + 16];
  int sq, h, xt;
  if (!latent_tile(p, sq, h, xt)) return;
  const LatentShape &s = p.s;
  const int seq = p.first_seq + sq;
  const int q0 = p.cu_q[seq], lq = p.cu_q[seq + 1] - q0, start = p.starts[seq];
  const int row0 = xt * kPQ;
  if (row0 >= lq) return;
  const int kv0 = p.kv_off[sq], kv_n = p.kv_off[sq + 1] - kv0;
  const int kbase = max(0, start - p.window + 1);            // position of the portion's first dense row
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int last_row = min(row0 + kPQ, lq) - 1;
  const int i_first = start + row0, i_last = start + last_row;
  const int wave_first = i_first + wave * 32, wave_last = min(wave_first + 31, i_last);

  int upos[CT];
  bool uok[CT];
  bf16x8 qf[CT][DC];
#pragma unroll
  for (int k = 0; k < CT; ++k) {
    const int r = row0 + wave * 32 + k * 16 + n;
    uok[k] = r <= last_row;
    const int row = uok[k] ? r : last_row;
    upos[k] = start + row;
    const unsigned short *qp = p.q + (static_cast<int64_t>(q0 + row) * s.H + h) * s.Dq + g * 8;
#pragma unroll
    for (int kc = 0; kc < DC; ++kc) {
      Pack16 t;
      t.u = kc * 32 < s.Dq ? *reinterpret_cast<const uint4 *>(qp + kc * 32) : make_uint4(0, 0, 0, 0);
      t.u = make_uint4((t.u.x & p.q_keep) ^ p.q_flip, (t.u.y & p.q_keep) ^ p.q_flip, (t.u.z & p.q_keep) ^ p.q_flip, (t.u.w & p.q_keep) ^ p.q_flip);
      qf[k][kc] = t.v;
    }
  }

  // four threads copy a row of a tile, every fourth piece of 8 each: own part, rotated part or zeros; then the value
  const int tr = tid >> 2, td = (tid & 3) * 8;
  uint4 kreg[DC], vreg[VC];
  auto load_tile = [&](int k0) __attribute__((always_inline)) {
    const int64_t row = kv0 + min(k0 - kbase + tr, kv_n - 1);
    const unsigned short *er = p.expanded + row * p.lde, *kr = er + h * s.Da, *vr = er + s.H * s.Da + h * s.Va;
    const unsigned short *lr = p.latents + row * s.Lp + s.Ra - s.Da;
#pragma unroll
    for (int i = 0; i < DC; ++i) {
      const int d = td + i * 32;
      kreg[i] = make_uint4(0, 0, 0, 0);
      if (d < s.Da + s.Ta) kreg[i] = *reinterpret_cast<const uint4 *>((d < s.Da ? kr : lr) + d);
    }
#pragma unroll
    for (int i = 0; i < VC; ++i) {
      const int d = td + i * 32;
      vreg[i] = make_uint4(0, 0, 0, 0);
      if (d < s.Va) vreg[i] = *reinterpret_cast<const uint4 *>(vr + d);
    }
  };
  const int kw = prefill_tile_row(tr);
  auto store_tile = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < DC; ++i) *reinterpret_cast<uint4 *>(&Ks[kw][td + i * 32]) = kreg[i];
#pragma unroll
    for (int i = 0; i < VC; ++i) *reinterpret_cast<uint4 *>(&Vs[tr][td + i * 32]) = vreg[i];
  };

  floatx4 acc[CT][2 * VC];
  float m[CT], l[CT];
#pragma unroll
  for (int k = 0; k < CT; ++k) {
    m[k] = -INFINITY;
    l[k] = 0.f;
#pragma unroll
    for (int d = 0; d < 2 * VC; ++d) acc[k][d] = floatx4{0.f, 0.f, 0.f, 0.f};
  }

  const int w0 = max(0, i_first - p.window + 1);             // >= kbase
  const int tiles = (i_last - w0) / kPK + 1;
  load_tile(w0);
  store_tile();
  lds_barrier();
  for (int t = 0; t < tiles; ++t) {
    const bool more = t + 1 < tiles;
    const int k0 = w0 + t * kPK;
    if (more) load_tile(k0 + kPK);
    if (k0 <= wave_last && k0 + kPK - 1 > wave_first - p.window) {   // wave uniform: some row sees some key
      const bool need_mask = k0 + kPK - 1 > wave_first || k0 <= wave_last - p.window;
      float w[CT][2][8];
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
#pragma unroll
        for (int k = 0; k < CT; ++k) {
#pragma unroll
          for (int j = 0; j < 8; ++j) w[k][hf][j] = (j < 4 ? s0[k][j & 3] : s1[k][j & 3]) * p.scale_log2;
          if (need_mask) {
            const int key = k0 + hf * 32 + g * 8;
#pragma unroll
            for (int j = 0; j < 8; ++j) w[k][hf][j] = key + j <= upos[k] && key + j > upos[k] - p.window ? w[k][hf][j] : -INFINITY;
          }
        }
      }
      float mt[CT];
      bool grown = false;
#pragma unroll
      for (int k = 0; k < CT; ++k) {
        float x = w[k][0][0];
#pragma unroll
        for (int j = 1; j < 16; ++j) x = fmaxf(x, w[k][j >> 3][j & 7]);
        mt[k] = max_lanes_16_32_48(x);
        grown = grown || mt[k] > m[k] + 8.f;
      }
      if (__any(grown)) {
#pragma unroll
        for (int k = 0; k < CT; ++k) {
          const float mn = fmaxf(m[k], mt[k]);
          const float back = mn == m[k] ? 1.f : __builtin_amdgcn_exp2f(m[k] - mn);
          m[k] = mn;
          l[k] *= back;
#pragma unroll
          for (int d = 0; d < 2 * VC; ++d) acc[k][d] *= back;
        }
      }
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        uint4 ph[CT], pl[CT];
#pragma unroll
        for (int k = 0; k < CT; ++k) {
          const float ms = m[k] == -INFINITY ? 0.f : m[k];
          float e[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) e[j] = __builtin_amdgcn_exp2f(w[k][hf][j] - ms);
          l[k] += ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
          unsigned int hi[4], lo[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) weight_pairs(e[2 * j], e[2 * j + 1], hi[j], lo[j]);
          ph[k] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
          pl[k] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        }
        const int vt = hf * 32 + g * 8 + (n >> 2);
#pragma unroll
        for (int d = 0; d < 2 * VC; ++d) {
          const uint2 v0 = __builtin_bit_cast(uint2, prefill_read_tr16(&Vs[vt][d * 16 + (n & 3) * 4]));
          const uint2 v1 = __builtin_bit_cast(uint2, prefill_read_tr16(&Vs[vt + 4][d * 16 + (n & 3) * 4]));
          const bf16x8 vb = __builtin_bit_cast(bf16x8, make_uint4(v0.x, v0.y, v1.x, v1.y));
#pragma unroll
          for (int k = 0; k < CT; ++k) {
            acc[k][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb, __builtin_bit_cast(bf16x8, ph[k]), acc[k][d], 0, 0, 0);
            acc[k][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb, __builtin_bit_cast(bf16x8, pl[k]), acc[k][d], 0, 0, 0);
          }
        }
      }
    }
    lds_barrier();
    if (more) {
      store_tile();
      lds_barrier();
    }
  }

  latent_finish<VC, CT>(p, acc, l, uok, upos, q0, start, h, g);
}

inline int fit_units(int units) { return units <= 4 ? units : units <= 6 ? 6 : 8; }   // of 32, as instantiated

}  // namespace tlf

extern "C" int tlf_latent_prefill_supported(int32_t heads, int32_t dim, int32_t rot_dim, int32_t rank, int32_t vdim) {
  tlf::LatentShape s;
  return tlf::latent_shape(s, heads, dim, rot_dim, rank, vdim) && s.Dq <= 256 && vdim <= 128;
}

extern "C" int tlf_latent_prefill(const void *q, const void *expanded, int64_t expanded_stride, const void *latents,
                                  const int32_t *cu_seqlens_q, const int32_t *seq_starts, const int32_t *kv_offsets,
                                  int32_t first_seq, int32_t num_seqs, int32_t max_tokens, const float *gate, void *out, int64_t out_stride,
                                  int32_t heads, int32_t dim, int32_t rot_dim, int32_t rank, int32_t vdim, int32_t window,
                                  float scale, void *stream) {
  using namespace tlf;
  LatentPrefillArgs a{};
  if (num_seqs < 0 || max_tokens < 0 || first_seq < 0 || window <= 0 || !latent_shape(a.s, heads, dim, rot_dim, rank, vdim)) return TLF_E_SHAPE;
  if (a.s.Dq > 256 || vdim > 128) return TLF_E_UNSUPPORTED;
  if (expanded_stride < static_cast<int64_t>(heads) * (a.s.Da + a.s.Va) || expanded_stride % 8 || out_stride < static_cast<int64_t>(heads) * vdim) return TLF_E_SHAPE;
  if (num_seqs == 0 || max_tokens == 0) return TLF_OK;
  if (!q || !expanded || !latents || !cu_seqlens_q || !seq_starts || !kv_offsets || !out) return TLF_E_NULL;
  if (!aligned16(q) || !aligned16(expanded) || !aligned16(latents)) return TLF_E_ALIGN;
  a.q = static_cast<const unsigned short *>(q); a.expanded = static_cast<const unsigned short *>(expanded);
  a.latents = static_cast<const unsigned short *>(latents); a.cu_q = cu_seqlens_q; a.starts = seq_starts; a.kv_off = kv_offsets;
  a.out = static_cast<unsigned short *>(out); a.lde = expanded_stride; a.ldo = out_stride; a.first_seq = first_seq;
  a.gate = gate; a.window = window; a.scale_log2 = scale == 0.f ? 1.f : fabsf(scale) * 1.4426950408889634f;
  a.q_keep = scale == 0.f ? 0u : ~0u; a.q_flip = scale < 0.f ? 0x80008000u : 0u;
  const int dc = fit_units(a.s.Dq / 32), vc = (vdim + 31) / 32;
  constexpr int rows = 128;
  a.by_heads = max_tokens <= rows;
  const int blocks = a.by_heads ? prompt_tiles_make(a.tiles, heads, 1, num_seqs, 1) : prompt_tiles_make(a.tiles, (max_tokens + rows - 1) / rows, heads, num_seqs);
  const dim3 grid = prompt_grid<dim3>(blocks);
  if (!blocks) return TLF_E_SHAPE;
  hipStream_t st = static_cast<hipStream_t>(stream);
#define TLF_LP(DC, VC) TLF_LAUNCH((latent_prefill_kernel<DC, VC>), grid, dim3(256), 0, st, a)
#define TLF_LW(DC, VC) TLF_LAUNCH((latent_prefill_wide_kernel<DC, VC>), grid, dim3(256), 0, st, a)
#define TLF_LP_V(KERNEL, DC)          \
  case DC:                            \
    if (vc == 1) KERNEL(DC, 1);       \
    else if (vc == 2) KERNEL(DC, 2);  \
    else KERNEL(DC, 4);               \
    break;
  switch (dc) {
    TLF_LP_V(TLF_LP, 1) TLF_LP_V(TLF_LP, 2) TLF_LP_V(TLF_LP, 3) TLF_LP_V(TLF_LP, 4) TLF_LP_V(TLF_LW, 6) TLF_LP_V(TLF_LW, 8)
    default: return TLF_E_UNSUPPORTED;
  }
#undef TLF_LP_V
#undef TLF_LW
#undef TLF_LP
  return launch_status();
}
