// The loop that the prompt kernels of sink_prefill.hip, pooled_prefill.hip and latent_prefill.hip share: bf16, on the matrix cores.
//
// A workgroup of four waves has 64 CT units, a query row of one head each, 16 CT per wave, and walks its keys in tiles of 64:
//   S^T[key, unit] = K . Q^T         v_mfma_f32_16x16x32_bf16
//   weights of S                     fp32; what they are is the kernel's
//   O^T[dim, unit] += V^T . W^T      V^T by LDS transpose reads; W as a bf16 hi + lo pair (16 significant bits)
// K rows are permuted inside a tile so that the accumulators of two 16-key sub-tiles are the 32-key B operand of the second product.
//
// What bounds it: the vector ALU and the matrix cores take about as long (per half tile and wave 80 + 16 quarter-rate instructions
// beside 48 products of 16 cycles), so the loop is built to run them side by side.  Half tiles go through three stages a step
// apart: scores of half h + 1, weights of h, values of h - 1, all in one block without branches.  Tiles travel from memory into LDS
// directly, a whole tile ahead, which leaves the registers that staging took to the stages, and one barrier per tile: between odd
// halves, where the steps read K of one tile and V of one tile, so two buffers each are enough.
//
// Sinks, 32 heads of 128 on 8 KV heads, kernel alone, before (a tile's stages one after the other, staged through registers) and
// after: 4 x 2048 tokens 260 us, 530 TFLOP/s -> 205, 669; eight prompts of 1061 to 2048 355 -> 282 us.
// Measured and not taken: eight waves per workgroup (8 % slower), LDS reads of a whole step ahead of its products (4 %
// slower), wave priorities around the products (no difference).
#pragma once
#include "gemm_shared.h"

namespace tlf {

constexpr int kPromptKeys = 64;       // keys per tile
constexpr int kPromptWaves = 4;

template <typename T>
__device__ __forceinline__ T prompt_lds(unsigned int at) {
  return *reinterpret_cast<const T __attribute__((address_space(3))) *>(at);
}
__device__ __forceinline__ uint2 prompt_lds_tr16(unsigned int at) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<shortx4 __attribute__((address_space(3))) *>(at)));
}
// 16 bytes per lane into LDS at a wave's address: from a uniform base and an offset per lane, or from an address per lane.
__device__ __forceinline__ void prompt_copy(unsigned int offset, const void *base, unsigned int lds) { TLF_DL_COPY(offset, base, lds); }
__device__ __forceinline__ void prompt_copy_at(const void *from, unsigned int lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(lds) : "memory");
}

// DC, VC: key and value dimensions in units of 32.  LDS holds two tiles of K and two of V, rows unpadded; the 16-byte pieces of a K row
// are swapped with its neighbours in groups of 4 or 8 and pairs of pieces of a V row permuted by the row, against bank conflicts.
template <bool LEAD, bool MASK, bool START = false>
struct PromptPart {
  static constexpr bool lead = LEAD, mask = MASK, start = START;
};

template <int DC, int VC, int CT>
struct PromptCore {
  template <bool LEAD, bool MASK, bool START = false>
  using Part = PromptPart<LEAD, MASK, START>;
  static constexpr int DP = DC * 32, VP = VC * 32, KCH = DC * 4, VCH = VC * 4, KX = KCH % 8 == 0 ? 7 : 3;
  static constexpr int KB = kPromptKeys * DP * 2, VB = kPromptKeys * VP * 2;        // bytes of a tile
  typedef floatx4 Scores[2][CT];      // of a half: [16 keys][16 units]; lane (n, g): keys g * 8 + 4 s + r of unit n
  struct Weights {
    uint4 hi[CT], lo[CT];
  };
  bf16x8 qf[CT][DC], kf[2][DC], vf[2 * VC];
  floatx4 acc[CT][2 * VC];
  unsigned int klds, vlds, kat, vat;
  int wave;

  // the tile's row in LDS row r of a K tile
  static __device__ __forceinline__ int key_of(int r) { return (r & 32) | ((r & 16) >> 2) | ((r & 12) << 1) | (r & 3); }
  static __device__ __forceinline__ int pair_of(int row) { return VC >= 4 ? (row & 3) | (row >> 1 & 4) : VC == 2 ? (row >> 1 & 1) | (row >> 2 & 2) : row >> 3 & 1; }
  // Which 16-byte piece of which of the tile's rows this lane's copy i brings (DC copies of K and VC of V per wave), and where to.
  __device__ __forceinline__ void k_piece(int i, int lane, int &row, int &piece) const {
    const int slot = (i * kPromptWaves + wave) * 64 + lane, r = slot / KCH;
    row = key_of(r);
    piece = slot % KCH ^ (r & KX);
  }
  __device__ __forceinline__ void v_piece(int i, int lane, int &row, int &piece) const {
    const int slot = (i * kPromptWaves + wave) * 64 + lane;
    row = slot / VCH;
    piece = slot % VCH ^ (pair_of(row) * 2);
  }
  __device__ __forceinline__ unsigned int k_place(int t, int i) const { return klds + (t & 1) * KB + (i * kPromptWaves + wave) * 1024; }
  __device__ __forceinline__ unsigned int v_place(int t, int i) const { return vlds + (t & 1) * VB + (i * kPromptWaves + wave) * 1024; }

  __device__ __forceinline__ void start(unsigned int k, unsigned int v, int tid) {
    const int lane = tid & 63, n = lane & 15, g = lane >> 4, vrow = g * 8 + (n >> 2);
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    klds = k;
    vlds = v;
    kat = k + n * (DP * 2) + ((g ^ (n & KX)) * 16);
    vat = v + vrow * (VP * 2) + pair_of(vrow) * 32 + (n & 3) * 8;
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int d = 0; d < 2 * VC; ++d) acc[c][d] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  __device__ __forceinline__ void read_k(int h) {
    const unsigned int at = kat + (h >> 1 & 1) * KB + (h & 1) * (32 * DP * 2);
#pragma unroll
    for (int kc = 0; kc < DC; ++kc) {
      const unsigned int to = KX == 7 ? (at ^ ((kc & 1) * 64)) + kc / 2 * 128 : at + kc * 64;
      kf[0][kc] = prompt_lds<bf16x8>(to);
      kf[1][kc] = prompt_lds<bf16x8>(to + 16 * DP * 2);
    }
  }
  __device__ __forceinline__ void read_v(int h) {
    const unsigned int at = vat + (h >> 1 & 1) * VB + (h & 1) * (32 * VP * 2);
#pragma unroll
    for (int d = 0; d < 2 * VC; ++d) {
      const unsigned int to = VC == 3 ? (at ^ ((d & 1) * 32)) + d / 2 * 64 : at ^ (d * 32);   // rows of 192 bytes swap neighbours only
      const uint2 v0 = prompt_lds_tr16(to), v1 = prompt_lds_tr16(to + 8 * VP);
      vf[d] = __builtin_bit_cast(bf16x8, make_uint4(v0.x, v0.y, v1.x, v1.y));
    }
  }
  __device__ __forceinline__ void scores(const float (&from)[CT], Scores &s) const {     // from: a unit's scores begin here
#pragma unroll
    for (int c = 0; c < CT; ++c) s[0][c] = s[1][c] = floatx4{from[c], from[c], from[c], from[c]};
#pragma unroll
    for (int kc = 0; kc < DC; ++kc)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        s[0][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[0][kc], qf[c][kc], s[0][c], 0, 0, 0);
        s[1][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[1][kc], qf[c][kc], s[1][c], 0, 0, 0);
      }
  }
  __device__ __forceinline__ void values(const Weights &w) {
#pragma unroll
    for (int d = 0; d < 2 * VC; ++d) {
#pragma unroll
      for (int c = 0; c < CT; ++c) acc[c][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[d], __builtin_bit_cast(bf16x8, w.hi[c]), acc[c][d], 0, 0, 0);
#pragma unroll
      for (int c = 0; c < CT; ++c) acc[c][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[d], __builtin_bit_cast(bf16x8, w.lo[c]), acc[c][d], 0, 0, 0);
    }
  }
  static __device__ __forceinline__ void split(int c, const float (&e)[8], Weights &w) {
    unsigned int hi[4], lo[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) weight_pairs(e[2 * j], e[2 * j + 1], hi[j], lo[j]);
    w.hi[c] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    w.lo[c] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
  }

  // The workgroup's walk over `tiles` tiles, of which the wave computes first_tile <= t < end: those that some of its units see.  A value
  // behind or before them, infinite or no number as it may be, does not reach its rows.  The kernel's parts:
  //   copy_k(t, part), copy_v     the tile's copies; called for t = 0, 1, .. in turn
  //   from(f)                     where a unit's scores begin (read once per half)
  //   finish(h, s, part)          what is done to the scores of half h as soon as they are there
  //   before(h, s, w, part)       ahead of the weights of half h; `w`: weights of half h - 1 whose values are not added yet (add_values),
  //                               none with part.start, which is set in the wave's first half
  //   weights(h, s, w, part)
  // part.mask is not set where all keys of the half's tile are seen by all units: tiles clear_from <= t < clear_to of them (wave
  // uniform), clear_from 0 without LEAD.  part.lead is set where t may be below clear_from, part.start in the wave's first tile.
  // BOTH: `before` is first called when the scores of both halves of that tile are there.
  // SOME: it may be some only; otherwise first_tile is 0 and `end` is `tiles`.
  template <bool LEAD, bool SOME, bool BOTH, class CopyK, class CopyV, class From, class Finish, class Before, class Weigh>
  __device__ __forceinline__ void walk(int tiles, int first_tile, int end, int clear_from, int clear_to, CopyK copy_k, CopyV copy_v, From from, Finish finish, Before before, Weigh weights) {
    constexpr Part<true, true> lead{};
    constexpr Part<false, false> plain{};
    constexpr Part<false, true> tail{};
    constexpr Part<LEAD, true, true> first{};
    Scores se, so;                    // of even and odd halves
    Weights we{}, wo{};
    auto make_scores = [&](Scores &s) __attribute__((always_inline)) {
      float f[CT];
      from(f);
      scores(f, s);
    };
    // K of tile t and V of tile t - 1 are there; the buffers of K t - 1 and V t - 2 are free
    auto arrive = [&](int t, auto part) __attribute__((always_inline)) {
      TLF_DL_BARRIER(0);
      if (t < tiles) copy_v(t, part);
      if (t + 1 < tiles) copy_k(t + 1, part);
    };
    copy_k(0, first);
    int t = SOME ? first_tile : 0;
    if constexpr (LEAD && SOME)
      for (int i = 0; i < t; ++i) arrive(i, first);
    TLF_DL_BARRIER(0);
    copy_v(t, first);
    if (t + 1 < tiles) copy_k(t + 1, first);
    read_k(2 * t);
    make_scores(se);
    finish(2 * t, se, first);
    if constexpr (!BOTH) before(2 * t, se, wo, first);
    read_k(2 * t + 1);
    make_scores(so);
    if constexpr (BOTH) {
      finish(2 * t + 1, so, first);
      before(2 * t, se, wo, first);
    }
    weights(2 * t, se, we, first);
    if constexpr (!BOTH) finish(2 * t + 1, so, first);
    // scores of 2 t + 2 and 2 t + 3, weights of 2 t + 1 and 2 t + 2, values of 2 t and 2 t + 1
    auto two_steps = [&](int t, auto part) __attribute__((always_inline)) {
      TLF_DL_BARRIER(0);
      copy_v(t + 1, part);
      if (t + 2 < tiles) copy_k(t + 2, part);
      before(2 * t + 1, so, we, part);
      read_k(2 * t + 2);
      read_v(2 * t);
      make_scores(se);
      weights(2 * t + 1, so, wo, part);
      values(we);
      finish(2 * t + 2, se, part);
      before(2 * t + 2, se, wo, part);
      read_k(2 * t + 3);
      read_v(2 * t + 1);
      make_scores(so);
      weights(2 * t + 2, se, we, part);
      values(wo);
      finish(2 * t + 3, so, part);
    };
    // loops of their own: as a choice inside one loop the two forms do not fit the registers
    if constexpr (LEAD)
      for (; t + 1 < end && t < clear_from; ++t) two_steps(t, lead);
    for (; t + 1 < clear_to; ++t) two_steps(t, plain);
    for (; t + 1 < end; ++t) two_steps(t, tail);
    if constexpr (SOME) {
      arrive(t + 1, first);
    } else {
      TLF_DL_BARRIER(0);
      t = tiles - 1;
    }
    before(2 * t + 1, so, we, tail);
    weights(2 * t + 1, so, wo, first);
    read_v(2 * t);
    values(we);
    read_v(2 * t + 1);
    values(wo);
    if constexpr (SOME)
      for (t += 2; t <= tiles; ++t) arrive(t, first);        // for the other waves
  }
  // For `before`: the values of half h with weights `w`, which are used up.
  __device__ __forceinline__ void add_values(int h, Weights &w) {
    read_v(h);
    values(w);
#pragma unroll
    for (int c = 0; c < CT; ++c) w.hi[c] = w.lo[c] = make_uint4(0, 0, 0, 0);
  }
};

}  // namespace tlf
