// The loop that the prompt kernels of sink_prefill.hip, pooled_prefill.hip and latent_prefill.hip share, bf16, on the matrix cores; talk_prefill.hip
// takes its scores.
//
// A workgroup of four waves has 128 units, a query row of one head each, 32 per wave, and walks its keys in tiles of 64:
//   S^T[key, unit] = K . Q^T         v_mfma_f32_32x32x16_bf16
//   weights of S                     fp32; what they are is the kernel's
//   O^T[dim, unit] += V^T . W^T      V^T by LDS transpose reads; W as a bf16 hi + lo pair (16 significant bits)
// K rows are permuted inside a tile so that the accumulators of 32 keys are the two 16-key B operands of the second product, and a lane
// holds one unit: 16 of a half tile's keys, the others are 32 lanes away.
//
// What bounds it: the vector ALU and the matrix cores take about as long (per half tile and wave 140 instructions beside 24 products of 32
// cycles), one after the other in a wave, so it takes the two waves of a SIMD to keep both at work.  A half tile is one stretch of products
// (values of the half before, then scores) and one of weights, with the reads of the next operands in between.  Tiles travel from memory into
// LDS directly, a whole tile ahead, with one barrier per tile; two buffers of K and of V are enough.
//
// Kernels alone or layers, eight prompts of 1061 to 2048 tokens, with 16x16x32 products in three stages of half tiles a step apart (two units a
// lane, weights of one half beside the scores of the next) and so: pooled 296 -> 286 us a layer, sinks 366 -> 364, latents 175 -> 166 and on a
// faster card 161 -> 152; 250, 198 and 168 registers a lane (251, 236 and 192 before).  In a stream of nothing but these products and weights from
// registers two waves take 2150 cycles where the products alone take 1540: beside another wave's vector instructions a product takes a
// fifth longer.  Without copies sinks take 331, without LDS reads of V pooled heads 287.
// Halves of masked tiles that none of the wave's units sees are left out (half of the row tiles end in the first half of a tile, a pooled window begins in a
// second one as often): layers 261.2 -> 258.9 us (pooled), 347.2 -> 344.7 (sinks) and 141.2 -> 141.1 (latents), where runs of one side differ by 1.5 %.
// Measured and not taken: scores in front of the values (no difference), reads kept behind the products (3 % slower), wave priorities around the
// products (3 % slower), workgroups that take their row tiles from a list (1 - 2 % slower, though a new one starts 3.5 us after the one before
// it ends: while one is away the other runs faster).
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

// DC, VC: key and value dimensions in units of 32.  LDS holds two tiles of K and two of V, rows unpadded; the 16-byte pieces of K rows and
// the 64-byte pieces of V rows are permuted by the row, so that 16 rows of a K piece, or four rows of a V piece, cover all banks.
template <bool LEAD, bool MASK>
struct PromptPart {
  static constexpr bool lead = LEAD, mask = MASK;
};

template <int DC, int VC>
struct PromptCore {
  static constexpr int DP = DC * 32, VP = VC * 32, KCH = DC * 4, VCH = VC * 4;
  static constexpr int KB = kPromptKeys * DP * 2, VB = kPromptKeys * VP * 2;        // bytes of a tile
  // Pieces of a row are found by an exclusive or on its address, so rows of an even number of units have to be a power of two, and buffers begin at a multiple of one
  static_assert((DC % 2 == 1 || (DC & (DC - 1)) == 0) && (VC % 2 == 1 || (VC & (VC - 1)) == 0), "rows whose pieces an exclusive or finds");
  typedef floatx16 Scores;              // of a half; lane (n, g): keys 16 (r >> 3) + 8 g + (r & 7) of unit n
  struct Weights {
    uint4 hi[2], lo[2];
  };
  bf16x8 qf[2 * DC], kf[2 * DC], vf[2][VC];
  floatx16 acc[VC];
  unsigned int klds, vlds, kat, vat;
  int wave;

  static __device__ __forceinline__ int key_of(int r) { return (r & ~12) | ((r & 8) >> 1) | ((r & 4) << 1); }       // the tile's row in LDS row r of K
  static __device__ __forceinline__ int kswap(int r) { return DC % 4 == 0 ? r & 15 : DC % 4 == 2 ? r >> 1 & 7 : r >> 2 & 3; }
  static __device__ __forceinline__ int vswap(int r) { return VC % 4 == 0 ? r & 3 : VC % 4 == 2 ? r >> 1 & 1 : 0; }
  // Which 16-byte piece of which of the tile's rows this lane's copy i brings (DC copies of K and VC of V per wave), and where to.
  __device__ __forceinline__ void k_piece(int i, int lane, int &row, int &piece) const {
    const int slot = (i * kPromptWaves + wave) * 64 + lane, r = slot / KCH;
    row = key_of(r);
    piece = slot % KCH ^ kswap(r);
  }
  __device__ __forceinline__ void v_piece(int i, int lane, int &row, int &piece) const {
    const int slot = (i * kPromptWaves + wave) * 64 + lane;
    row = slot / VCH;
    piece = slot % VCH ^ (vswap(row) * 4);
  }
  __device__ __forceinline__ unsigned int k_place(int t, int i) const { return klds + (t & 1) * KB + (i * kPromptWaves + wave) * 1024; }
  __device__ __forceinline__ unsigned int v_place(int t, int i) const { return vlds + (t & 1) * VB + (i * kPromptWaves + wave) * 1024; }

  // k, v: LDS addresses of the buffers, aligned(1024)
  __device__ __forceinline__ void start(unsigned int k, unsigned int v, int tid) {
    const int lane = tid & 63, n = lane & 31, g = lane >> 5, vrow = g * 8 + (lane >> 2 & 3);
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    klds = k;
    vlds = v;
    kat = k + n * (DP * 2) + ((g ^ kswap(n)) * 16);
    vat = v + vrow * (VP * 2) + vswap(vrow) * 64 + (lane >> 4 & 1) * 32 + (lane & 3) * 8;
#pragma unroll
    for (int d = 0; d < VC; ++d) {
      vf[0][d] = vf[1][d] = __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[d][r] = 0.f;
    }
  }
  __device__ __forceinline__ void read_k(int t, int hf) {
    const unsigned int at = kat + (t & 1) * KB + hf * (32 * DP * 2);
#pragma unroll
    for (int kc = 0; kc < 2 * DC; ++kc) kf[kc] = prompt_lds<bf16x8>(DC % 2 ? (at ^ ((kc & 1) * 32)) + kc / 2 * 64 : at ^ (kc * 32));
  }
  __device__ __forceinline__ void read_v(int t, int hf) {
    const unsigned int at = vat + (t & 1) * VB + hf * (32 * VP * 2);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int d = 0; d < VC; ++d) {
        const unsigned int to = (VC % 2 ? at + d * 64 : at ^ (d * 64)) + q * (16 * VP * 2);
        const uint2 v0 = prompt_lds_tr16(to), v1 = prompt_lds_tr16(to + 8 * VP);
        vf[q][d] = __builtin_bit_cast(bf16x8, make_uint4(v0.x, v0.y, v1.x, v1.y));
      }
  }
  __device__ __forceinline__ void scores(const Scores &from, Scores &s) const {     // from: where a unit's scores begin
    s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[0], qf[0], from, 0, 0, 0);
#pragma unroll
    for (int kc = 1; kc < 2 * DC; ++kc) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[kc], qf[kc], s, 0, 0, 0);
  }
  __device__ __forceinline__ void values(const Weights &w) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
      for (int d = 0; d < VC; ++d) acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[q][d], __builtin_bit_cast(bf16x8, w.hi[q]), acc[d], 0, 0, 0);
#pragma unroll
      for (int d = 0; d < VC; ++d) acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[q][d], __builtin_bit_cast(bf16x8, w.lo[q]), acc[d], 0, 0, 0);
    }
  }
  static __device__ __forceinline__ void split(const float (&e)[16], Weights &w) {
    unsigned int hi[8], lo[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) weight_pairs(e[2 * j], e[2 * j + 1], hi[j], lo[j]);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      w.hi[q] = make_uint4(hi[4 * q], hi[4 * q + 1], hi[4 * q + 2], hi[4 * q + 3]);
      w.lo[q] = make_uint4(lo[4 * q], lo[4 * q + 1], lo[4 * q + 2], lo[4 * q + 3]);
    }
  }
  static __device__ __forceinline__ Scores all(float x) {
    Scores s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = x;
    return s;
  }
  static __device__ __forceinline__ float largest(const Scores &s) {        // of this lane
    float x = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) x = fmaxf(x, s[r]);
    return x;
  }
  static __device__ __forceinline__ float sum(const float (&e)[16]) {
    return (((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]))) + (((e[8] + e[9]) + (e[10] + e[11])) + ((e[12] + e[13]) + (e[14] + e[15])));
  }
  __device__ __forceinline__ void rescale(float by) {
#pragma unroll
    for (int d = 0; d < VC; ++d) acc[d] *= by;
  }

  // The workgroup's walk over `tiles` tiles, of which the wave computes first_tile <= t < end: those that some of its units see.  A value
  // behind or before them, infinite or no number as it may be, does not reach its rows.  The kernel's parts:
  //   copy(t, part)               the tile's copies; called for t = 1, 2, .. in turn, the first one's are under way
  //   seen(t, hf, part)           whether any of the wave's units sees a key of half hf of tile t, which is masked
  //   from()                      where the unit's scores begin (registers that are kept: set anew for each half they are a ninth of a wave's vector work)
  //   weights(t, hf, s, w, part)  of half hf of tile t, when all values of the halves before are in acc
  // part.mask is not set where all keys of the tile are seen by all units: tiles clear_from <= t < clear_to of them (wave uniform),
  // clear_from 0 without LEAD.  part.lead is set where t may be below clear_from.
  // SOME: the wave's tiles may be some only; otherwise first_tile is 0 and `end` is `tiles`.
  template <bool LEAD, bool SOME, class Copy, class Seen, class From, class Weigh>
  __device__ __forceinline__ void walk(int tiles, int first_tile, int end, int clear_from, int clear_to, Copy copy, Seen seen, From from, Weigh weights) {
    constexpr PromptPart<true, true> lead{};
    constexpr PromptPart<false, false> plain{};
    constexpr PromptPart<false, true> tail{};
    constexpr PromptPart<LEAD, true> first{};
    Weights w{};
    // tile t is there, and what was in the other buffers has been read
    auto arrive = [&](int t, auto part) __attribute__((always_inline)) {
      TLF_DL_BARRIER(0);
      if (t + 1 < tiles) copy(t + 1, part);
    };
    auto step = [&](int t, auto part) __attribute__((always_inline)) {
      arrive(t, part);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        if (part.mask && !seen(t, hf, part)) continue;       // wave uniform
        Scores s;
        read_k(t, hf);
        values(w);
        scores(from(), s);
        read_v(t, hf);
        weights(t, hf, s, w, part);
      }
    };
    int t = 0;
    if constexpr (LEAD && SOME)
      for (; t < first_tile; ++t) arrive(t, first);
    // loops of their own: as a choice inside one loop the forms do not fit the registers
    if constexpr (LEAD)
      for (; t < end && t < clear_from; ++t) step(t, lead);
    for (; t < clear_to; ++t) step(t, plain);
    for (; t < end; ++t) step(t, tail);
    values(w);
    if constexpr (SOME)
      for (; t < tiles; ++t) arrive(t, first);               // for the other waves
  }

  // Results of dimensions d * 32 + 8 i + 4 g .. of a unit, times `by`, gates and all that `at(col)` knows, at `o`: rows of `dims`.
  // vec: o is aligned to 8 bytes and dims a multiple of 4, wide: 16 and 8.
  template <class Times>
  __device__ __forceinline__ void store(unsigned short *o, int dims, bool vec, bool wide, int g, Times times) const {
#pragma unroll
    for (int d = 0; d < VC; ++d)
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        unsigned int v[2][2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int r = (i + k) * 4, col = d * 32 + r * 2 + g * 4;
          float f[4] = {acc[d][r], acc[d][r + 1], acc[d][r + 2], acc[d][r + 3]};
          times(col, f);
          v[k][0] = pack_bf16x2(f[0], f[1]);
          v[k][1] = pack_bf16x2(f[2], f[3]);
        }
        if (wide) {                                          // pieces of 8 from the two lanes of a unit
          const auto a = __builtin_amdgcn_permlane32_swap(v[0][0], v[1][0], false, false), b = __builtin_amdgcn_permlane32_swap(v[0][1], v[1][1], false, false);
          const int col = d * 32 + (i + g) * 8;
          if (col < dims) *reinterpret_cast<uint4 *>(o + col) = make_uint4(a[0], b[0], a[1], b[1]);
          continue;
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int col = d * 32 + (i + k) * 8 + g * 4;
          if (vec) {
            if (col < dims) *reinterpret_cast<uint2 *>(o + col) = make_uint2(v[k][0], v[k][1]);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (col + r < dims) o[col + r] = static_cast<unsigned short>(v[k][r / 2] >> (16 * (r & 1)));
          }
        }
      }
  }
};

// Over the two lanes of a unit.
__device__ __forceinline__ float prompt_unit_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float prompt_unit_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace tlf
