// State-space portions of prompts (ssd.hip), bf16: the heads of a group, which share B and C, in one workgroup.
//
//   ssd_group_kernel   one workgroup per (sequence or segment, up to eight pairs of a head and 32 columns of P), a wave each, sequential
//                      over chunks of 64 tokens.  The formulas are ssd_chunk_kernel's:
//                        G[t, s] = C_t . B_s      once per chunk, 16 x 16 tiles dealt to the waves, through LDS
//                        Y^T = S^T C^T + X^T (w_s G)^T, y = 2^(c_t) Y with w_s = dt_s 2^(-c_s)
//                        S = 2^(c_end) S + B^T (dt_s 2^(c_end - c_s) X)
//                      S stays in fp32 accumulators, and their layout is the next product's operand: rows of S are labelled so that C
//                      is read in whole granules.  S and w G enter as bf16 hi + lo pairs, x, B and C are exact.  The scaled X enters as
//                      three pieces: what it lacks stays in the state.  A chunk's rows come into LDS one chunk ahead, granules of
//                      16 bytes swizzled by the row.  Where some w_s leaves 2^63 (or a head decays by more than 2^100 within a
//                      chunk), the head takes 2^(c_t - c_s) dt_s pair by pair instead.
//
// A segment's contribution comes from a first pass over B and X (MODE 1); a segment adds up what lies before it as it starts.  The first pass
// also goes through the beginning of each sequence for good (ssd_groups_begun).
//
// 128 heads of 64 in 8 groups, state 128, 4 sequences of up to 3000 tokens, medians under the profiler: 437 us with ssd_chunk_kernel, which
// forms G for every head and passes S through LDS as pairs; here 254 + 95, or 104 + 178 at steady clocks where it was 82 + 220 without beginnings.  With the scaled X as pairs 249 + 81, but then 1 to 4 % more outputs
// than with ssd_chunk_kernel missed their nearest bf16 value (1.3 in a thousand do; the state's error is 1.1e-6 to 2.6e-6 on both, and 2e-7
// to 8e-7 with pieces).  With pairs a chunk of 4 heads took 18700 cycles, 5000 of them products and 9200 vector instructions on each SIMD, the
// rest latency of two waves per SIMD (S alone takes 64 registers).  16 columns per wave and four waves per SIMD were slower (285 + 71, the
// least of twelve, where this took 209 + 68: twice the reads of B and C, twice the weights), and so were copies issued in a row (+2300 cycles
// a chunk: a wave waits where several are queued) and step sizes masked as they are loaded (+2200: that waits for them).
#include <algorithm>
#include <type_traits>

#include "gemm_shared.h"
#include "ssd.h"

namespace tlf {

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
constexpr int kSG = 68;   // floats from row to row of G: reads of 16 bytes down a column fall on different banks

// LDS of a workgroup, in bytes: two buffers of C, B and the waves' X, G, the waves' three values per token.
constexpr int ssd_group_lds(int np, int waves, bool contribution) {
  return 2 * ((contribution ? 1 : 2) * kSC * np * 2 + waves * kSC * 64) + (contribution ? 0 : kSC * kSG * 4) + waves * 3 * kSC * 4;
}

// N in units of 32.  MODE 0: a whole sequence, 1: what segment `seg` adds to it, 2: segment `seg` from there, 3: a sequence's beginning, 4: none, the state
// is only handed on.
template <int NN, int MODE>
__device__ __forceinline__ void ssd_group(const SsdArgs &a, const int sq, const int seg, unsigned char *smem) {
  typedef unsigned short T;
  constexpr int NP = NN * 32, GPR = NP / 8, ROW = NP * 2, CB = MODE == 1 ? 0 : kSC * ROW, BB = kSC * ROW;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, hi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  // workgroup w runs on XCD w % 8: those of one group on one where the groups are a multiple of 8
  const int grp = blockIdx.x % a.G, share = a.H / a.G, cols = a.P / 32, units = share * cols, unit = blockIdx.x / a.G * waves + wave;
  const bool active = unit < units;
  const int h = grp * share + min(unit, units - 1) / cols, p0 = min(unit, units - 1) % cols * 32;
  const int seq = a.first_seq + sq, slot = a.state_slots[seq];
  const bool slot_ok = slot >= 0 && slot < a.num_slots;
  const int begin = a.cu_q[seq], tokens = a.cu_q[seq + 1] - begin, chunks = (tokens + kSC - 1) / kSC;
  int c0 = 0, c1 = chunks, begun = 0;
  if (MODE != 0) {
    begun = static_cast<int>(static_cast<int64_t>(chunks) * a.begun >> 16);
    const int per = (chunks - begun + a.segs - 1) / a.segs;
    c0 = MODE == 3 ? 0 : min(begun + seg * per, chunks);
    c1 = MODE == 3 ? begun : min(c0 + per, chunks);
  }
  const unsigned int bufs = TLF_DL_LDSADDR(smem), BUF = CB + BB + waves * kSC * 64;
  float *const g_lds = reinterpret_cast<float *>(smem + 2 * BUF);
  float *const cum = g_lds + (MODE == 1 ? 0 : kSC * kSG) + wave * 3 * kSC, *const weight = cum + kSC, *const into_end = cum + 2 * kSC;
  const int64_t plane = static_cast<int64_t>(a.N) * a.P;
  float *st = a.state + (static_cast<int64_t>(slot_ok ? slot : 0) * a.H + h) * plane + p0 + n;

  // register r of tile i: row 32 i + 16 (r / 8) + 8 hi + r % 8, column p0 + n
  auto state_at = [&](int i, int r) __attribute__((always_inline)) { return static_cast<int64_t>(i * 32 + (r >> 3) * 16 + hi * 8 + (r & 7)) * a.P; };
  floatx16 S[NN];
#pragma unroll
  for (int i = 0; i < NN; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) S[i][r] = 0.f;
  // The last segment writes the state back while others may yet have to start: the second pass reads the state behind a sequence's beginning
  // from the last segment's place, which holds no contribution and where the first pass has put it.
  const bool held = slot_ok && a.starts[seq] != 0;
  float *const between = a.seg_state + ((static_cast<int64_t>(sq) * a.segs + a.segs - 1) * a.H + h) * plane + p0 + n;
  if (MODE != 1 && active && (held || (MODE == 2 && begun))) {
    const float *from = MODE == 2 ? between : st;
#pragma unroll
    for (int i = 0; i < NN; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) S[i][r] = from[state_at(i, r)];
  }
  if constexpr (MODE == 4) {
    if (active && held) {
#pragma unroll
      for (int i = 0; i < NN; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) between[state_at(i, r)] = S[i][r];
    }
    return;
  }
  if (MODE == 2 && active) {
    for (int e = 0; e < seg; ++e) {
      const int64_t sg = (static_cast<int64_t>(sq) * a.segs + e) * a.H + h;
      const float *own = a.seg_state + sg * plane + p0 + n, dec = a.seg_decay[sg];
#pragma unroll
      for (int i = 0; i < NN; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) S[i][r] = fmaf(dec, S[i][r], own[state_at(i, r)]);
    }
  }

  // C and B: four rows of 64 bytes, and eight of 16, on different banks.  A granule's turn repeats every sixteen rows, so rows further down
  // are a constant away and other granules an exclusive or.
  auto at_row = [&](int row, int granule) __attribute__((always_inline)) {
    const int turn = GPR == 16 ? (row & 3) << 2 | (row >> 2 & 3) : GPR == 8 ? (row >> 1 & 1) << 2 | (row >> 2 & 3) : row >> 2 & 3;
    return static_cast<unsigned int>(row * ROW + ((granule ^ turn) << 4));
  };
  // 32 columns of a wave's rows, sixteen of them at a time; behind the last row, that one
  auto rows_of_own = [&](const T *p, int ld, int last, unsigned int to, int i) __attribute__((always_inline)) {
    const int first = min(i * 16, last);
    const unsigned int down = static_cast<unsigned int>(min(static_cast<int>(__umul24(lane >> 2, ld)), (last - first) * ld));
    dl_copy(down * 2 + (((lane & 3) ^ (lane >> 4 & 3)) << 4), p + static_cast<int64_t>(first) * ld, to + i * 1024);
  };
  // a chunk's copies in six parts: B and C's first and second half, the wave's x
  constexpr int kParts = 6;
  auto copy = [&](int c, int buf, int part) __attribute__((always_inline)) {
    const T *first = static_cast<const T *>(a.xbc) + (begin - a.first_row + static_cast<int64_t>(c) * kSC) * a.channels;
    const T *bp = first + a.inner + grp * a.N, *cp = bp + a.G * a.N, *xp = first + h * a.P + p0;
    const int last = min(kSC, tokens - c * kSC) - 1;
    const unsigned int at = bufs + buf * BUF;
    if (part >= 2) {
      rows_of_own(xp, a.channels, last, at + CB + BB + wave * (kSC * 64), part - 2);
      return;
    }
    for (int i = part * (BB / 2048) + wave; i < (part + 1) * (BB / 2048); i += waves) {
      const int item = i * 64 + lane, row = item / GPR, granule = static_cast<int>(at_row(row, item % GPR) - row * ROW) >> 4;
      const unsigned int offset = static_cast<unsigned int>(__umul24(min(row, last), a.channels)) * 2 + granule * 16;
      dl_copy(offset, bp, at + CB + i * 1024);
      if (MODE != 1) dl_copy(offset, cp, at + i * 1024);
    }
  };
  float dt_next = 0.f, dec_next = 0.f;                       // as loaded: what is done with them waits for them
  auto steps = [&](int c) __attribute__((always_inline)) {
    const int64_t at = (begin - a.first_row + static_cast<int64_t>(c) * kSC + min(lane, min(kSC, tokens - c * kSC) - 1)) * a.H + h;
    dt_next = a.dt[at];
    dec_next = a.decay[at];
  };
  auto granule_of = [&](unsigned int at) __attribute__((always_inline)) { return *reinterpret_cast<const bf16x8 __attribute__((address_space(3))) *>(at); };
  auto turned = [&](unsigned int at) __attribute__((always_inline)) {
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<shortx4 __attribute__((address_space(3))) *>(at)));
  };
  auto pairs = [&](const float (&x)[8], bf16x8 &h8, bf16x8 &l8) __attribute__((always_inline)) {
    unsigned int p[4], q[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) weight_pairs(x[2 * j], x[2 * j + 1], p[j], q[j]);
    h8 = __builtin_bit_cast(bf16x8, make_uint4(p[0], p[1], p[2], p[3]));
    l8 = __builtin_bit_cast(bf16x8, make_uint4(q[0], q[1], q[2], q[3]));
  };
  if constexpr (MODE != 1) {                                 // the tiles above G's diagonal that are read with others
    for (int i = tid; i < 512; i += blockDim.x) g_lds[((i >> 8) * 32 + (i >> 4 & 15)) * kSG + (i >> 8) * 32 + 16 + (i & 15)] = 0.f;
  }
  const float D = MODE == 1 ? 0.f : Elem<T>::ld(static_cast<const T *>(a.D) + h);
  float total = 0.f;                                         // log2 decay of the whole segment

  if (c0 < c1) {
    steps(c0);
#pragma unroll
    for (int i = 0; i < kParts; ++i) copy(c0, 0, i);
  }
  for (int c = c0; c < c1; ++c) {
    // addresses are made from the lane anew in each chunk: kept, they would not fit beside the state
    int here = tid & 63;
    asm volatile("" : "+v"(here));
    const int lane = here, n = here & 31, hi = here >> 5;
    const unsigned int buf = bufs + ((c - c0) & 1) * BUF, bs = buf + CB, xs = bs + BB + wave * (kSC * 64);
    TLF_DL_BARRIER(0);
    const bool in = lane < tokens - c * kSC;                 // a token per lane
    const float sum = ssd_wave_scan(in ? dec_next : 0.f), dt = in ? dt_next : 0.f;
    auto own = [&](int row, int granule) __attribute__((always_inline)) { return xs + row * 64 + ((granule ^ (row >> 2 & 3)) << 4); };
    bf16x8 xf[4];                                            // lane (hi, p): column p, tokens 16 ks + 8 hi ..
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      uint2 x[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int row = ks * 16 + hi * 8 + (lane >> 2 & 3) + q * 4, chunk = lane & 3;
        x[q] = turned(xs + row * 64 + (((lane >> 4 & 1) * 2 + (chunk >> 1)) ^ (row >> 2 & 3)) * 16 + (chunk & 1) * 8);
      }
      xf[ks] = __builtin_bit_cast(bf16x8, make_uint4(x[0].x, x[0].y, x[1].x, x[1].y));
    }
    u32x2 xt[MODE == 1 ? 1 : 2][4];                          // lane (hi, t): columns 8 q + 4 hi ..
    if constexpr (MODE != 1) {
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int q = 0; q < 4; ++q) xt[tt][q] = *reinterpret_cast<const u32x2 __attribute__((address_space(3))) *>(own(tt * 32 + n, q) + hi * 8);
    }
    if (c + 1 < c1) steps(c + 1);
    // A copy takes the memory pipeline some sixty cycles and a wave waits where several are queued, so they are issued one by one between
    // products: the gate, which takes the place of x, then the next chunk's (the last one's once more where there is none)
    const int next = min(c + 1, c1 - 1);
    constexpr int kIssues = MODE == 1 ? kParts : kParts + 4;
    auto issue = [&](int i) __attribute__((always_inline)) {
      if (MODE != 1 && i < 4)
        rows_of_own(static_cast<const T *>(a.proj) + (begin + static_cast<int64_t>(c) * kSC) * a.ld + h * a.P + p0, static_cast<int>(a.ld), min(kSC, tokens - c * kSC) - 1, xs, i);
      else
        copy(next, ((c - c0) & 1) ^ 1, MODE == 1 ? i : i - 4);
    };
    if constexpr (MODE != 1) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // x has been read
    const float keep = __builtin_amdgcn_exp2f(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(sum), 63)));
    const float end = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sum), 63));
    const float w = dt * __builtin_amdgcn_exp2f(-sum);
    const bool mild = __ballot(!(w < 0x1p63f)) == 0 && end > -100.f;
    total += end;
    cum[lane] = sum;
    weight[lane] = mild ? w : dt;
    into_end[lane] = dt * __builtin_amdgcn_exp2f(end - sum);
    wave_lds_fence();
    if constexpr (MODE != 1) {
      const int m = lane & 15, g = lane >> 4;
      for (int tile = wave; tile < 10; tile += waves) {      // 16 x 16 tiles of G up to the diagonal
        const int tb = tile < 1 ? 0 : tile < 3 ? 1 : tile < 6 ? 2 : 3, sb = tile - tb * (tb + 1) / 2;
        floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
        const unsigned int at = at_row(m, g);
#pragma unroll
        for (int k = 0; k < NN; ++k)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(granule_of(bs + sb * 16 * ROW + (at ^ k << 6)), granule_of(buf + tb * 16 * ROW + (at ^ k << 6)), acc, 0, 0, 0);
        if (tb == sb)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[e] = g * 4 + e <= m ? acc[e] : 0.f;
        *reinterpret_cast<floatx4 *>(g_lds + (tb * 16 + m) * kSG + sb * 16 + g * 4) = acc;
      }
    }
    if constexpr (MODE != 1) {
      const unsigned int c_at = at_row(n, hi);
      floatx16 y[2];                                         // Y^T: columns t, rows p
#pragma unroll
      for (int r = 0; r < 16; ++r) y[0][r] = y[1][r] = 0.f;
#pragma unroll
      for (int kb = 0; kb < NN * 2; ++kb) {
#pragma unroll
        for (int i = kb * kIssues / (NN * 2); i < (kb + 1) * kIssues / (NN * 2); ++i) issue(i);
        float s8[8];
        bf16x8 sh, sl;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          s8[j] = S[kb >> 1][(kb & 1) * 8 + j];
          S[kb >> 1][(kb & 1) * 8 + j] *= keep;
        }
        pairs(s8, sh, sl);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
          const bf16x8 cf = granule_of(buf + tt * 32 * ROW + (c_at ^ kb << 5));
          y[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sh, cf, y[tt], 0, 0, 0);
          y[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sl, cf, y[tt], 0, 0, 0);
        }
      }
      lds_barrier();                                         // G is there
      float scale[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) scale[tt] = __builtin_amdgcn_exp2f(cum[tt * 32 + n]);
      // G's part, grow(tt, ks, m): the weights of eight values; what lies above the diagonal is zero, to be dropped anew where they may be infinite
      auto inside = [&](auto drop, auto grow) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
          for (int tt = ks >> 1; tt < 2; ++tt) {
            float m8[8];
            Elem<float>::ld8(g_lds + (tt * 32 + n) * kSG + ks * 16 + hi * 8, m8);
            grow(tt, ks, m8);
            if (drop && tt == ks >> 1) {
              const int last = n - (ks & 1) * 16 - hi * 8;
#pragma unroll
              for (int j = 0; j < 8; ++j) m8[j] = j <= last ? m8[j] : 0.f;
            }
            bf16x8 mh, ml;
            pairs(m8, mh, ml);
            y[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[ks], mh, y[tt], 0, 0, 0);
            y[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[ks], ml, y[tt], 0, 0, 0);
          }
      };
      if (mild) {
        inside(std::false_type{}, [&](int, int ks, float (&m)[8]) __attribute__((always_inline)) {
          float w8[8];
          Elem<float>::ld8(weight + ks * 16 + hi * 8, w8);
#pragma unroll
          for (int j = 0; j < 8; ++j) m[j] *= w8[j];
        });
      } else {
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
          for (int r = 0; r < 16; ++r) y[tt][r] *= scale[tt];
          scale[tt] = 1.f;
        }
        inside(std::true_type{}, [&](int tt, int ks, float (&m)[8]) __attribute__((always_inline)) {
          const float ct = cum[tt * 32 + n];
#pragma unroll
          for (int j = 0; j < 8; ++j) m[j] *= weight[ks * 16 + hi * 8 + j] * __builtin_amdgcn_exp2f(ct - cum[ks * 16 + hi * 8 + j]);
        });
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // the gate has landed; rows of the result take its place, to be stored in one piece
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const auto at = reinterpret_cast<u32x2 __attribute__((address_space(3))) *>(own(tt * 32 + n, q) + hi * 8);
          const u32x2 z2 = *at, x2 = xt[tt][q];
          const float x[4] = {__uint_as_float(x2.x << 16), __uint_as_float(x2.x & 0xffff0000u), __uint_as_float(x2.y << 16), __uint_as_float(x2.y & 0xffff0000u)};
          const float gate[4] = {__uint_as_float(z2.x << 16), __uint_as_float(z2.x & 0xffff0000u), __uint_as_float(z2.y << 16), __uint_as_float(z2.y & 0xffff0000u)};
          float o[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = fmaf(D, x[e], scale[tt] * y[tt][q * 4 + e]) * ssd_silu<T>(gate[e]);
          *at = u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
        }
      wave_lds_fence();
      T *const op = static_cast<T *>(a.out) + (begin + static_cast<int64_t>(c) * kSC) * a.ldo + static_cast<int64_t>(h) * a.P + p0 + (lane & 3) * 8;
      const int len = active ? tokens - c * kSC : 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = i * 16 + (lane >> 2);
        const u32x4 v = *reinterpret_cast<const u32x4 __attribute__((address_space(3))) *>(own(row, lane & 3));
        if (row < len) *reinterpret_cast<u32x4 *>(op + row * a.ldo) = v;
      }
    }
    if constexpr (MODE == 1) {
#pragma unroll
      for (int i = 0; i < NN; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) S[i][r] *= keep;
    }
    unsigned int b_at[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {                            // row m of the operand is state row m with bits 2 and 3 exchanged
      const int chunk = (lane & 1) * 2 + (lane >> 1 & 1);
      b_at[q] = at_row(hi * 8 + (lane >> 2 & 3) + q * 4, (lane >> 4 & 1) * 2 + (chunk >> 1)) + (chunk & 1) * 8;
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if constexpr (MODE == 1) {
#pragma unroll
        for (int i = ks * 2; i < ks * 2 + 2 && i < kIssues; ++i) issue(i);
      }
      float f8[8], x8[8];
      Elem<float>::ld8(into_end + ks * 16 + hi * 8, f8);
      unpack8(__builtin_bit_cast(uint4, xf[ks]), x8);
#pragma unroll
      for (int j = 0; j < 8; ++j) x8[j] *= f8[j];
      uint4 x3[3];
      bf16_pieces(x8, x3);
#pragma unroll
      for (int i = 0; i < NN; ++i) {
        uint2 b[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) b[q] = turned(bs + ks * 16 * ROW + (b_at[q] ^ i << 6));
        const bf16x8 bt = __builtin_bit_cast(bf16x8, make_uint4(b[0].x, b[0].y, b[1].x, b[1].y));
#pragma unroll
        for (int e = 0; e < 3; ++e) S[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bt, __builtin_bit_cast(bf16x8, x3[e]), S[i], 0, 0, 0);
      }
    }
  }
  if (MODE == 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // no copy is under way when the LDS is given back
  if (!active) return;
  if constexpr (MODE == 1) {
    const int64_t sg = (static_cast<int64_t>(sq) * a.segs + seg) * a.H + h;
    if (p0 == 0 && lane == 0) a.seg_decay[sg] = __builtin_amdgcn_exp2f(total);
    st = a.seg_state + sg * plane + p0 + n;
  } else if constexpr (MODE == 3) {
    if (!held && !begun) return;
    st = between;
  } else {
    if ((MODE == 2 && seg != a.segs - 1) || !slot_ok || tokens == 0) return;
  }
#pragma unroll
  for (int i = 0; i < NN; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) st[state_at(i, r)] = S[i][r];
}

template <int NN, int MODE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void ssd_group_kernel(const SsdArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int z = blockIdx.z;
  if constexpr (MODE == 0) ssd_group<NN, 0>(a, z, 0, smem);
  else if constexpr (MODE == 2) ssd_group<NN, 2>(a, z / a.segs, z % a.segs, smem);
  else if (z < a.seqs) ssd_group<NN, MODE == 1 ? 3 : 4>(a, z, 0, smem);
  else ssd_group<NN, 1>(a, (z - a.seqs) / (a.segs - 1), (z - a.seqs) % (a.segs - 1), smem);
}

// A workgroup has the work of up to eight waves, so there are fewer of them than of ssd_chunk_kernel's, and short sequences have to be many:
// with 8 chunks it is faster with segments (1 x 700 tokens, 32 or 128 heads: 56 -> 47 us, 69 -> 57; 1 x 3000: 100 -> 74, 225 -> 167), with 4
// once the chip is full (8 x 200, 128 heads: 116 -> 64), not below that (2 x 300: 42 -> 52).  Segments: two workgroups per CU, one after the
// other, even out the sequences where they keep 6 chunks; else one per CU, of at least 2 (1 x 1500: 8 segments 77 us, 6 83, 12 98).  Where many
// segments would have to make up for few groups, ssd.hip: ssd_chunks_suffice keeps a head per workgroup.
int ssd_groups_segments(int H, int P, int N, int G, int seqs, int max_tokens, int dtype) {
  const int64_t channels = static_cast<int64_t>(H) * P + 2ll * G * N, units = static_cast<int64_t>(H / G) * (P / 32);
  if (dtype != TLF_DT_BF16 || (N != 32 && N != 64 && N != 128) || P % 32 || units < 4 || channels % 8 || channels >= (1 << 24)) return 0;
  const int64_t wgs = seqs * G * ((units + 7) / 8), chunks = (max_tokens + kSC - 1) / kSC;
  if (wgs < 256 && chunks < 8) return 0;
  const int64_t twice = wgs >= 384 ? 1 : (512 + wgs - 1) / wgs, once = std::min<int64_t>(256 / wgs, chunks / 2);
  const int64_t segs = std::max<int64_t>(1, std::min<int64_t>(chunks >= 6 * twice ? twice : once, 16));
  return seqs * segs > 65535 ? 1 : static_cast<int>(segs);
}

// The part of each sequence, in 1/65536, that the first pass goes through for good: beside the workgroups that gather contributions half the
// chip or more has nothing to do, and what is done there is not gone through twice.  The estimate is in tenths of a microsecond: 110 a chunk and
// 39 where it only adds to the state, 40 to start (128 rows of state; fewer take less in all passes alike); rounds of the average length, but none shorter
// than the longest sequence takes.  Four sequences of 2035 to 3000 tokens, 128 heads in 8 groups: 82 + 220 us without, 104 + 178 with the first 7 of 47 chunks.
//
// Layer, us, without and with, states of 32, 64 and 128 rows: 12 sequences of up to 900 tokens, 32 heads of 64, 110 / 108, 24 heads in 4 groups 114 / 108,
// 32 heads 140 / 136; 3 of up to 1000, 64 heads, 73 / 68, 78 / 73.5, 93 / 87; 4 of up to 3000 184 / 181, 195 / 191, 225 / 223; of 33 such sets none was slower but 12 of up
// to 450, 70.4 / 72.2, 74.0 / 75.9, 86.9 / 88.2, where the estimate promises 4.6 us: so less than 8 does not count.
int ssd_groups_begun(const SsdArgs &a, int max_tokens) {
  const int64_t units = static_cast<int64_t>(a.H / a.G) * (a.P / 32), wgs = a.seqs * a.G * ((units + 7) / 8);
  const int64_t chunks = (static_cast<int64_t>(max_tokens) + kSC - 1) / kSC, most = (chunks + a.segs - 1) / a.segs;
  if (wgs > 128) return 0;
  const double share = std::min(1.0, static_cast<double>(a.rows) / (static_cast<double>(a.seqs) * max_tokens));
  auto pass = [&](int64_t jobs, int64_t cus, int64_t longest, int per_chunk) {
    return std::max(per_chunk * longest + 40.0, static_cast<double>((jobs + cus - 1) / cus) * (per_chunk * longest * share + 40.0));
  };
  const double without = pass(wgs * (a.segs - 1), 256, most, 39) + pass(wgs * a.segs, 256, most, 110);
  double least = std::min(0.97 * without, without - 80);
  int64_t first = 0;
  for (int64_t each = most - 1; each > 0 && chunks - a.segs * each <= chunks / 2; --each) {
    const int64_t begun = chunks - a.segs * each;
    if (begun <= 0) continue;
    const double t = std::max(110.0 * begun + 40, pass(wgs * (a.segs - 1), 256 - wgs, each, 39)) + pass(wgs * a.segs, 256, each, 110);
    if (t < least) {
      least = 0.99 * t;
      first = begun;
    }
  }
  return static_cast<int>((first * 65536 + chunks - 1) / chunks);
}

template <int NN>
int launch_ssd_groups_of(const SsdArgs &a, hipStream_t stream) {
  static const hipError_t allowed = [] {
    hipError_t e = hipSuccess;
    for (const void *k : {reinterpret_cast<const void *>(&ssd_group_kernel<NN, 0>), reinterpret_cast<const void *>(&ssd_group_kernel<NN, 1>),
                          reinterpret_cast<const void *>(&ssd_group_kernel<NN, 2>), reinterpret_cast<const void *>(&ssd_group_kernel<NN, 3>)})
      if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, ssd_group_lds(NN * 32, 8, false));
    return e;
  }();
  if (allowed != hipSuccess) return static_cast<int>(allowed);
  const int units = a.H / a.G * (a.P / 32), waves = std::min(8, units);
  const dim3 grid(a.G * ((units + waves - 1) / waves), 1, a.seqs * a.segs), block(waves * 64);
  if (a.segs == 1) {
    TLF_LAUNCH((ssd_group_kernel<NN, 0>), grid, block, ssd_group_lds(NN * 32, waves, false), stream, a);
  } else {
    // Without beginnings the first pass needs no C and no G, so that workgroups of four waves, of which registers allow two a CU, find the LDS for it.  20 sequences of up to
    // 2000 tokens, 16 heads of 64 in 8 groups, layer 331 us with all of it and 328 so, state 64 258 and 251; 18 of up to 4000 540 and 534, 409 and 398.
    if (a.begun) TLF_LAUNCH((ssd_group_kernel<NN, 1>), grid, block, ssd_group_lds(NN * 32, waves, false), stream, a);
    else TLF_LAUNCH((ssd_group_kernel<NN, 3>), grid, block, ssd_group_lds(NN * 32, waves, true), stream, a);
    TLF_LAUNCH((ssd_group_kernel<NN, 2>), grid, block, ssd_group_lds(NN * 32, waves, false), stream, a);
  }
  return launch_status();
}
int launch_ssd_groups(SsdArgs a, int max_tokens, hipStream_t stream) {
  a.begun = a.segs > 1 ? ssd_groups_begun(a, max_tokens) : 0;
  return a.N == 32 ? launch_ssd_groups_of<1>(a, stream) : a.N == 64 ? launch_ssd_groups_of<2>(a, stream) : launch_ssd_groups_of<4>(a, stream);
}

}  // namespace tlf
