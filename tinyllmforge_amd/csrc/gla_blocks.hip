// Gated linear attention of prompt portions (gla.hip) on the bf16 matrix cores, in blocks of 32 tokens and at 32-bit precision.
//
// A product of fp32 values is the sum of products of their bf16 pieces: three pieces of 8 significant bits are an fp32 value, v is
// one piece by itself.  Kd^T V and A V take three products, Qd S takes six (those of at least 2^-16 of the whole), and a bf16 product
// runs at sixteen times the rate of an fp32 one.
//
//   gla_block_kernel       per (block of a sequence, head), parallel: b_t = sum of log2 alpha within the block,
//                          Qd = q 2^b_t, Kd = k 2^(b_end - b_t), A[t, s] = sum_d q k 2^(b_t - b_s) for s <= t, each as three pieces in
//                          the order the matrix cores read.  A = (q 2^b_t) (k 2^-b_s)^T as products of pieces, too, unless some channel
//                          decays by more than 2^64 within the block.  Then every exponent is kept <= 0: the 8 x 8 blocks on A's
//                          diagonal are formed pair by pair, those left of it through the value at the boundary in front of them
//   gla_block_scan_kernel  per (sequence or stretch, head) a workgroup with 32 columns of v per wave, sequential over the blocks:
//                          O^T = S^T Qd^T + V^T A^T, out = norm and output gate of O;  S = diag(2^b_end) S + Kd^T V.  S stays in fp32
//                          accumulators; their layout is the next block's operand when the summation index is labelled as Qd is laid
//                          out.  A block's record and rows of v come into LDS one block ahead, and the rows' sums of squares
//                          go from wave to wave across the barrier in front of the next block.
//                          A value that is no number reaches no row before its half of a block
// Where (sequences, heads) alone leave CUs idle, the blocks of all sequences in a row are cut into `units` equal stretches, one workgroup per
// stretch and head: a stretch has the end of a sequence, whole ones, the beginning of another.  What a stretch adds to the sequence that it does
// not end comes from a first pass over that sequence's blocks in it (MODE 1), gla_stretches_kernel chains these, and the second pass starts from
// them.  Segments of a sequence's own length waited for the longest: 8 sequences of 1061 to 2048 tokens, 16 heads of 128 x 256, with
// segments 59 + 18 + 255 us, so 58 + 15 + 209; 12 of 450 to 900 48 + 24 + 216, and in one pass over whole ones 204.
//
// Eight prompts of 1061 to 2048 tokens, 16 heads, key dim 128, value dim 256, medians under the profiler: chunk 122 + scan 470 (both
// passes) + segments 18 + norm and gate 92 us over 16-token chunks with fp32 products; here blocks 103 - 120 + first pass 58 - 65 + chaining 15 + scan
// 169 - 205 us (whole layer 614 and 343 us).  The blocks write 55 KB a record, 3.7 TB/s with what they read: a workgroup waits for its rows, its decays and
// its sums in turn, so what counts is how many a CU holds.  With keys towards the boundaries in LDS it held two and not three, and one workgroup in two
// was launched for the second chunk of a block and left: 141 us where this took 115, with strong decays, which make those keys anew for each
// token, layer 450 and 425.  The decays' projection by the vector ALU took 13 more (layer 355 -> 343 us as a product).  The scan is held by its barriers, two waves on a SIMD: a block took 13900 cycles, 5000 of them products and some 7200
// vector instructions on each SIMD, the second wave came to the barrier 4100 cycles behind the first.  10900 with the copies on four waves and
// the block before finished in front of the products by these and behind them by the others: 198 -> 169 us.  The state's error against 64 bits is 5e-8 to 1.1e-7 on both, the
// output's is its rounding to bf16.
#include <algorithm>

#include "gemm_shared.h"
#include "gla.h"

namespace tlf {

constexpr int kGB = 32, kGlaBlockMaxR = 64;   // tokens per block, rank of the decay projection

template <int DK>
struct GlaBlock {   // a record, in bytes: pieces of Qd, of Kd, of A, decays
  static constexpr int kPiece = DK * kGB * 2, kAPiece = kGB * kGB * 2;
  static constexpr int kK = 3 * kPiece, kA = 6 * kPiece, kDec = kA + 3 * kAPiece, kSize = kDec + 1024;
};
size_t gla_block_record(int dk) { return dk * kGB * 2 * 6 + kGB * kGB * 2 * 3 + 1024; }
// Records of sequence s begin at (first chunk + s + 1) / 2: two chunks of 16 tokens are a block, and a sequence may end on one.
__device__ __forceinline__ int gla_first_block(int first_chunk, int seq) { return (first_chunk + seq + 1) / 2; }

template <int DK>
__global__ __launch_bounds__(DK * 4) void gla_block_kernel(const GlaArgs a) {
  typedef unsigned short T;
  using Rec = GlaBlock<DK>;
  constexpr int TH = DK * 4, LD = DK + 4, LPT = DK / 8;      // lanes per token, eight channels each
  constexpr int NW = DK / 16;
  static_assert(NW * kGB * kGB <= 2 * kGB * LD, "the waves' parts of A take the place of keys and decays");
  __shared__ __attribute__((aligned(16))) float kb2[2][kGB][LD], am[kGB][kGB + 4];
  float (&ks)[kGB][LD] = kb2[0], (&bs)[kGB][LD] = kb2[1];
  __shared__ float tots[4][DK];
  __shared__ int harsh;
  const int block = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  if (tid == 0) harsh = 0;
  int seq = -1, cbeg = 0, cend = 0;                          // each wave finds the block's sequence, 64 at a time
  for (int i0 = 0; i0 < a.seqs && seq < 0; i0 += 64) {
    const int i = min(i0 + (tid & 63), a.seqs - 1), lo = a.cu_chunks[i], hi = a.cu_chunks[i + 1], first = gla_first_block(lo, i);
    const unsigned long long here = __ballot(block >= first && block < first + (hi - lo + 1) / 2);
    if (here == 0) continue;
    const int at = __builtin_ctzll(here);
    seq = min(i0 + at, a.seqs - 1);
    cbeg = __builtin_amdgcn_readlane(lo, at);
    cend = __builtin_amdgcn_readlane(hi, at);
  }
  if (seq < 0) return;                                       // a slot that no sequence has
  const int chunk = cbeg + (block - gla_first_block(cbeg, seq)) * 2;
  const int64_t tok0 = a.chunk_tok[chunk];
  const int len = a.chunk_len[chunk] + (chunk + 1 < cend ? a.chunk_len[chunk + 1] : 0);
  const int64_t hk = static_cast<int64_t>(a.H) * DK, hv = static_cast<int64_t>(a.H) * a.dv;
  const T *pr = static_cast<const T *>(a.proj) + tok0 * a.ld;
  unsigned char *rec = reinterpret_cast<unsigned char *>(a.rec) + (static_cast<int64_t>(block) * a.H + h) * Rec::kSize;
  for (int i = tid; i < kGB * (kGB + 4); i += TH) (&am[0][0])[i] = 0.f;
  // token t, channels l * 4 .. and DK / 2 + l * 4 .. of it
  const int t = tid / LPT, l = tid % LPT;
  auto load_bf16 = [&](const T *p, float (&x)[8], int apart) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; i += 4) {
      const uint2 u = *reinterpret_cast<const uint2 *>(p + i / 4 * apart);
      x[i] = __uint_as_float(u.x << 16); x[i + 1] = __uint_as_float(u.x & 0xffff0000u);
      x[i + 2] = __uint_as_float(u.y << 16); x[i + 3] = __uint_as_float(u.y & 0xffff0000u);
    }
  };
  bool large;
  {
    float k[8];
    load_bf16(pr + min(t, len - 1) * a.ld + hk + h * DK + l * 4, k, DK / 2);
#pragma unroll
    for (int i = 0; i < 8; i += 4)
      *reinterpret_cast<float4 *>(&ks[t][i / 4 * (DK / 2) + l * 4]) = t < len ? make_float4(k[i], k[i + 1], k[i + 2], k[i + 3]) : make_float4(0.f, 0.f, 0.f, 0.f);
    float most = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) most = fmaxf(most, fabsf(k[i]));
    large = !(most < 1e9f);                                  // 2^64 times a key stays finite
  }
  // this thread's item of a 16-channel operand: token lane & 31, channels 16 (tid / 64) + 4 hi .. and + 8 + 4 hi ..
  const int lane = tid & 63, hi = lane >> 5, kb = tid >> 6, qt = lane & 31, qc = kb * 16 + hi * 4;
  float q[8], v[8], left[8];                                 // left: decay from a token to the block's end, in Kd's order
  load_bf16(pr + min(qt, len - 1) * a.ld + h * DK + qc, q, 8);
#pragma unroll
  for (int j = 0; j < 8; ++j) q[j] = qt < len ? q[j] * a.q_scale : 0.f;
  {
    // Decays: a thread has one channel and eight tokens, summed up here; the sums of the eights around them through LDS.  Sums towards the
    // end are made on their own: as differences they would lose what the tokens before have decayed by.  Their projection is a product of the matrix
    // cores, 32 channels a wave by its 16 tokens (twice), rows labelled so that a lane's first eight results are its tokens in turn
    const int d = (tid >> 7) * 32 + qt, t16 = (tid >> 6 & 1) * 16, t0 = t16 + hi * 8;
    const T *const rp = pr + min(t16 + ((lane & 3) | (lane & 4) << 1 | (lane & 8) >> 1), len - 1) * a.ld + 2 * hk + 2 * hv;
    const T *const w = static_cast<const T *>(a.a2) + (static_cast<int64_t>(h) * DK + d) * a.R;
    floatx16 zs;
#pragma unroll
    for (int r = 0; r < 16; ++r) zs[r] = 0.f;
    const bool whole = a.R % 8 == 0 && (reinterpret_cast<uintptr_t>(a.a2) & 15) == 0;
    for (int r0 = 0; r0 < a.R; r0 += 16) {
      const int at = r0 + hi * 8;
      uint4 x = make_uint4(0, 0, 0, 0), y = x;
      if (whole) {
        if (at < a.R) {
          x = *reinterpret_cast<const uint4 *>(rp + at);
          y = *reinterpret_cast<const uint4 *>(w + at);
        }
      } else {
        unsigned int xs[4] = {0, 0, 0, 0}, ys[4] = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (at + e < a.R) {
            xs[e / 2] |= static_cast<unsigned int>(rp[at + e]) << (e & 1) * 16;
            ys[e / 2] |= static_cast<unsigned int>(w[at + e]) << (e & 1) * 16;
          }
        x = make_uint4(xs[0], xs[1], xs[2], xs[3]);
        y = make_uint4(ys[0], ys[1], ys[2], ys[3]);
      }
      zs = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), zs, 0, 0, 0);
    }
    const float bias = Elem<T>::ld(static_cast<const T *>(a.a2_bias) + h * DK + d);
    float z[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) z[j] = zs[j] + bias;
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      left[j] = t0 + j < len ? log2_alpha(z[j], a.inv_tau) : 0.f;
      z[j] = sum += left[j];
    }
    tots[t0 / 8][d] = sum;
    __syncthreads();
    float before = 0.f, after = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      before += i < t0 / 8 ? tots[i][d] : 0.f;
      after += 3 - i > t0 / 8 ? tots[3 - i][d] : 0.f;
    }
#pragma unroll
    for (int j = 7; j >= 0; --j) {
      const float own = left[j];
      left[j] = after;
      after += own;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) bs[t0 + j][d] = before + z[j];
    if (large || !(before + sum >= -64.f)) harsh = 1;
  }
  __syncthreads();
  const bool apart = harsh != 0;
  uint4 p3[3], k3[3];
  float bq[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) bq[j] = bs[qt][qc + (j >> 2) * 8 + (j & 3)];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = q[j] * __builtin_amdgcn_exp2f(bq[j]);
  bf16_pieces(v, p3);
#pragma unroll
  for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4 *>(rec + i * Rec::kPiece + tid * 16) = p3[i];
  floatx16 part;                                             // A^T over the wave's 16 channels: lane (hi, t), rows s
#pragma unroll
  for (int r = 0; r < 16; ++r) part[r] = 0.f;
  if (!apart) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = ks[qt][qc + (j >> 2) * 8 + (j & 3)] * __builtin_amdgcn_exp2f(-bq[j]);
    bf16_pieces(v, k3);
    bf16x8 x[3], y[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      x[i] = __builtin_bit_cast(bf16x8, k3[i]);
      y[i] = __builtin_bit_cast(bf16x8, p3[i]);
    }
    part = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[2], y[0], part, 0, 0, 0);
    part = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[0], y[2], part, 0, 0, 0);
    part = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[1], y[1], part, 0, 0, 0);
    part = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[1], y[0], part, 0, 0, 0);
    part = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[0], y[1], part, 0, 0, 0);
    part = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[0], y[0], part, 0, 0, 0);
  }
  {
    const int d = (tid >> 7) * 32 + qt, s0 = (tid >> 6 & 1) * 16 + hi * 8;    // Kd's: channel d, eight tokens
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = ks[s0 + j][d] * __builtin_amdgcn_exp2f(left[j]);
    bf16_pieces(v, k3);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4 *>(rec + Rec::kK + i * Rec::kPiece + tid * 16) = k3[i];
  }
  if (tid < DK) reinterpret_cast<float *>(rec + Rec::kDec)[tid] = __builtin_amdgcn_exp2f(bs[kGB - 1][tid]);
  __syncthreads();
  if (!apart) {                                              // the waves' parts added up
    float (*parts)[kGB][kGB] = reinterpret_cast<float (*)[kGB][kGB]>(&kb2[0][0][0]);     // [wave][s][t]
#pragma unroll
    for (int r = 0; r < 16; ++r) parts[kb][(r >> 2) * 8 + hi * 4 + (r & 3)][qt] = part[r];
    __syncthreads();
    for (int i = tid; i < kGB * kGB; i += TH) {
      const int s = i / kGB, tt = i % kGB;
      float x = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) x += parts[w][s][tt];
      am[tt][s] = s <= tt ? x : 0.f;
    }
  } else {
    auto load_row = [&](const float *row, float (&x)[8]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 8; i += 4) {
        const float4 y = *reinterpret_cast<const float4 *>(row + i / 4 * (DK / 2) + l * 4);
        x[i] = y.x; x[i + 1] = y.y; x[i + 2] = y.z; x[i + 3] = y.w;
      }
    };
    float bt[8], q[8];
    load_row(bs[t], bt);
    load_bf16(pr + min(t, len - 1) * a.ld + h * DK + l * 4, q, DK / 2);
#pragma unroll
    for (int i = 0; i < 8; ++i) q[i] = t < len ? q[i] * a.q_scale : 0.f;
    const int my = t >> 3;
    if (my) {
      float ref[8], qh[8];
      load_row(bs[my * 8 - 1], ref);
#pragma unroll
      for (int i = 0; i < 8; ++i) qh[i] = q[i] * __builtin_amdgcn_exp2f(bt[i] - ref[i]);
      for (int s = 0; s < my * 8; ++s) {                     // keys towards the boundary
        float kv[8], bv[8], acc = 0.f;
        load_row(ks[s], kv);
        load_row(bs[s], bv);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc = fmaf(qh[i], kv[i] * __builtin_amdgcn_exp2f(ref[i] - bv[i]), acc);
        acc = group_sum<LPT>(acc);
        if (l == 0) am[t][s] = acc;
      }
    }
    for (int s = my * 8; s < my * 8 + 8; ++s) {
      float kv[8], bv[8], acc = 0.f;
      load_row(ks[s], kv);
      load_row(bs[s], bv);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc = fmaf(q[i] * kv[i], __builtin_amdgcn_exp2f(fminf(bt[i] - bv[i], 0.f)), acc);
      acc = group_sum<LPT>(acc);
      if (l == 0 && s <= t) am[t][s] = acc;
    }
  }
  __syncthreads();
  if (tid < 128) {                                           // A's items: token lane & 31, eight tokens s
    const int s0 = (tid >> 6) * 16 + hi * 8;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = am[qt][s0 + j];
    bf16_pieces(v, p3);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4 *>(rec + Rec::kA + i * Rec::kAPiece + tid * 16) = p3[i];
  }
}

// Inclusive sum over the wave's lanes, on the vector ALU.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_add_int(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ int wave_sums_up_to(int v) {
  v = dpp_add_int<0x111, 0xf>(v);      // row_shr 1, 2, 4, 8: within rows of 16 lanes
  v = dpp_add_int<0x112, 0xf>(v);
  v = dpp_add_int<0x114, 0xf>(v);
  v = dpp_add_int<0x118, 0xf>(v);
  v = dpp_add_int<0x142, 0xa>(v);      // row_bcast 15 into rows 1 and 3
  return dpp_add_int<0x143, 0xc>(v);   // row_bcast 31 into rows 2 and 3
}

// The blocks of up to 64 sequences in a row, cut into `units` equal stretches: lane s has sequence s of `own` blocks,
// first .. end - 1 of all.  Products stay within 2^31: there are up to 2^22 blocks and 512 stretches.
__device__ __forceinline__ void stretch_ranges(int own, int &first, int &end, int &all) {
  end = wave_sums_up_to(own);
  first = end - own;
  all = __builtin_amdgcn_readlane(end, 63);
}
__device__ __forceinline__ int stretch_begin(int unit, int units, int all) { return static_cast<unsigned int>(unit) * all / static_cast<unsigned int>(units); }
__device__ __forceinline__ int stretch_of(int block, int units, int all) { return (static_cast<unsigned int>(block + 1) * units - 1) / static_cast<unsigned int>(all); }

// Lane s: blocks of sequence s.
__device__ __forceinline__ int gla_own_blocks(const GlaArgs &a, int lane) { return lane < a.seqs ? (a.cu_chunks[lane + 1] - a.cu_chunks[lane] + 1) / 2 : 0; }

// MODE 0: the whole sequence from the state slot and back.  MODE 1: from zero, what a stretch adds to the sequence that goes on behind it.
// MODE 2: a stretch; that sequence starts from seg_state[unit], one that began before the stretch and ends in it from seg_state[units + unit].
template <int DK, int MODE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gla_block_scan_kernel(const GlaArgs a, int first_seq) {
  typedef unsigned short T;
  using Rec = GlaBlock<DK>;
  constexpr int NI = DK / 32, VB = kGB * 32 * 2;             // tiles of S, bytes of a wave's rows of v
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, hi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = a.dv / 32;
  const int h = blockIdx.x;
  const unsigned int recs = TLF_DL_LDSADDR(lds), vs = recs + 2 * Rec::kSize + wave * 2 * VB;
  float *rowsum = reinterpret_cast<float *>(lds + 2 * Rec::kSize + waves * 2 * VB);        // [2][waves][32]
  int *const ranges = reinterpret_cast<int *>(rowsum + 2 * waves * 32);                    // MODE 1 and 2: [2][64]
  unsigned long long left = 1;                               // sequences of the stretch
  int lo = 0, hi_block = 0;
  if constexpr (MODE != 0) {
    int first, end, all;
    stretch_ranges(gla_own_blocks(a, lane), first, end, all);
    if (all == 0) return;
    lo = stretch_begin(blockIdx.z, a.units, all);
    hi_block = stretch_begin(blockIdx.z + 1, a.units, all);
    left = __ballot(first < hi_block && end > lo);
    if (left == 0) return;
    if constexpr (MODE == 1) {
      const int last = 63 - __builtin_clzll(left);
      if (__builtin_amdgcn_readlane(end, last) <= hi_block) return;    // the stretch ends with it
      left = 1ull << last;
    }
    if (wave == 0) {
      ranges[lane] = first;
      ranges[64 + lane] = end;
    }
    lds_barrier();
  }
  do {
  const int seq = MODE == 0 ? blockIdx.z : __builtin_ctzll(left);
  const int first_block = MODE == 0 ? 0 : __builtin_amdgcn_readfirstlane(ranges[seq]), end_block = MODE == 0 ? 0 : __builtin_amdgcn_readfirstlane(ranges[64 + seq]);
  const bool ends = MODE == 0 || end_block <= hi_block, begins = MODE == 0 || first_block >= lo;
  const int slot = load_uniform(a.state_slots + first_seq + seq);
  const bool slot_ok = slot >= 0 && slot < a.num_slots;
  float *st = a.state + (static_cast<int64_t>(slot_ok ? slot : 0) * a.H + h) * DK * a.dv;
  const int64_t sg = static_cast<int64_t>(MODE != 0 && ends ? a.units + blockIdx.z : blockIdx.z) * a.H + h;
  float *gst = ends && begins ? st : a.seg_state + sg * DK * a.dv;
  const bool from_zero = MODE == 1 || (ends && begins && (!slot_ok || a.starts[first_seq + seq] == 0));
  // lane (hi, n), register r of tile i: row 32 i + 8 (r / 4) + 4 hi + r % 4 of column n.  A row's address is the same in all lanes and the lane's part
  // one register: 64 addresses would go to memory, and each that comes back waits for all values before it.
  const unsigned int mine = static_cast<unsigned int>(hi * 4 * a.dv + wave * 32 + n) * 4;
  auto row_of = [&](int i, int r) __attribute__((always_inline)) { return static_cast<int64_t>(i * 32 + (r >> 2) * 8 + (r & 3)) * a.dv * 4; };
  floatx16 S[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) S[i][r] = 0.f;
  if (!from_zero) {
    const char *from = reinterpret_cast<const char *>(gst);
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) S[i][r] = *reinterpret_cast<const float *>(from + row_of(i, r) + mine);
  }
  const int64_t hk = static_cast<int64_t>(a.H) * DK;
  const int cbeg = load_uniform(a.cu_chunks + seq), cend = load_uniform(a.cu_chunks + seq + 1), blocks = (cend - cbeg + 1) / 2;
  const int64_t row0 = cbeg < cend ? load_uniform(a.chunk_tok + cbeg) : 0;
  const int tokens = cbeg < cend ? (cend - 1 - cbeg) * 16 + load_uniform(a.chunk_len + cend - 1) : 0;
  const int b0 = MODE == 0 ? 0 : max(lo - first_block, 0), b1 = MODE == 0 ? blocks : min(hi_block - first_block, blocks);
  const T *vbase = static_cast<const T *>(a.proj) + 2 * hk + static_cast<int64_t>(h) * a.dv + wave * 32;
  const T *gbase = vbase + static_cast<int64_t>(a.H) * a.dv + hi * 4;
  const unsigned char *rbase = reinterpret_cast<const unsigned char *>(a.rec) + (static_cast<int64_t>(gla_first_block(cbeg, a.seq0 + seq)) * a.H + h) * Rec::kSize;
  // Two waves of a SIMD leave a barrier together and would go through products, and through what is vector instructions, at the same time.
  // So the first four waves take the copies and finish the block before, then come to the products; the others begin with the products and
  // finish the block before behind them.
  const int early = min(waves, 4);
  auto copy = [&](int b, int buf) __attribute__((always_inline)) {
    const unsigned char *rec = rbase + static_cast<int64_t>(b) * a.H * Rec::kSize;
    if (MODE == 1 || wave < early) {
      const int step = MODE == 1 ? waves : early;
      for (int i = (MODE == 1 ? Rec::kK / 1024 : 0) + wave; i < (MODE == 1 ? Rec::kA : Rec::kSize) / 1024; i += step)
        dl_copy(lane * 16, rec + i * 1024, recs + buf * Rec::kSize + i * 1024);
    }
    if (MODE == 1 && wave == waves - 1) dl_copy(lane * 16, rec + Rec::kDec, recs + buf * Rec::kSize + Rec::kDec);
    const T *vp = vbase + (row0 + static_cast<int64_t>(b) * kGB) * a.ld;
    const int last = min(kGB, tokens - b * kGB) - 1;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = min(j * 16 + (lane >> 2), last);
      dl_copy(static_cast<unsigned int>(row * static_cast<int>(a.ld) * 2 + (lane & 3) * 16), vp, vs + buf * VB + j * 1024);
    }
  };
  uint2 nw[MODE == 1 ? 1 : 4];
  if constexpr (MODE != 1) {
#pragma unroll
    for (int c = 0; c < 4; ++c) nw[c] = *reinterpret_cast<const uint2 *>(static_cast<const T *>(a.norm_w) + wave * 32 + c * 8 + hi * 4);
  }
  floatx16 o;                                                // of the block before: lane (hi, n): token n, columns 8 (r / 4) + 4 hi + r % 4
  uint2 gate[4];
  auto put = [&](int b, int buf) __attribute__((always_inline)) {
    float ss = 0.f;
    if (waves == 8) {                                        // all at once; with room for eight, fewer lose (4 heads of 64 x 64, one of 3000 tokens, layer 56.7 us, 55.4 so)
      float parts[8];
#pragma unroll
      for (int w = 0; w < 8; ++w) parts[w] = rowsum[(buf * 8 + w) * 32 + n];
#pragma unroll
      for (int w = 0; w < 8; ++w) ss += parts[w];
    } else {
      for (int w = 0; w < waves; ++w) ss += rowsum[(buf * waves + w) * 32 + n];
    }
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(a.dv) + a.eps);
    if (n >= tokens - b * kGB) return;
    T *out = static_cast<T *>(a.out) + (row0 + static_cast<int64_t>(b) * kGB + n) * a.ldo + static_cast<int64_t>(h) * a.dv + wave * 32 + hi * 4;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float g[4] = {__uint_as_float(gate[c].x << 16), __uint_as_float(gate[c].x & 0xffff0000u), __uint_as_float(gate[c].y << 16),
                          __uint_as_float(gate[c].y & 0xffff0000u)};
      const float w[4] = {__uint_as_float(nw[c].x << 16), __uint_as_float(nw[c].x & 0xffff0000u), __uint_as_float(nw[c].y << 16), __uint_as_float(nw[c].y & 0xffff0000u)};
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        y[e] = o[c * 4 + e] * inv * w[e] * g[e] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * g[e]));
      *reinterpret_cast<uint2 *>(out + c * 8) = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
    }
  };
  float sd[DK >= 64 ? DK / 64 : 1];                          // MODE 1: decay of the whole segment
#pragma unroll
  for (float &x : sd) x = 1.f;

  if (b0 < b1) copy(b0, 0);
  for (int b = b0; b < b1; ++b) {
    const int buf = (b - b0) & 1;
    // addresses are made from the lane anew in each block: kept, they would not fit beside the state
    int here = tid & 63;
    asm volatile("" : "+v"(here));
    const int lane = here, n = here & 31, hi = here >> 5;
    TLF_DL_BARRIER_KNOWN();                                  // the gate of the block before, too
    if (b + 1 < b1) copy(b + 1, buf ^ 1);
    if constexpr (MODE != 1) {
      if (wave < early && b > b0) put(b - 1, buf ^ 1);
    }
    const int len = min(kGB, tokens - b * kGB);
    const unsigned int rec = recs + buf * Rec::kSize, vt = vs + buf * VB;
    if (len < kGB) {                                         // rows behind the sequence: zeros, whatever lies there
      for (int i = len * 4 + lane; i < kGB * 4; i += 64)
        *reinterpret_cast<u32x4 __attribute__((address_space(3))) *>(vt + i * 16) = u32x4{0, 0, 0, 0};
      wave_lds_fence();
    }
    auto tile = [&](unsigned int at) __attribute__((always_inline)) {
      return *reinterpret_cast<const bf16x8 __attribute__((address_space(3))) *>(at + lane * 16);
    };
    bf16x8 vf[2];                                            // lane (hi, n): column n, tokens 16 tb + 8 hi ..
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      const unsigned int at = vt + (tb * 16 + hi * 8 + (lane >> 2 & 3)) * 64 + (lane >> 4 & 1) * 32 + (lane & 3) * 8;
      const uint2 x = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<shortx4 __attribute__((address_space(3))) *>(at)));
      const uint2 y = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<shortx4 __attribute__((address_space(3))) *>(at + 256)));
      vf[tb] = __builtin_bit_cast(bf16x8, make_uint4(x.x, x.y, y.x, y.y));
    }
    if constexpr (MODE != 1) {
      const T *gp = gbase + (row0 + static_cast<int64_t>(b) * kGB + min(n, len - 1)) * a.ld;
      auto load_gate = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; ++c) gate[c] = *reinterpret_cast<const uint2 *>(gp + c * 8);
      };
      if (wave < early) load_gate();
      floatx16 o0, o1;
#pragma unroll
      for (int r = 0; r < 16; ++r) o0[r] = o1[r] = 0.f;
      // a step of 16 channels: its products, behind them the pieces of the next and the reads of the one after that
      bf16x8 s3[2][3], q3[2][3];
      auto pieces = [&](int kb) __attribute__((always_inline)) {
        float x[8];
        uint4 p[3];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = S[kb / 2][kb % 2 * 8 + j];
        bf16_pieces(x, p);
#pragma unroll
        for (int i = 0; i < 3; ++i) s3[kb & 1][i] = __builtin_bit_cast(bf16x8, p[i]);
      };
      auto read = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 3; ++i) q3[kb & 1][i] = tile(rec + i * Rec::kPiece + kb * 1024);
      };
      // The block's second half of tokens first: for the tokens before it these are zeros times values that may be no number, which
      // they drop.
      bf16x8 af[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) af[i] = tile(rec + Rec::kA + i * Rec::kAPiece + 1024);
      read(0);
      read(1);
#pragma unroll
      for (int i = 0; i < 3; ++i) o1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[1], af[i], o1, 0, 0, 0);
      pieces(0);
#pragma unroll
      for (int r = 0; r < 16; ++r) o1[r] = n < 16 ? 0.f : o1[r];
#pragma unroll
      for (int kb = 0; kb < DK / 16; ++kb) {
        __builtin_amdgcn_sched_barrier(0);
        const auto &x = s3[kb & 1], &q = q3[kb & 1];
        o0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[0], q[0], o0, 0, 0, 0);
        o1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[0], q[1], o1, 0, 0, 0);
        o0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[1], q[0], o0, 0, 0, 0);
        o1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[1], q[1], o1, 0, 0, 0);
        o0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[0], q[2], o0, 0, 0, 0);
        o1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[2], q[0], o1, 0, 0, 0);
        if (kb + 1 < DK / 16) pieces(kb + 1);
        if (kb + 2 < DK / 16) read(kb + 2);
        if (kb + 2 == DK / 16) {
#pragma unroll
          for (int i = 0; i < 3; ++i) af[i] = tile(rec + Rec::kA + i * Rec::kAPiece);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 3; ++i) o0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[0], af[i], o0, 0, 0, 0);
      if (wave >= early) {
        if (b > b0) put(b - 1, buf ^ 1);
        load_gate();
      }
      float ss = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        o[r] = o0[r] + o1[r];
        ss = fmaf(o[r], o[r], ss);
      }
      const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(ss), __float_as_uint(ss), false, false);
      ss = __uint_as_float(both[0]) + __uint_as_float(both[1]);
      if (hi == 0) rowsum[(buf * waves + wave) * 32 + n] = ss;
    }
    const unsigned int dec = rec + Rec::kDec;
    if constexpr (MODE == 1) {
#pragma unroll
      for (int j = 0; j < static_cast<int>(sizeof(sd) / 4); ++j) sd[j] *= *reinterpret_cast<const float __attribute__((address_space(3))) *>(dec + (j * 64 + lane % DK) * 4);
    }
    // six groups of products, the operands of the next group read behind those of this one
    bf16x8 kf[2][NI];
    auto read_k = [&](int at) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NI; ++i) kf[at & 1][i] = tile(rec + Rec::kK + at / 2 * Rec::kPiece + (i * 2 + (at & 1)) * 1024);
    };
    read_k(0);
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const floatx4 f = *reinterpret_cast<const floatx4 __attribute__((address_space(3))) *>(dec + (i * 32 + c * 8 + hi * 4) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) S[i][c * 4 + e] *= f[e];
      }
#pragma unroll
    for (int at = 0; at < 6; ++at) {                         // piece at / 2, tokens 16 (at & 1) ..
      __builtin_amdgcn_sched_barrier(0);
      if (at + 1 < 6) read_k(at + 1);
#pragma unroll
      for (int i = 0; i < NI; ++i) S[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[at & 1][i], vf[at & 1], S[i], 0, 0, 0);
    }
  }
  if constexpr (MODE == 1) {
    if (wave == 0) {
#pragma unroll
      for (int j = 0; j < static_cast<int>(sizeof(sd) / 4); ++j)
        if (lane < DK) a.seg_dec[sg * DK + j * 64 + lane] = sd[j];
    }
  } else {
    if (b0 < b1) {
      TLF_DL_BARRIER_KNOWN();
      put(b1 - 1, (b1 - 1 - b0) & 1);
    }
  }
  if (MODE == 1 || (ends && slot_ok)) {
    char *to = reinterpret_cast<char *>(MODE == 1 ? gst : st);
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) *reinterpret_cast<float *>(to + row_of(i, r) + mine) = S[i][r];
  }
  left &= left - 1;
  } while (MODE == 2 && left);
}

// What the stretches add to a sequence -> the states they start from: seg_state[unit] in place, seg_state[units + unit] where it ends.
__global__ __launch_bounds__(256) void gla_stretches_kernel(const GlaArgs a, int first_seq) {
  const int64_t plane = static_cast<int64_t>(a.dk) * a.dv, e = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  const int h = blockIdx.y, seq = blockIdx.z;
  int first, end, all;
  stretch_ranges(gla_own_blocks(a, threadIdx.x & 63), first, end, all);
  first = __builtin_amdgcn_readlane(first, seq);
  end = __builtin_amdgcn_readlane(end, seq);
  if (first == end) return;
  const int from = stretch_of(first, a.units, all), to = stretch_of(end - 1, a.units, all);
  if (from == to || e >= plane) return;                      // in one stretch
  const int slot = a.state_slots[first_seq + seq];
  const bool from_zero = slot < 0 || slot >= a.num_slots || a.starts[first_seq + seq] == 0;
  auto at = [&](float *states, int64_t i) __attribute__((always_inline)) { return reinterpret_cast<float4 *>(states + (i * a.H + h) * plane + e); };
  float4 run = from_zero ? make_float4(0.f, 0.f, 0.f, 0.f) : *at(a.state, slot);
  const int d = static_cast<int>(e / a.dv);
  for (int u = from; u < to; ++u) {
    float4 *const p = at(a.seg_state, u);
    const float4 own = *p;
    const float dec = a.seg_dec[(static_cast<int64_t>(u) * a.H + h) * a.dk + d];
    *p = run;
    run = make_float4(fmaf(dec, run.x, own.x), fmaf(dec, run.y, own.y), fmaf(dec, run.z, own.z), fmaf(dec, run.w, own.w));
  }
  *at(a.seg_state, a.units + to) = run;
}

// A workgroup of the scan has a wave per 32 value columns and holds two records, 117 KB with 128 keys: with fewer than three waves there, or
// two otherwise, a CU has too few to hide their latencies, and the 16-token chunks are faster.  8 heads, 16-token chunks / blocks, us, at
// 64 x 128, 8 x 300 and 8 x 2048 tokens: 128 x 32 90 / 118, 68 / 81, 231 / 288, 128 x 64 99 / 118, 69 / 71, 268 / 278, 128 x 96 128 / 118,
// 68 / 68, 345 / 283; 64 x 32 66 / 69, 49 / 54, 137 / 142, 64 x 64 71 / 73, 50 / 49, 152 / 151; 32 x 32 55 / 52, 36 / 42, 111 / 105 (1 x 1500
// 50 / 53).
bool gla_blocks_sizes(int32_t dk, int32_t dv) {
  return (dk == 32 || dk == 64 || dk == 128) && dv % 32 == 0 && dv >= (dk == 128 ? 96 : 64) && dv <= 256;
}

// Segments that a sequence would have: a workgroup for every CU (two where LDS holds two), segments of at least 8 blocks.
int gla_block_segments(int chunks, int seqs, int heads, int dk) {
  const int64_t wgs = static_cast<int64_t>(seqs) * heads, full = dk == 128 ? 256 : 512, want = wgs >= full ? 1 : (full + wgs - 1) / wgs, most = chunks / seqs / 16;
  const int64_t s = want < most ? want : most;
  return static_cast<int>(s < 1 || seqs * s > 65535 ? 1 : s > 32 ? 32 : s);
}

// A launch cuts up to 64 sequences; more go in groups, one after the other.
constexpr int kGroup = 64;
inline int gla_groups(int seqs) { return (seqs + kGroup - 1) / kGroup; }

// Stretches of each group, 0: sequences are never cut.  A workgroup for every CU, with a stretch of at least 8 blocks.
int gla_block_units(int chunks, int seqs, int heads, int dk) {
  if (chunks > (1 << 22) || gla_block_segments(chunks, seqs, heads, dk) == 1) return 0;
  const int units = std::min((dk == 128 ? 256 : 512) / heads, chunks / 16 / gla_groups(seqs));
  return units > 1 ? units : 0;
}

// Whether that is faster than whole sequences, the longest of `longest` tokens (0: not known).  With half as many stretches again as sequences
// it always is.  Otherwise a launch of whole ones takes as long as its longest, and the two passes over stretches 1.3 x an even share and some
// eight blocks' time more.  16 heads of 128 x 256, the layer, us, cut / whole: 12 sequences of 700 tokens 343 / 307, of 450 to 900 289 / 294, of 300
// to 1500 382 / 444; one of 1500 with 11 of 450 242 / 377, one of 8192 with 11 of 100 330 / 1630; 2 heads, one of 8192 with 99 of 450 300 / 1590.
bool gla_blocks_cut(int units, int chunks, int seqs, int longest) {
  const int64_t groups = gla_groups(seqs), most = (static_cast<int64_t>(longest) + kGB - 1) / kGB, all = (static_cast<int64_t>(chunks) + 1) / 2;
  if (units == 0) return false;
  if (longest <= 0 || (groups == 1 && units * 2 >= seqs * 3)) return true;
  return most * 10 * units >= all * 13 + groups * units * 80;
}

// Whether the scan over 16-token chunks does as well: where its waves, one per 16 value columns, are all on the chip at once, in one segment,
// and go through few chunks.  A block takes a workgroup of dv / 32 waves as long as it takes them for two and a half chunks (eight waves
// wait at one barrier), so with wide values five chunks are enough to be faster, with narrower ones fourteen, and only where CUs are
// idle; and a second segment is not worth its first pass there.  Layer, us, chunks / blocks: 16 heads of 128 x 256, 1 x 70 tokens 32 / 31,
// 1 x 130 36 / 42, 1 x 400 65 / 90, 1 x 550 (two segments) 117 / 100, 4 x 130 46 / 51, 5 x 200 (1280 waves) 81 / 67, 4 x 500 95 / 127,
// 4 x 1000 183 / 168; 8 of 64 x 128 1 x 130 31 / 27, 1 x 400 43 / 46, 12 x 400 (96 workgroups) 65 / 60; 16 of 128 x 128 8 x 500 118 / 143.
bool gla_chunks_suffice(const GlaArgs &a, int chunk_segs) {
  const int64_t wgs = static_cast<int64_t>(a.seqs) * a.H, waves = (a.dv + 15) / 16 * wgs;
  const int each = (a.chunks + a.seqs - 1) / a.seqs;
  if (waves > 1024 || chunk_segs > 1 || each > 40) return false;
  if (a.dv > 128) return each >= 5;
  return gla_block_segments(a.chunks, a.seqs, a.H, a.dk) > 1 || (wgs <= 64 && each >= 14);
}

bool gla_blocks_take(const GlaArgs &a, int32_t dtype, int chunk_segs) {
  return dtype == TLF_DT_BF16 && gla_blocks_sizes(a.dk, a.dv) && a.R <= kGlaBlockMaxR && a.ld % 8 == 0 && a.ld < (1 << 24) && a.ldo % 4 == 0 && aligned16(a.proj) &&
         (reinterpret_cast<uintptr_t>(a.out) & 7) == 0 && (reinterpret_cast<uintptr_t>(a.norm_w) & 7) == 0 &&
         !gla_chunks_suffice(a, chunk_segs);
}

size_t gla_blocks_workspace_bytes(int32_t chunks, int32_t seqs, int32_t heads, int32_t dk, int32_t dv) {
  const size_t slots = (static_cast<size_t>(chunks) + seqs + 1) / 2 + 1, units = gla_block_units(chunks, seqs, heads, dk);
  return slots * heads * gla_block_record(dk) + 4 * units * heads * (dk + 2 * static_cast<size_t>(dk) * dv);
}

template <int DK>
int launch_gla_blocks_of(GlaArgs &a, int first_seq, hipStream_t stream) {
  const int waves = a.dv / 32;
  const size_t lds = 2 * GlaBlock<DK>::kSize + waves * (2 * kGB * 32 * 2 + 2 * 32 * 4) + (a.units ? 2 * 64 * 4 : 0);
  constexpr int kMost = 2 * GlaBlock<DK>::kSize + 8 * (2 * kGB * 32 * 2 + 2 * 32 * 4) + 2 * 64 * 4;
  static const hipError_t allowed = [] {
    hipError_t e = hipSuccess;
    for (const void *k : {reinterpret_cast<const void *>(&gla_block_scan_kernel<DK, 0>), reinterpret_cast<const void *>(&gla_block_scan_kernel<DK, 1>),
                          reinterpret_cast<const void *>(&gla_block_scan_kernel<DK, 2>)})
      if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kMost);
    return e;
  }();
  if (allowed != hipSuccess) return static_cast<int>(allowed);
  TLF_LAUNCH((gla_block_kernel<DK>), dim3((a.chunks + a.seqs + 1) / 2, a.H), dim3(DK * 4), 0, stream, a);
  if (!a.units) {
    TLF_LAUNCH((gla_block_scan_kernel<DK, 0>), dim3(a.H, 1, a.seqs), dim3(waves * 64), lds, stream, a, first_seq);
    return launch_status();
  }
  const dim3 grid(a.H, 1, a.units);
  const int seqs = a.seqs, each = (seqs + gla_groups(seqs) - 1) / gla_groups(seqs);
  const int32_t *cu_chunks = a.cu_chunks;
  for (a.seq0 = 0; a.seq0 < seqs; a.seq0 += each) {
    a.seqs = std::min(each, seqs - a.seq0);
    a.cu_chunks = cu_chunks + a.seq0;
    TLF_LAUNCH((gla_block_scan_kernel<DK, 1>), grid, dim3(waves * 64), lds, stream, a, first_seq + a.seq0);
    TLF_LAUNCH(gla_stretches_kernel, dim3((DK * a.dv + 1023) / 1024, a.H, a.seqs), dim3(256), 0, stream, a, first_seq + a.seq0);
    TLF_LAUNCH((gla_block_scan_kernel<DK, 2>), grid, dim3(waves * 64), lds, stream, a, first_seq + a.seq0);
  }
  return launch_status();
}

int launch_gla_blocks(GlaArgs &a, int first_seq, int longest, void *workspace, hipStream_t stream) {
  a.units = aligned16(a.state) ? gla_block_units(a.chunks, a.seqs, a.H, a.dk) : 0;
  if (!gla_blocks_cut(a.units, a.chunks, a.seqs, longest)) a.units = 0;
  const size_t slots = (static_cast<size_t>(a.chunks) + a.seqs + 1) / 2 + 1;
  a.rec = static_cast<float *>(workspace);
  a.seg_dec = a.rec + slots * a.H * gla_block_record(a.dk) / 4;
  a.seg_state = a.seg_dec + static_cast<size_t>(a.units) * a.H * a.dk;
  switch (a.dk) {
    case 32: return launch_gla_blocks_of<32>(a, first_seq, stream);
    case 64: return launch_gla_blocks_of<64>(a, first_seq, stream);
    default: return launch_gla_blocks_of<128>(a, first_seq, stream);
  }
}

}  // namespace tlf
