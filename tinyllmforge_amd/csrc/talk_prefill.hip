// Attention of talk_attn.h for prompt portions, bf16, on the matrix cores, from the paged cache.  Mixing needs every head's
// weights, and weights need their denominators, so there are two kernels:
//
//   talk_stats_kernel    log2 of every (row, head)'s sum of exponentials: m + log2 l.  A workgroup owns one KV head and 128 units
//                        (row, head) of it and walks the keys 64 at a time through LDS; S^T[key, unit] = K . Q^T (prompt_core.h).
//   talk_prefill_kernel  a workgroup owns 16 RT query rows with all their heads, a wave 16 rows of four heads, or 32 rows of two, or 64
//                        of one (those that share a KV head), and walks the keys 32 at a time:
//     S^T[key, row] = K . Q^T per head, K straight from the caches in operand order, half a tile ahead;
//     W = 2^(S - m - log2 l), complete weights, as a bf16 hi + lo pair (16 significant bits) into LDS, [row][key][head];
//     per row (dealt to the waves) M^T[key, head] = W^T . talk^T, back into the row's place in LDS as a pair, [row][head][key];
//     O^T[dim, row] += V^T . M^T per head, V^T by LDS transpose reads of a tile that all waves share.
//
// Nothing is rescaled.  The rows of two 16-key tiles are picked so that their accumulators are eight consecutive keys.  V travels
// from the cache into LDS directly, behind the weights and the mix; rows are unpadded and pairs of their 16-byte pieces swizzled
// against bank conflicts (the lane that fills a position picks the matching piece).
//
// A wave of the second kernel has 128 accumulators and 64 registers of q, and the scheduler is held back where it would gather operands:
// with q partly in memory a tile of 32 rows took 14800 cycles, 9800 of them before the mix, waiting for it behind the loads of K; so 11000,
// 3600 of them products.  Eight prompts of 1061 to 2048 tokens, 128 dimensions, both kernels: 16 heads on 8 KV heads 500 -> 357 us, on 4
// 455 -> 331, 32 heads 734 -> 612.
//
// A workgroup fills a compute unit, and a launch of whole tiles ends with its longest one, 64 steps of 4.8 us at 2048 keys where an even share is
// 39.  So the keys of long tiles are cut (talk_split.h): a workgroup of the first kernel plans it beside the others' work, the second one's take
// tiles and parts from its list, and talk_join_kernel adds up what the parts of a tile have left in fp32: 312 -> 246 + 15 us.
#include <algorithm>

#include "gemm_shared.h"
#include "prompt_core.h"
#include "prompt_tiles.h"
#include "talk_attn.h"
#include "talk_split.h"

namespace tlf {

constexpr int kTK = 32;             // keys per tile
constexpr int kTM = kTK + 8;        // keys of a head's mixed weights, padded

// How row tiles are cut; plan NULL: they stay whole, a workgroup each.
struct TalkSplit {
  int32_t *plan;                    // steps of a part, items, tiles that are cut, items taken beyond each workgroup's first
  int4 *items, *cuts;               // (sequence, row tile, first key tile, slot); (sequence, row tile, its first extra part's slot, extra parts)
  floatx4 *parts;                   // slots of `size`: `most` extra parts, then what stays with a tile
  int32_t seqs, xtiles, tq, most, size;
};

struct TalkPrefillArgs {
  SinkCache c;
  const unsigned short *q;          // [rows, H, Dp]
  const unsigned short *talk;       // [H, H]
  float *stats;                     // [rows, H]
  const int32_t *cu_q, *starts;
  unsigned short *out;
  int64_t ldo;
  int32_t H, group;
  int32_t hpp, passes, bq;          // stats: query heads per pass, passes, rows per workgroup
  PromptTiles tiles;
  TalkSplit split;
  int32_t first_seq, table_cols;
};

// Where a sequence's portion lies; rows that the block table does not reach are left out.
__device__ __forceinline__ void talk_portion(const TalkPrefillArgs &p, int sq, int &start, int &tokens) {
  const int seq = p.first_seq + sq;
  start = p.starts[seq];
  tokens = p.cu_q[seq + 1] - p.cu_q[seq];
  if (start + static_cast<int64_t>(tokens) > static_cast<int64_t>(p.table_cols) * p.c.bs) tokens = 0;
}

// Key tiles from `first` on; slot: where partial sums go, < 0: the result itself.
struct TalkItem {
  int sq, xt, first, slot;
};

// One workgroup of 256: how the row tiles of the second kernel are cut, and the order of the work.  A thread has a row tile.
__device__ __forceinline__ void talk_plan(const TalkPrefillArgs &p, int32_t *shared) {
  const TalkSplit &sp = p.split;
  constexpr int kMine = (kTalkTiles + 255) / 256;
  const int tid = threadIdx.x;
  int sq[kMine], xt[kMine], steps[kMine], all = 0;
#pragma unroll
  for (int m = 0; m < kMine; ++m) steps[m] = 0;
  for (int first = 0; first < sp.seqs; first += 256) {
    int start = 0, tokens = 0;
    if (first + tid < sp.seqs) talk_portion(p, first + tid, start, tokens);
    __syncthreads();
    shared[tid] = start;
    shared[256 + tid] = min(talk_tiles(tokens, sp.tq), sp.xtiles);
    shared[512 + tid] = tokens;
    __syncthreads();
    for (int s = 0; s < min(256, sp.seqs - first); ++s) {
      const int n = min(shared[256 + s], kTalkTiles - all);
#pragma unroll
      for (int m = 0; m < kMine; ++m) {
        const int x = tid + m * 256 - all;
        if (x < 0 || x >= n) continue;
        sq[m] = first + s;
        xt[m] = x;
        steps[m] = talk_steps(shared[s], shared[512 + s], sp.tq, x);
      }
      all += n;
    }
  }
  __syncthreads();
  auto sum_of = [&](auto value) {                                    // over all tiles
    int v = 0;
#pragma unroll
    for (int m = 0; m < kMine; ++m) v += steps[m] ? value(steps[m]) : 0;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) v += __shfl_xor(v, d);
    __syncthreads();
    if ((tid & 63) == 0) shared[tid >> 6] = v;
    __syncthreads();
    return (shared[0] + shared[1]) + (shared[2] + shared[3]);
  };
  const int64_t work = sum_of([](int n) { return n >> 12; }) * 4096ll + sum_of([](int n) { return n & 4095; });
  auto extras_of = [&](int per) { return sum_of([&](int n) { return min(talk_extras(n, per), kTalkExtras); }); };
  const int per = talk_per(work, all, extras_of), items = all + extras_of(per);
  int32_t *const count = shared + 4, *const taken = shared + 4 + 128;      // by length; slots, cut tiles
  __syncthreads();
  if (tid < 128 + 2) count[tid] = 0;
  __syncthreads();
#pragma unroll
  for (int m = 0; m < kMine; ++m)
    if (steps[m]) {
      const int extras = talk_extras(steps[m], per);
      if (extras) atomicAdd(count, extras);
      atomicAdd(count + talk_class(steps[m] - extras * per, per), 1);
    }
  __syncthreads();
  int before = 0;                                                    // a class's place
  if (tid < 128)
    for (int i = 0; i < tid; ++i) before += count[i];
  __syncthreads();
  if (tid < 128) count[tid] = before;
  __syncthreads();
#pragma unroll
  for (int m = 0; m < kMine; ++m)
    if (steps[m]) {
      const int extras = talk_extras(steps[m], per);
      int slot = -1;
      if (extras) {
        const int first = atomicAdd(taken, extras), cut = atomicAdd(taken + 1, 1);
        for (int i = 0; i < extras; ++i) sp.items[atomicAdd(count, 1)] = make_int4(sq[m], xt[m], i * per, first + i);
        sp.cuts[cut] = make_int4(sq[m], xt[m], first, extras);
        slot = sp.most + cut;
      }
      sp.items[atomicAdd(count + talk_class(steps[m] - extras * per, per), 1)] = make_int4(sq[m], xt[m], extras * per, slot);
    }
  __syncthreads();
  if (tid == 0) {
    sp.plan[0] = per;
    sp.plan[1] = items;
    sp.plan[2] = taken[1];
    sp.plan[3] = 0;
  }
}

constexpr int kTS = kPromptKeys;   // keys per tile of the first kernel

// A wave has 32 units, a unit's scores of 32 keys two lanes, each with a maximum and a sum of its own.  Bound by products and then
// exponentials, 33 us of products at the rate of a large one: 16 heads, eight prompts of 1061 to 2048 tokens, 59 us, and 68 on 16x16x32 products
// with K by way of registers, where a sixth of the time went to bank conflicts and a maximum was taken off every score.
template <int DC, bool PLAN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void talk_stats_kernel(const TalkPrefillArgs p) {
  typedef PromptCore<DC, 1> Core;
  __shared__ __attribute__((aligned(1024))) unsigned char Ks[2 * Core::KB];
  int sq, plane, xt, block = prompt_block(blockIdx.x, blockIdx.y);
  if constexpr (PLAN) {                                              // eight workgroups in front: the XCDs keep their tiles
    if (block == 0) talk_plan(p, reinterpret_cast<int32_t *>(Ks));
    block -= 8;
    if (block < 0) return;
  }
  if (!prompt_tile(p.tiles, block, sq, plane, xt)) return;
  const SinkCache &c = p.c;
  const int seq = p.first_seq + sq, kvh = plane / p.passes, pass = plane % p.passes;
  const int q0 = p.cu_q[seq], lq = p.cu_q[seq + 1] - q0, start = p.starts[seq];
  const int row0 = xt * p.bq;
  if (row0 >= lq || start + lq > static_cast<int64_t>(p.table_cols) * c.bs) return;
  const int32_t *bt = c.bt + seq * c.bt_stride;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
  const int nh = min(p.hpp, p.group - pass * p.hpp);
  const int last_row = min(row0 + p.bq, lq) - 1, i_last = start + last_row;
  Core core;
  core.start(TLF_DL_LDSADDR(Ks), TLF_DL_LDSADDR(Ks), tid);           // no values
  const int wave_first = start + min(row0 + core.wave * 32 / p.hpp, last_row);
  const int wave_last = min(start + row0 + ((core.wave + 1) * 32 - 1) / p.hpp, i_last);
  const int u = core.wave * 32 + n, r = row0 + u / p.hpp, hh = u % p.hpp;
  const bool uok = u < p.bq * p.hpp && r <= last_row && hh < nh;
  const int row = min(r, last_row), upos = start + row;
  const int64_t uat = static_cast<int64_t>(q0 + row) * p.H + kvh * p.group + pass * p.hpp + (hh < nh ? hh : 0);
#pragma unroll
  for (int kc = 0; kc < 2 * DC; ++kc) {
    Pack16 t;
    t.u = *reinterpret_cast<const uint4 *>(p.q + uat * Core::DP + g * 8 + kc * 16);
    core.qf[kc] = t.v;
  }
  unsigned int koff[DC];                                             // this lane's pieces in a tile, which is one piece of a page
#pragma unroll
  for (int i = 0; i < DC; ++i) {
    int at, piece;
    core.k_piece(i, lane, at, piece);
    koff[i] = (at * Core::KCH + piece) * 16;
  }
  // A scalar load: by way of the vector memory it would be waited for together with the copies that were issued before it
  // (342 us a layer of the above and 63 with 87 tokens behind 768; so 334 and 59.5).
  auto page_of = [&](int t) __attribute__((always_inline)) { return load_uniform(bt + sink_page_of(c, min(t * kTS, i_last))); };
  int page_next = page_of(0);                                        // looked up a tile ahead
  auto copy = [&](int t) __attribute__((always_inline)) {            // rows past the last query are masked
    const int64_t at = sink_row(c, page_next, sink_page_of(c, t * kTS), kvh, t * kTS);
    page_next = page_of(t + 1);
    const unsigned char *kp = static_cast<const unsigned char *>(c.k) + at * (Core::DP * 2);
#pragma unroll
    for (int i = 0; i < DC; ++i) prompt_copy(koff[i], kp, core.k_place(t, i));
  };
  float m = -INFINITY, l = 0.f, over = -INFINITY;                    // over: what a score must not exceed; no key yet
  typename Core::Scores from = Core::all(0.f);                       // the score less what stands for the maximum
  const int tiles = i_last / kTS + 1;
  copy(0);
  for (int t = 0; t < tiles; ++t) {
    TLF_DL_BARRIER(0);
    if (t + 1 < tiles) copy(t + 1);
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const int k0 = t * kTS + hf * 32;
      if (k0 > wave_last) continue;                                  // wave uniform: some unit sees some key
      typename Core::Scores s;
      core.read_k(t, hf);
      core.scores(from, s);
      if (k0 + 31 > wave_first) {                                    // the diagonal cuts the half
        const int seen = upos - (k0 + g * 8);
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = (j & 8) * 2 + (j & 7) <= seen ? s[j] : -INFINITY;
      }
      const float x = Core::largest(s);
      if (__any(x > over)) {
        const bool up = x > over;
        const float top = up ? (m != -INFINITY ? m : 0.f) + x : m;
        l *= up ? __builtin_amdgcn_exp2f(m - top) : 1.f;
        s -= up ? x : 0.f;
        m = top;
        from = Core::all(top == -INFINITY ? 0.f : -top);
        over = top == -INFINITY ? top : 8.f;
      }
      float e[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) e[j] = __builtin_amdgcn_exp2f(s[j]);
      l += Core::sum(e);
    }
  }
  const float top = prompt_unit_max(m);                              // a row sees itself: finite
  const float sum = prompt_unit_sum(l * __builtin_amdgcn_exp2f(m - top));
  if (g == 0 && uok) p.stats[uat] = top + __builtin_amdgcn_logf(sum);
}

// Four values of a head's output.
__device__ __forceinline__ bool talk_out_in_fours(const TalkPrefillArgs &p) {
  return (p.c.Dv & 3) == 0 && (p.ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 7) == 0;
}
__device__ __forceinline__ void talk_put(unsigned short *o, int col, int dims, bool vec, const floatx4 &x) {
  const uint2 v = make_uint2(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]));
  if (vec) {
    if (col < dims) *reinterpret_cast<uint2 *>(o + col) = v;
  } else {
    const unsigned int y[2] = {v.x, v.y};
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (col + r < dims) o[col + r] = static_cast<unsigned short>(y[r / 2] >> (16 * (r & 1)));
  }
}

// A row's place in LDS for heads of WV waves: W [key][head], later M [head][key]; hi and lo apart; rows begin in different banks.
__host__ __device__ constexpr int talk_heads_held(int wv) { return wv == 1 ? 8 : wv * 4; }
__host__ __device__ constexpr int talk_row_size(int wv) {
  return (talk_heads_held(wv) * kTM > kTK * talk_heads_held(wv) ? talk_heads_held(wv) * kTM : kTK * talk_heads_held(wv)) + 8;
}

__device__ __forceinline__ shortx4 talk_read_tr16_at(unsigned int lds) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<shortx4 __attribute__((address_space(3))) *>(lds));
}

// LDS by byte address: one register and constants instead of a pointer per place
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
template <typename T>
__device__ __forceinline__ T talk_ld(unsigned int at) {
  return *reinterpret_cast<const T __attribute__((address_space(3))) *>(at);
}
template <typename T>
__device__ __forceinline__ void talk_st(unsigned int at, const T &v) {
  *reinterpret_cast<T __attribute__((address_space(3))) *>(at) = v;
}

// WV: quads of heads, RT: tiles of 16 rows; DC: key dimensions in units of 32, VC: of values, rounded up to 2 or 4; GS: heads of a
// quad that share a KV head (1, 2 or 4).  A wave has RW row tiles of HW heads of KV KV heads, HK each: item e = (KV head, row tile, head).
template <int WV, int RT, int DC, int VC, int GS>
__device__ __forceinline__ void talk_prefill_tile(const TalkPrefillArgs &p, const TalkItem item, const int wave, const int lane, unsigned short *lds) {
  constexpr int HP = talk_heads_held(WV), HT = (HP + 15) / 16, KH = (HP + 31) / 32, ROW = talk_row_size(WV), TQ = RT * 16, NW = WV * RT;
  constexpr int VP = VC * 32, PIECES = VP / 8, RW = RT < 4 / GS ? RT : 4 / GS, HW = 4 / RW, KV = HW > GS ? HW / GS : 1, HK = HW / KV;
  constexpr int PER = 4 / KV;                                        // items of a KV head
  constexpr int TS = KH * 32 + 8;                                    // heads of a talk row in LDS
  constexpr int kAtOnce = HT == 1 ? 4 : 1;                           // rows of the mix, as registers allow
  unsigned short *Vs = lds, *Wh = lds + p.c.G * kTK * VP, *Wl = Wh + TQ * ROW, *Ts = Wl + TQ * ROW;    // Vs [G][32][VP], Ts [16 HT][TS]
  const SinkCache &c = p.c;
  const int seq = p.first_seq + item.sq;
  const int q0 = load_uniform(p.cu_q + seq), lq = load_uniform(p.cu_q + seq + 1) - q0, start = load_uniform(p.starts + seq);
  const int row0 = item.xt * TQ;
  if (row0 >= lq || start + lq > static_cast<int64_t>(p.table_cols) * c.bs) return;
  const int32_t *bt = c.bt + seq * c.bt_stride;
  const int G = c.G;
  const int tid = wave * 64 + lane, n = lane & 15, g = lane >> 4;
  const int h0 = wave % (WV * 4 / HW) * HW, rt = wave / (WV * 4 / HW) * RW * 16;
  const int last_row = min(row0 + TQ, lq) - 1, i_last = start + last_row;
  const int wave_first = start + min(row0 + rt, last_row);           // keys behind it are masked for some row of the wave
  auto head_of = [](int e) { return e / PER * HK + e % HK; };        // of the wave's heads; and the row tile
  auto tile_of = [](int e) { return e % PER / HK; };
  const int first = item.first, tiles = item.slot >= 0 && item.slot < p.split.most ? first + load_uniform(p.split.plan) : i_last / kTK + 1;
  // where a tile lies: its page (an unmapped one reads page 0) and its first row there, stepped tile by tile
  struct Place {
    int index, page, row;
  };
  auto page_at = [&](int index) __attribute__((always_inline)) {
    const int page = load_uniform(bt + index);
    return page >= 0 && page < c.pages ? page : 0;
  };
  auto after = [&](const Place &at, bool more) __attribute__((always_inline)) {       // the next tile's, if there is one
    const bool turn = at.row + kTK == c.bs;
    Place b{at.index + (turn && more ? 1 : 0), at.page, turn ? 0 : at.row + kTK};
    if (turn && more) b.page = page_at(b.index);
    return more ? b : at;
  };
  auto row_of = [&](const Place &at, int kv) __attribute__((always_inline)) { return (static_cast<int64_t>(at.page) * G + kv) * c.bs + at.row; };

  // heads that no wave has, and keys that a first tile does not, are read by the mix (times zero)
  for (int i = tid; i < 2 * TQ * ROW / 8; i += NW * 64) reinterpret_cast<uint4 *>(Wh)[i] = make_uint4(0, 0, 0, 0);
  for (int i = tid; i < HT * 16 * TS; i += NW * 64) {
    const int h = i / TS, k = i % TS;
    Ts[i] = h < p.H && k < p.H ? p.talk[h * p.H + k] : 0;
  }
  bf16x8 qf[4][DC];
  int kvh[KV];
  float m[4];
#pragma unroll
  for (int i = 0; i < KV; ++i) kvh[i] = min(h0 + i * HK, p.H - 1) / p.group;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int h = min(h0 + head_of(e), p.H - 1), row = q0 + min(row0 + rt + tile_of(e) * 16 + n, last_row);
    m[e] = p.stats[static_cast<int64_t>(row) * p.H + h];
    const unsigned short *qp = p.q + (static_cast<int64_t>(row) * p.H + h) * c.Dp + g * 8;
#pragma unroll
    for (int kc = 0; kc < DC; ++kc) {
      Pack16 t;
      t.u = *reinterpret_cast<const uint4 *>(qp + kc * 32);
      qf[e][kc] = t.v;
    }
  }
  const int krow = (n >> 2) * 8 + (n & 3);
  const unsigned int koff = (krow * DC * 32 + g * 8) * 2;
  auto load_k = [&](bf16x8 (&kf)[DC], const Place &at, int kv, int s) __attribute__((always_inline)) {    // half s of a tile's rows
    const char *kp = static_cast<const char *>(c.k) + row_of(at, kv) * (DC * 64);    // uniform
#pragma unroll
    for (int kc = 0; kc < DC; ++kc) {
      Pack16 t;
      t.u = *reinterpret_cast<const uint4 *>(kp + koff + (s * 4 * DC * 64 + kc * 64));
      kf[kc] = t.v;
    }
  };
  floatx4 acc[4][2 * VC];
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int d = 0; d < 2 * VC; ++d) acc[e][d] = floatx4{0.f, 0.f, 0.f, 0.f};
  const unsigned int vlds = TLF_DL_LDSADDR(Vs);
  // V's 16-byte pieces in LDS: pairs of them are permuted within a row, so that a transpose read (rows 8 g + 0 .. 3, or four on)
  // meets every bank twice.  Byte address of this lane's part of the first pair; pair d is d * 32 away by exclusive or.
  auto pair_of = [](int row) __attribute__((always_inline)) { return VC >= 4 ? (row & 3) | (row >> 1 & 4) : (row >> 1 & 1) | (row >> 2 & 2); };
  const int vrow = g * 8 + (n >> 2);
  unsigned int vat = vlds + (vrow * VP + pair_of(vrow) * 16 + (n & 3) * 4) * 2;
  constexpr unsigned int LO = TQ * ROW * 2;                          // from a pair's high half to its low one
  const unsigned int w0 = TLF_DL_LDSADDR(Wh);
  unsigned int tat = TLF_DL_LDSADDR(Ts) + (n * TS + g * 8) * 2;
  unsigned int wat = w0 + ((rt + n) * ROW + g * 8 * HP + h0) * 2;    // where this lane puts weights
  unsigned int mat = w0 + ((rt + n) * ROW + h0 * kTM + g * 8) * 2;   // where it finds mixed ones
  unsigned int rat = w0 + (wave * ROW + krow * HP + g % (HP < 32 ? HP / 8 : 4) * 8) * 2;     // a row's weights as the mix's operand; heads that
                                                                     // there is no room for read others, times zeros
  unsigned int pat = w0 + (wave * ROW + n * kTM + g * 8) * 2;        // and its result

  bf16x8 kb[DC];
  Place at{sink_page_of(c, first * kTK), 0, 0};
  at.page = page_at(at.index);
  at.row = first * kTK - at.index * c.bs;
  load_k(kb, at, kvh[0], 0);
  lds_barrier();
  for (int t = first; t < tiles; ++t) {
    const int j0 = t * kTK;
    const Place next = after(at, t + 1 < tiles);
    auto copy_v = [&]() __attribute__((always_inline)) {
      const int pieces = c.Vp / 8;
      for (int i = wave; i < G * (VP / 16); i += NW) {
        const int kv = i / (VP / 16), slot = i % (VP / 16) * 64 + lane, row = slot / PIECES, piece = (slot % PIECES) ^ (pair_of(row) * 2);
        const unsigned char *base = reinterpret_cast<const unsigned char *>(static_cast<const unsigned short *>(c.v) + row_of(at, kv) * c.Vp);
        TLF_DL_COPY(static_cast<unsigned int>((row * pieces + (piece < pieces ? piece : 0)) * 16), base, vlds + i * 1024);
      }
    };
#pragma unroll
    for (int u = 0; u < 2 * KV; ++u) {                               // (KV head, half a tile)
      const int e0 = u / 2 * PER, s = u % 2;
      floatx4 w[PER];
#pragma unroll
      for (int e = 0; e < PER; ++e) w[e] = floatx4{0.f, 0.f, 0.f, 0.f};
      // lane (n, g): keys j0 + g * 8 + s * 4 + 0 .. 3 of row n
#pragma unroll
      for (int kc = 0; kc < DC; ++kc)
#pragma unroll
        for (int e = 0; e < PER; ++e) w[e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb[kc], qf[e0 + e][kc], w[e], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (u == 2 * KV - 1) copy_v();                                 // this tile's K is there: V's copies follow it
      if (u + 1 < 2 * KV) load_k(kb, at, kvh[(u + 1) / 2], (u + 1) % 2);
      else if (t + 1 < tiles) load_k(kb, next, kvh[0], 0);
      if (j0 + kTK - 1 > wave_first)                                 // the diagonal cuts the tile
#pragma unroll
        for (int e = 0; e < PER; ++e) {
          const int pos = start + min(row0 + rt + tile_of(e0 + e) * 16 + n, last_row) - j0 - g * 8 - s * 4;
#pragma unroll
          for (int r = 0; r < 4; ++r) w[e][r] = r <= pos ? w[e][r] : -INFINITY;
        }
#pragma unroll
      for (int x = 0; x < PER / HK; ++x)                             // row tiles
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const unsigned int to = wat + (x * 16 * ROW + (s * 4 + r) * HP + u / 2 * HK) * 2;
          const int e1 = x * HK;
          if constexpr (HK == 1) {
            const float a = __builtin_amdgcn_exp2f(w[e1][r] - m[e0 + e1]);
            const unsigned short hi = float_to_bf16_bits(a);
            talk_st<unsigned short>(to, hi);
            talk_st<unsigned short>(to + LO, float_to_bf16_bits(a - bf16_bits_to_float(hi)));
          } else {
            unsigned int hi[HK / 2], lo[HK / 2];
#pragma unroll
            for (int e = 0; e < HK; e += 2) {
              const float a = __builtin_amdgcn_exp2f(w[e1 + e][r] - m[e0 + e1 + e]), b = __builtin_amdgcn_exp2f(w[e1 + e + 1][r] - m[e0 + e1 + e + 1]);
              weight_pairs(a, b, hi[e / 2], lo[e / 2]);
              __builtin_amdgcn_sched_barrier(0);                     // one pair at a time, for the registers' sake
            }
            if constexpr (HK == 4) {
              talk_st<u32x2>(to, u32x2{hi[0], hi[1]});
              talk_st<u32x2>(to + LO, u32x2{lo[0], lo[1]});
            } else {
              talk_st<unsigned int>(to, hi[0]);
              talk_st<unsigned int>(to + LO, lo[0]);
            }
          }
        }
    }
    lds_barrier();
    // talk^T as the mix's B operand: lane (n, g) of tile t holds talk[16 t + n][32 k + 8 g ..]
    bf16x8 tf[HT][KH];
    asm volatile("" : "+v"(tat), "+v"(rat), "+v"(pat));              // read here, not kept in registers
#pragma unroll
    for (int ht = 0; ht < HT; ++ht)
#pragma unroll
      for (int k = 0; k < KH; ++k) tf[ht][k] = talk_ld<bf16x8>(tat + (ht * 16 * TS + k * 32) * 2);
#pragma unroll kAtOnce
    for (int i = 0; i < TQ / NW; ++i) {                              // a row's W is read and its M written by the same wave
      const unsigned int row_at = i * (NW * ROW * 2);
      floatx4 mx[HT][2];
#pragma unroll
      for (int ht = 0; ht < HT; ++ht) mx[ht][0] = mx[ht][1] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KH; ++k) {
        bf16x8 hi[2], lo[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          hi[s] = lo[s] = __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
          if (HP < 32 || k * 32 + g * 8 < HP) {                      // heads there are room for
            hi[s] = talk_ld<bf16x8>(rat + row_at + (s * 4 * HP + k * 32) * 2);
            lo[s] = talk_ld<bf16x8>(rat + row_at + (s * 4 * HP + k * 32) * 2 + LO);
          }
        }
#pragma unroll
        for (int ht = 0; ht < HT; ++ht)
#pragma unroll
          for (int s = 0; s < 2; ++s) mx[ht][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi[s], tf[ht][k], mx[ht][s], 0, 0, 0);
#pragma unroll
        for (int ht = 0; ht < HT; ++ht)
#pragma unroll
          for (int s = 0; s < 2; ++s) mx[ht][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo[s], tf[ht][k], mx[ht][s], 0, 0, 0);
      }
      wave_lds_fence();
#pragma unroll
      for (int ht = 0; ht < HT; ++ht) {                              // lane (n, g): head 16 ht + n, keys 8 g ..
        const float x[8] = {mx[ht][0][0], mx[ht][0][1], mx[ht][0][2], mx[ht][0][3], mx[ht][1][0], mx[ht][1][1], mx[ht][1][2], mx[ht][1][3]};
        bf16x8 hi, lo;
        talk_pair(x, hi, lo);
        if (HP >= 16 || n < HP) {
          talk_st<bf16x8>(pat + row_at + ht * 16 * kTM * 2, hi);
          talk_st<bf16x8>(pat + row_at + ht * 16 * kTM * 2 + LO, lo);
        }
      }
    }
    // this wave's copies are there when at most the loads of the next K, issued after them, are on their way
    if (t + 1 < tiles) TLF_DL_BARRIER(DC);
    else TLF_DL_BARRIER(0);
    asm volatile("" : "+v"(vat), "+v"(mat), "+v"(wat));                                    // addresses are made here, not kept in registers
#pragma unroll
    for (int e0 = 0; e0 < 4; e0 += 2) {
      bf16x8 mh[2], ml[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const unsigned int from = mat + (tile_of(e0 + e) * 16 * ROW + head_of(e0 + e) * kTM) * 2;
        mh[e] = talk_ld<bf16x8>(from);
        ml[e] = talk_ld<bf16x8>(from + LO);
      }
#pragma unroll
      for (int d = 0; d < 2 * VC; ++d) {
        // V's reads stay beside their products: gathered ahead they push parts of q out of the registers, and each half of a tile then waits
        // for q to come back from memory behind the loads of K
        __builtin_amdgcn_sched_barrier(0);
        bf16x8 vb[2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
          if (e == 0 || PER == 1) {
            const unsigned int at = (vat + kvh[(e0 + e) / PER] * (kTK * VP * 2)) ^ (d * 32);
            const uint2 v0 = __builtin_bit_cast(uint2, talk_read_tr16_at(at)), v1 = __builtin_bit_cast(uint2, talk_read_tr16_at(at + 8 * VP));
            vb[e] = __builtin_bit_cast(bf16x8, make_uint4(v0.x, v0.y, v1.x, v1.y));
          } else {
            vb[e] = vb[0];
          }
#pragma unroll
        for (int e = 0; e < 2; ++e) acc[e0 + e][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb[e], mh[e], acc[e0 + e][d], 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 2; ++e) acc[e0 + e][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb[e], ml[e], acc[e0 + e][d], 0, 0, 0);
      }
    }
    lds_barrier();                                                   // V and M have been read by all
    at = next;
  }

  if (item.slot >= 0) {                                              // as it lies in the registers: whole lines
    floatx4 *const part = p.split.parts + static_cast<int64_t>(item.slot) * p.split.size + (wave * (8 * VC)) * 64 + lane;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int d = 0; d < 2 * VC; ++d) part[(e * 2 * VC + d) * 64] = acc[e][d];
    return;
  }
  const bool vec = talk_out_in_fours(p);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = row0 + rt + tile_of(e) * 16 + n, h = h0 + head_of(e);
    if (row > last_row || h >= p.H) continue;
    unsigned short *o = p.out + static_cast<int64_t>(q0 + row) * p.ldo + static_cast<int64_t>(h) * c.Dv;
#pragma unroll
    for (int d = 0; d < 2 * VC; ++d) {
      talk_put(o, d * 16 + g * 4, c.Dv, vec, acc[e][d]);
    }
  }
}

// Whole tiles: a workgroup has the tile of its place.  Its own kernel: the loop below costs registers, and with 32 heads 14 % of the time (eight
// prompts of 1061 to 2048 tokens 643 us, 734 in that loop; nine of 2048 with 16 heads 599, 621).
template <int WV, int RT, int DC, int VC, int GS>
__global__ __launch_bounds__(WV * RT * 64) void talk_prefill_kernel(const TalkPrefillArgs p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned short lds[];
  int sq, plane, xt;
  if (!prompt_tile(p.tiles, prompt_block(blockIdx.x, blockIdx.y), sq, plane, xt)) return;
  talk_prefill_tile<WV, RT, DC, VC, GS>(p, TalkItem{sq, xt, 0, -1}, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), threadIdx.x & 63, lds);
}

// With a plan, a workgroup per compute unit takes items until there are none: the hardware deals workgroups to XCDs and shader engines by their
// number, whatever runs there.
template <int WV, int RT, int DC, int VC, int GS>
__global__ __launch_bounds__(WV * RT * 64) void talk_cut_kernel(const TalkPrefillArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned short lds[];
  int *const at = reinterpret_cast<int *>(lds);                      // the item, where the tile's arrays begin
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (bool more = false;; more = true) {
    // the arguments are read anew for each item: kept across the loop, what follows from them would not fit into the scalar registers
    auto args = (const TalkPrefillArgs __attribute__((address_space(4))) *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    const TalkPrefillArgs &p = *(const TalkPrefillArgs *)args;
    if (wave == 0 && __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0)) == 0) {
      int4 item = make_int4(0, 0, 0, -1);
      const int i = more ? gridDim.x + atomicAdd(p.split.plan + 3, 1) : blockIdx.x;
      at[4] = i < p.split.plan[1];
      if (i < p.split.plan[1]) item = p.split.items[i];
      *reinterpret_cast<int4 *>(at) = item;
    }
    lds_barrier();
    auto same = [&](int i) { return __builtin_amdgcn_readfirstlane(at[i]); };
    if (!same(4)) return;
    const TalkItem item{same(0), same(1), same(2), same(3)};
    lds_barrier();
    int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));
    asm volatile("" : "+v"(lane));                                   // what follows from it is made anew for each item, not kept in registers
    talk_prefill_tile<WV, RT, DC, VC, GS>(p, item, wave, lane, lds);
  }
}

// Row tiles that were cut: their parts, added up in the order of the keys.  blockIdx.x: the tile, blockIdx.y: a wave of the second kernel.
template <int WV, int RT, int VC, int GS>
__global__ __launch_bounds__(256) void talk_join_kernel(const TalkPrefillArgs p) {
  constexpr int RW = RT < 4 / GS ? RT : 4 / GS, HW = 4 / RW, KV = HW > GS ? HW / GS : 1, HK = HW / KV, PER = 4 / KV;
  const TalkSplit &sp = p.split;
  if (static_cast<int>(blockIdx.x) >= sp.plan[2]) return;
  const int4 cut = sp.cuts[blockIdx.x];
  const int seq = p.first_seq + cut.x, row0 = cut.y * (RT * 16), wave = blockIdx.y, lane = threadIdx.x & 63, e = threadIdx.x >> 6;
  const int q0 = p.cu_q[seq], lq = p.cu_q[seq + 1] - q0, n = lane & 15, g = lane >> 4;
  const int row = row0 + wave / (WV * 4 / HW) * RW * 16 + e % PER / HK * 16 + n, h = wave % (WV * 4 / HW) * HW + e / PER * HK + e % HK;
  const int64_t at = (wave * 4 + e) * 2 * VC * 64 + lane, size = sp.size;
  const floatx4 *const extra = sp.parts + cut.z * size + at, *const rest = sp.parts + (sp.most + blockIdx.x) * size + at;
  floatx4 sum[2 * VC];
#pragma unroll
  for (int d = 0; d < 2 * VC; ++d) sum[d] = extra[d * 64];
  for (int part = 1; part < cut.w; ++part)
#pragma unroll
    for (int d = 0; d < 2 * VC; ++d) sum[d] += extra[part * size + d * 64];
#pragma unroll
  for (int d = 0; d < 2 * VC; ++d) sum[d] += rest[d * 64];
  if (row >= lq || h >= p.H) return;
  const bool vec = talk_out_in_fours(p);
  unsigned short *const o = p.out + static_cast<int64_t>(q0 + row) * p.ldo + static_cast<int64_t>(h) * p.c.Dv;
#pragma unroll
  for (int d = 0; d < 2 * VC; ++d) talk_put(o, d * 16 + g * 4, p.c.Dv, vec, sum[d]);
}

// Quads of heads as instantiated, 0: too many.
inline int talk_quads(int heads) { return heads <= 4 ? 1 : heads <= 8 ? 2 : heads <= 16 ? 4 : heads <= 32 ? 8 : 0; }
constexpr int kTalkLds = 160 * 1024;
inline int talk_units(int padded) { return padded <= 64 ? 2 : 4; }     // of 32, as instantiated
int talk_prefill_lds(int quads, int rt, int G, int Vp) {
  return 2 * (2 * rt * 16 * talk_row_size(quads) + G * kTK * talk_units(Vp) * 32 + (quads > 4 ? 32 : 16) * 40);
}
// Row tiles per workgroup: up to eight waves, with 16 heads fewer where LDS does not hold them; 0: no room.
int talk_row_tiles(int quads, int G, int Vp) {
  const int most = 8 / quads < 4 ? 8 / quads : 4;
  return talk_prefill_lds(quads, most, G, Vp) <= kTalkLds ? most : quads == 4 && talk_prefill_lds(quads, 1, G, Vp) <= kTalkLds ? 1 : 0;
}

// What a workspace holds; bytes = 0: row tiles stay whole.
struct TalkRoom {
  int most, size;
  int64_t cuts, parts, bytes;            // where they begin
};
TalkRoom talk_room(int64_t seqs, int64_t max_tokens, int64_t max_keys, int quads, int tq, int Vp) {
  TalkRoom r{0, quads * 4 * tq * talk_units(Vp) * 8, 0, 0, 0};
  if (!talk_cuts(seqs, max_tokens, max_keys, tq)) return r;
  const int64_t tiles = (max_tokens + tq - 1) / tq * seqs;
  r.most = static_cast<int>(std::min<int64_t>(kTalkExtras, tiles * std::min<int64_t>(kTalkExtras, (max_keys + kTK - 1) / kTK / kTalkLeast)));
  r.cuts = 16 + (kTalkTiles + kTalkExtras) * 16;
  r.parts = (r.cuts + kTalkTiles * 16 + 255) / 256 * 256;
  r.bytes = r.parts + (r.most + tiles) * r.size * 16;
  return r;
}

template <int DC>
int launch_talk_stats(TalkPrefillArgs &a, int num_seqs, int max_tokens, hipStream_t s) {
  constexpr int kUnits = 32 * kPromptWaves;
  a.hpp = a.group < kUnits ? a.group : kUnits;
  a.passes = (a.group + a.hpp - 1) / a.hpp;
  a.bq = kUnits / a.hpp;
  const int blocks = prompt_tiles_make(a.tiles, (max_tokens + a.bq - 1) / a.bq, a.c.G * a.passes, num_seqs);
  if (!blocks) return TLF_E_SHAPE;
  if (a.split.plan) TLF_LAUNCH((talk_stats_kernel<DC, true>), prompt_grid<dim3>(blocks + 8), dim3(256), 0, s, a);
  else TLF_LAUNCH((talk_stats_kernel<DC, false>), prompt_grid<dim3>(blocks), dim3(256), 0, s, a);
  return launch_status();
}

template <int WV, int RT, int DC, int VC, int GS>
int launch_talk_prefill(TalkPrefillArgs &a, int num_seqs, int max_tokens, hipStream_t s) {
  static const hipError_t allowed = [] {
    hipError_t e = hipSuccess;
    for (const void *k : {reinterpret_cast<const void *>(&talk_prefill_kernel<WV, RT, DC, VC, GS>), reinterpret_cast<const void *>(&talk_cut_kernel<WV, RT, DC, VC, GS>)})
      if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kTalkLds);
    return e;
  }();
  if (allowed != hipSuccess) return static_cast<int>(allowed);
  const int blocks = prompt_tiles_make(a.tiles, (max_tokens + RT * 16 - 1) / (RT * 16), 1, num_seqs);
  if (!blocks) return TLF_E_SHAPE;
  const size_t lds = talk_prefill_lds(WV, RT, a.c.G, a.c.Vp);
  if (!a.split.plan) {
    TLF_LAUNCH((talk_prefill_kernel<WV, RT, DC, VC, GS>), prompt_grid<dim3>(blocks), dim3(WV * RT * 64), lds, s, a);
    return launch_status();
  }
  TLF_LAUNCH((talk_cut_kernel<WV, RT, DC, VC, GS>), dim3(kTalkUnits), dim3(WV * RT * 64), lds, s, a);
  TLF_LAUNCH((talk_join_kernel<WV, RT, VC, GS>), dim3((max_tokens + RT * 16 - 1) / (RT * 16) * num_seqs, WV * RT), dim3(256), 0, s, a);
  return launch_status();
}
template <int WV, int RT>
int launch_talk_prefill_dims(TalkPrefillArgs &a, int num_seqs, int max_tokens, hipStream_t s) {
#define TLF_TP(DC, VC)                                                                                                    \
  do {                                                                                                                    \
    if (a.group % 4 == 0) return launch_talk_prefill<WV, RT, DC, VC, 4>(a, num_seqs, max_tokens, s);                      \
    if (a.group % 2 == 0) return launch_talk_prefill<WV, RT, DC, VC, 2>(a, num_seqs, max_tokens, s);                      \
    return launch_talk_prefill<WV, RT, DC, VC, 1>(a, num_seqs, max_tokens, s);                                            \
  } while (0)
#define TLF_TP_V(DC)                            \
  case DC:                                      \
    if (talk_units(a.c.Vp) == 2) TLF_TP(DC, 2); \
    TLF_TP(DC, 4);
  switch (a.c.Dp / 32) {
    TLF_TP_V(1) TLF_TP_V(2) TLF_TP_V(3) TLF_TP_V(4)
    default: return TLF_E_UNSUPPORTED;
  }
#undef TLF_TP_V
#undef TLF_TP
}

}  // namespace tlf

extern "C" int tlf_talk_attn_prefill_supported(int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim) {
  return heads > 0 && kv_heads > 0 && dim > 0 && vdim > 0 && heads <= 32 && dim <= 128 && vdim <= 128 &&
         tlf::talk_row_tiles(tlf::talk_quads(heads), kv_heads, (vdim + 31) / 32 * 32) > 0;
}

namespace tlf {
int talk_attn_prefill(const void *q, const void *k_cache, const void *v_cache, const int32_t *block_tables, int64_t bt_stride,
                      const int32_t *cu_seqlens_q, const int32_t *seq_starts, int32_t first_seq, int32_t num_seqs, int32_t max_tokens,
                      const void *talk, float *stats, void *out, int64_t out_stride, int32_t heads, int32_t kv_heads, int32_t dim,
                      int32_t vdim, int32_t block_size, int64_t num_pages, bool cut, void *workspace, size_t workspace_bytes,
                      void *stream) {
  if (num_seqs < 0 || max_tokens < 0 || first_seq < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads) return TLF_E_SHAPE;
  if (out_stride < static_cast<int64_t>(heads) * vdim || bt_stride <= 0) return TLF_E_SHAPE;
  if (num_seqs == 0 || max_tokens == 0) return TLF_OK;
  TalkPrefillArgs a{};
  if (int rc = sink_cache_make(a.c, k_cache, v_cache, block_tables, bt_stride, block_size, kv_heads, dim, vdim, num_pages)) return rc;
  if (!tlf_talk_attn_prefill_supported(heads, kv_heads, dim, vdim)) return TLF_E_UNSUPPORTED;
  if (!q || !block_tables || !cu_seqlens_q || !seq_starts || !talk || !stats || !out) return TLF_E_NULL;
  if (!aligned16(q)) return TLF_E_ALIGN;
  a.stats = stats; a.q = static_cast<const unsigned short *>(q); a.talk = static_cast<const unsigned short *>(talk); a.cu_q = cu_seqlens_q;
  a.starts = seq_starts; a.out = static_cast<unsigned short *>(out); a.ldo = out_stride; a.H = heads; a.group = heads / kv_heads;
  a.first_seq = first_seq; a.table_cols = static_cast<int32_t>(bt_stride);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int quads = talk_quads(heads), row_tiles = talk_row_tiles(quads, kv_heads, a.c.Vp);
  if (cut) {
    const TalkRoom room = talk_room(num_seqs, max_tokens, bt_stride * block_size, quads, row_tiles * 16, a.c.Vp);
    if (room.bytes) {
      if (!workspace || workspace_bytes < static_cast<size_t>(room.bytes)) return TLF_E_WORKSPACE;
      if (!aligned16(workspace)) return TLF_E_ALIGN;
      char *const ws = static_cast<char *>(workspace);
      a.split = TalkSplit{reinterpret_cast<int32_t *>(ws), reinterpret_cast<int4 *>(ws + 16), reinterpret_cast<int4 *>(ws + room.cuts),
                          reinterpret_cast<floatx4 *>(ws + room.parts), num_seqs, (max_tokens + row_tiles * 16 - 1) / (row_tiles * 16),
                          row_tiles * 16, room.most, room.size};
    }
  }
  int rc;
  switch (a.c.Dp / 32) {
    case 1: rc = launch_talk_stats<1>(a, num_seqs, max_tokens, s); break;
    case 2: rc = launch_talk_stats<2>(a, num_seqs, max_tokens, s); break;
    case 3: rc = launch_talk_stats<3>(a, num_seqs, max_tokens, s); break;
    default: rc = launch_talk_stats<4>(a, num_seqs, max_tokens, s); break;
  }
  if (rc != TLF_OK) return rc;
#define TLF_TP(WV, RT) \
  case (WV) * 8 + (RT): return launch_talk_prefill_dims<WV, RT>(a, num_seqs, max_tokens, s);
  switch (quads * 8 + row_tiles) {
    TLF_TP(1, 4) TLF_TP(2, 4) TLF_TP(4, 1) TLF_TP(4, 2) TLF_TP(8, 1)
    default: return TLF_E_UNSUPPORTED;
  }
#undef TLF_TP
}
}  // namespace tlf

extern "C" int tlf_talk_attn_prefill(const void *q, const void *k_cache, const void *v_cache, const int32_t *block_tables,
                                     int64_t bt_stride, const int32_t *cu_seqlens_q, const int32_t *seq_starts, int32_t first_seq,
                                     int32_t num_seqs, int32_t max_tokens, const void *talk, float *stats, void *out, int64_t out_stride,
                                     int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim, int32_t block_size,
                                     int64_t num_pages, void *stream) {
  return tlf::talk_attn_prefill(q, k_cache, v_cache, block_tables, bt_stride, cu_seqlens_q, seq_starts, first_seq, num_seqs, max_tokens, talk, stats,
                                out, out_stride, heads, kv_heads, dim, vdim, block_size, num_pages, false, nullptr, 0, stream);
}

extern "C" size_t tlf_talk_attn_prefill_workspace_bytes(int32_t num_seqs, int32_t max_tokens, int64_t max_keys, int32_t heads,
                                                        int32_t kv_heads, int32_t dim, int32_t vdim) {
  using namespace tlf;
  if (num_seqs <= 0 || max_tokens <= 0 || max_keys <= 0 || !tlf_talk_attn_prefill_supported(heads, kv_heads, dim, vdim)) return 0;
  const int Vp = (vdim + 31) / 32 * 32;
  return static_cast<size_t>(talk_room(num_seqs, max_tokens, max_keys, talk_quads(heads), talk_row_tiles(talk_quads(heads), kv_heads, Vp) * 16, Vp).bytes);
}

extern "C" int tlf_talk_attn_prefill_tile_rows(int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim) {
  using namespace tlf;
  return tlf_talk_attn_prefill_supported(heads, kv_heads, dim, vdim) ? talk_row_tiles(talk_quads(heads), kv_heads, (vdim + 31) / 32 * 32) * 16 : 0;
}

extern "C" int tlf_talk_attn_prefill_cuts(int32_t num_seqs, int32_t max_tokens, int32_t rows, int64_t reads, int64_t max_keys, int32_t heads,
                                          int32_t kv_heads, int32_t dim, int32_t vdim) {
  const int tq = tlf_talk_attn_prefill_tile_rows(heads, kv_heads, dim, vdim);
  return num_seqs > 0 && max_tokens > 0 && tq && tlf::talk_cuts_pay({num_seqs, max_tokens, rows, reads, max_keys}, tq);
}

extern "C" int tlf_talk_attn_prefill_route(int32_t singles, const int64_t *short_portions, const int64_t *long_portions, int32_t heads, int32_t kv_heads,
                                           int32_t dim, int32_t vdim) {
  using namespace tlf;
  const int tq = tlf_talk_attn_prefill_tile_rows(heads, kv_heads, dim, vdim);
  auto load = [](const int64_t *p) { return TalkLoad{p[0], p[1], p[2], p[3], p[4]}; };
  return tq && short_portions && long_portions ? talk_route(singles > 0, load(short_portions), load(long_portions), heads, tq) : kTalkByRows;
}

extern "C" int tlf_talk_attn_prefill_cut(const void *q, const void *k_cache, const void *v_cache, const int32_t *block_tables,
                                         int64_t bt_stride, const int32_t *cu_seqlens_q, const int32_t *seq_starts, int32_t first_seq,
                                         int32_t num_seqs, int32_t max_tokens, const void *talk, float *stats, void *out, int64_t out_stride,
                                         int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim, int32_t block_size, int64_t num_pages,
                                         void *workspace, size_t workspace_bytes, void *stream) {
  return tlf::talk_attn_prefill(q, k_cache, v_cache, block_tables, bt_stride, cu_seqlens_q, seq_starts, first_seq, num_seqs, max_tokens, talk, stats,
                                out, out_stride, heads, kv_heads, dim, vdim, block_size, num_pages, true, workspace, workspace_bytes, stream);
}
