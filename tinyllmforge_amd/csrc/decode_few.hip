// Decode attention for few sequences, with what comes before it where the projection is at hand: q / k norm, rotation and the
// K/V store of the new token (qknorm_rope.h).
//
// With a handful of sequences the time is launches and one memory latency after the other, not bytes, so this kernel spreads a sequence wider
// than decode_attn.hip does and takes the preparation along:
//   one workgroup per (share of a sequence, KV head, sequence), 16 teams of 16 lanes; a team takes every 16th token of the share, 8 dimensions a
//   lane, and asks for four tokens' rows of K and V at once, which is a whole share up to 64 tokens.  While they are on their way every
//   workgroup norms and rotates the queries of its KV head and the new token's K and V, and takes these where a token's row is the one they go to;
//   the share with the newest token stores them, and so does one with a page that another row's new token goes to (rows of one sequence).  Scores and sums in
//   fp32 on the vector ALU; partial results (maximum, sum, mix) per share, merged by a second kernel.
//
// Qwen3-8B shape (32 heads on 8), one sequence of 700 tokens, us: preparation 4.6, attention 9.5 on 12 workgroups, merge 3.9 before; layer 67.0 -> 60.7.
#include "qknorm_rope.h"

namespace tlf {

constexpr int kFewDim = 128, kFewAhead = 4, kFewShare = 64, kFewMaxSplits = 64;
constexpr float kFewLog2e = 1.4426950408889634f;

struct FewArgs {
  QkRopeStoreArgs prep;             // where the projection is given
  const unsigned short *x;          // its rows [q heads | k heads | v heads], or rows of prepared queries
  int64_t ldx;
  const unsigned char *k_cache, *v_cache;   // [blocks, block_size, Hkv, 128]
  const float *k_scale, *v_scale;   // [Hkv], e4m3 caches
  const int32_t *bt;
  int64_t bt_stride;
  const int32_t *ctx;
  unsigned short *out;              // [batch, Hq * 128]
  float *part, *ml;                 // [batch, Hq, splits, 128]; maximum (log2 units) and sum
  int64_t blocks;
  int32_t Hq, Hkv, bs, max_blocks, splits;
  float scale_log2;
};

// Tokens of a share: all shares of a sequence but the last have as many.
__device__ __forceinline__ int few_share(int ctx, int splits) { return max(kFewShare, ((ctx + splits - 1) / splits + 15) / 16 * 16); }

template <bool FP8>
struct FewRow;                      // eight values of a cache row
template <>
struct FewRow<false> {
  uint4 v;
  __device__ __forceinline__ void load(const unsigned char *row, int at) { v = load_nt_u4(row + at * 2); }
  __device__ __forceinline__ void zero() { v = make_uint4(0, 0, 0, 0); }
  __device__ __forceinline__ void put(const uint4 b, float) { v = b; }
  __device__ __forceinline__ void get(float (&f)[8]) const { unpack8(v, f); }
};
template <>
struct FewRow<true> {
  uint2 v;
  __device__ __forceinline__ void load(const unsigned char *row, int at) { v = *reinterpret_cast<const uint2 *>(row + at); }
  __device__ __forceinline__ void zero() { v = make_uint2(0, 0); }
  __device__ __forceinline__ void put(const uint4 b, float scale) {
    const int2 w = qk_piece_e4m3(b, scale);
    v = make_uint2(w.x, w.y);
  }
  __device__ __forceinline__ void get(float (&f)[8]) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const auto a = __builtin_amdgcn_cvt_pk_f32_fp8(i ? v.y : v.x, false), b = __builtin_amdgcn_cvt_pk_f32_fp8(i ? v.y : v.x, true);
      f[4 * i] = a[0]; f[4 * i + 1] = a[1]; f[4 * i + 2] = b[0]; f[4 * i + 3] = b[1];
    }
  }
};

// GROUP query heads per KV head.  RAW: x is the projection; otherwise the prepared queries, and the cache holds every token.
template <int GROUP, bool FP8, bool RAW>
__global__ __launch_bounds__(256) void decode_few_kernel(const FewArgs p) {
  constexpr int kBytes = FP8 ? 1 : 2;
  __shared__ __attribute__((aligned(16))) uint4 rows[GROUP + 2][16];        // queries, new K and V, bf16
  __shared__ __attribute__((aligned(16))) float mixes[4][GROUP][kFewDim];
  __shared__ float stats[4][GROUP][2];
  __shared__ int others[4];         // by wave: whether a page of the share gets another sequence's new row
  const int b = blockIdx.z, kvh = blockIdx.y, split = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, team = tid >> 4, j = tid & 15;
  const int ctx = min(p.ctx[b], p.max_blocks * p.bs), share = few_share(ctx, p.splits), t0 = split * share, t1 = min(ctx, t0 + share);
  const bool newest = RAW && (ctx > 0 ? t0 < ctx && ctx <= t0 + share : split == 0);
  if (t0 >= ctx && !newest) return;
  const int32_t *bt = p.bt + b * p.bt_stride;
  const int64_t row_bytes = static_cast<int64_t>(p.Hkv) * kFewDim * kBytes;
  const int at = kvh * kFewDim + j * 8, batch = gridDim.z;

  struct Tokens {
    FewRow<FP8> k[kFewAhead], v[kFewAhead];
    bool fresh[kFewAhead];          // the row that the new token is being written to
  };
  int64_t new_slot = -1;
  auto load = [&](int tb, Tokens &r) __attribute__((always_inline)) {
    int64_t at_row[kFewAhead];
#pragma unroll
    for (int u = 0; u < kFewAhead; ++u) {
      const int t = tb + u * 16 + team, bi = t / p.bs;
      const int64_t blk = bt[min(bi, p.max_blocks - 1)];
      at_row[u] = t < t1 && blk >= 0 && blk < p.blocks ? blk * p.bs + (t - bi * p.bs) : -1;
    }
#pragma unroll
    for (int u = 0; u < kFewAhead; ++u) {
      r.k[u].zero();
      r.v[u].zero();
      if (at_row[u] >= 0) {                                  // unmapped: zeros
        r.k[u].load(p.k_cache + at_row[u] * row_bytes, at);
        r.v[u].load(p.v_cache + at_row[u] * row_bytes, at);
      }
      r.fresh[u] = RAW && at_row[u] >= 0 && at_row[u] == new_slot;
    }
  };

  auto store = [&](const uint4 v, bool is_k, int64_t slot) __attribute__((always_inline)) {
    unsigned char *to = (is_k ? p.prep.k_cache : p.prep.v_cache) + slot * row_bytes;
    if constexpr (FP8) *reinterpret_cast<int2 *>(to + at) = qk_piece_e4m3(v, (is_k ? p.k_scale : p.v_scale)[kvh]);
    else *reinterpret_cast<uint4 *>(to + at * 2) = v;
  };

  // what the preparation needs, then the first rows
  QkPieceMeta meta;
  QkPieceTable table;
  uint4 raw = make_uint4(0, 0, 0, 0);
  const bool mine = RAW && team < GROUP + 2;
  const int head = team < GROUP ? kvh * GROUP + team : team == GROUP ? p.Hq + kvh : p.Hq + p.Hkv + kvh;
  if constexpr (RAW) {
    if (p.prep.slot_mapping) {
      new_slot = p.prep.slot_mapping[b];
      if (new_slot >= p.prep.num_slots) new_slot = -1;
    }
    if (mine) {
      meta = qk_piece_meta(b, head, p.prep);
      raw = *reinterpret_cast<const uint4 *>(p.x + b * p.ldx + head * kFewDim + j * 8);
      table = qk_piece_table(meta, head, j, p.prep);
    }
  }
  // another sequence's new row, and 32 pages of the share to look for it
  const int seq = tid & 7, at_page = t0 / p.bs + (tid >> 3), last_page = t0 < t1 ? (t1 - 1) / p.bs : -1;
  int to_slot = -1, page = -1;
  if (RAW && batch > 1) {
    if (seq < batch && seq != b && p.prep.slot_mapping) to_slot = p.prep.slot_mapping[seq];
    if (at_page <= last_page) page = bt[at_page];
  }
  Tokens cur;
  load(t0, cur);
  float q[GROUP][8];
  FewRow<FP8> new_k, new_v;
  if constexpr (RAW) {
    if (mine) {
      const uint4 v = qk_piece_value(raw, team <= GROUP, team < GROUP ? p.prep.qw : p.prep.kw, j, meta, table, p.prep);
      rows[team][j] = v;
      if (newest && team >= GROUP && meta.slot >= 0) store(v, team == GROUP, meta.slot);
    }
    if (batch > 1) {
      const int to_page = to_slot >= 0 && to_slot < p.prep.num_slots ? to_slot / p.bs : -1;
      bool other = to_page >= 0 && page == to_page;
      for (int i = at_page + 32; to_page >= 0 && i <= last_page; i += 32) other = other || bt[i] == to_page;
      const bool some = __any(other);
      if (lane == 0) others[wave] = some;
    }
    __syncthreads();
    if (ctx <= 0) return;
    if (batch > 1 && (others[0] | others[1] | others[2] | others[3])) {
      // rows of one sequence in a step: the workgroups that store the others' new rows may come later, so this one stores them, too, the same bits
      const int from = team >> 1;
      const bool is_k = team & 1;
      const int64_t slot = from < batch && from != b ? p.prep.slot_mapping[from] : -1;
      if (slot >= 0 && slot < p.prep.num_slots && slot != new_slot) {
        const int row = p.Hq + (is_k ? 0 : p.Hkv) + kvh;
        const QkPieceMeta m = qk_piece_meta(from, row, p.prep);
        store(qk_piece_value(*reinterpret_cast<const uint4 *>(p.x + from * p.ldx + row * kFewDim + j * 8), is_k, p.prep.kw, j, m,
                             qk_piece_table(m, row, j, p.prep), p.prep), is_k, slot);
      }
      __syncthreads();
      load(t0, cur);
    }
#pragma unroll
    for (int h = 0; h < GROUP; ++h) unpack8(rows[h][j], q[h]);
    new_k.put(rows[GROUP][j], FP8 ? p.k_scale[kvh] : 1.f);
    new_v.put(rows[GROUP + 1][j], FP8 ? p.v_scale[kvh] : 1.f);
  } else {
#pragma unroll
    for (int h = 0; h < GROUP; ++h) unpack8(*reinterpret_cast<const uint4 *>(p.x + b * p.ldx + (kvh * GROUP + h) * kFewDim + j * 8), q[h]);
  }
  const float to_log2 = p.scale_log2 * (FP8 ? p.k_scale[kvh] : 1.f);

  float m[GROUP], l[GROUP], o[GROUP][8];
#pragma unroll
  for (int h = 0; h < GROUP; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[h][e] = 0.f;
  }
  for (int tb = t0; tb < t1; tb += kFewShare) {
    if (tb != t0) load(tb, cur);
    float s[kFewAhead][GROUP];
#pragma unroll
    for (int u = 0; u < kFewAhead; ++u) {
      if (RAW && cur.fresh[u]) {
        cur.k[u] = new_k;
        cur.v[u] = new_v;
      }
      float k[8];
      cur.k[u].get(k);
#pragma unroll
      for (int h = 0; h < GROUP; ++h) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) d = fmaf(k[e], q[h][e], d);
        d += row_ror<8>(d);
        d += row_ror<4>(d);
        d += row_ror<2>(d);
        d += row_ror<1>(d);
        s[u][h] = tb + u * 16 + team < t1 ? d * to_log2 : -INFINITY;
      }
    }
#pragma unroll
    for (int h = 0; h < GROUP; ++h) {
      float top = m[h];
#pragma unroll
      for (int u = 0; u < kFewAhead; ++u) top = fmaxf(top, s[u][h]);
      const float base = top == -INFINITY ? 0.f : top, back = __builtin_amdgcn_exp2f(m[h] - base);
      m[h] = top;
      l[h] *= back;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[h][e] *= back;
#pragma unroll
      for (int u = 0; u < kFewAhead; ++u) {
        s[u][h] = __builtin_amdgcn_exp2f(s[u][h] - base);
        l[h] += s[u][h];
      }
    }
#pragma unroll
    for (int u = 0; u < kFewAhead; ++u) {
      float v[8];
      cur.v[u].get(v);
#pragma unroll
      for (int h = 0; h < GROUP; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) o[h][e] = fmaf(s[u][h], v[e], o[h][e]);
    }
  }

  // the four teams of a wave, then the waves
#pragma unroll
  for (int h = 0; h < GROUP; ++h) {
    const float top = max_lanes_16_32_48(m[h]), f = __builtin_amdgcn_exp2f(m[h] - (top == -INFINITY ? 0.f : top)), sum = sum_lanes_16_32_48(l[h] * f);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[h][e] = sum_lanes_16_32_48(o[h][e] * f);
    if (lane < 16) {
      float *to = &mixes[wave][h][j * 8];
      *reinterpret_cast<float4 *>(to) = make_float4(o[h][0], o[h][1], o[h][2], o[h][3]);
      *reinterpret_cast<float4 *>(to + 4) = make_float4(o[h][4], o[h][5], o[h][6], o[h][7]);
      if (j == 0) {
        stats[wave][h][0] = top;
        stats[wave][h][1] = sum;
      }
    }
  }
  __syncthreads();
  const float vs = FP8 ? p.v_scale[kvh] : 1.f;
  for (int i = tid; i < GROUP * kFewDim / 4; i += 256) {
    const int h = i / (kFewDim / 4), c = i % (kFewDim / 4) * 4, hh = kvh * GROUP + h;
    float top = stats[0][h][0], sum = 0.f;
#pragma unroll
    for (int w = 1; w < 4; ++w) top = fmaxf(top, stats[w][h][0]);      // some token: finite unless its score is not
    const float base = top == -INFINITY ? 0.f : top;
    float4 mix = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = __builtin_amdgcn_exp2f(stats[w][h][0] - base);
      const float4 t = *reinterpret_cast<const float4 *>(&mixes[w][h][c]);
      sum += f * stats[w][h][1];
      mix.x += f * t.x; mix.y += f * t.y; mix.z += f * t.z; mix.w += f * t.w;
    }
    if (ctx <= share) {                                      // nothing to merge
      const float inv = sum > 0.f ? vs / sum : 0.f;
      *reinterpret_cast<uint2 *>(p.out + (static_cast<int64_t>(b) * p.Hq + hh) * kFewDim + c) =
          make_uint2(pack_bf16x2(mix.x * inv, mix.y * inv), pack_bf16x2(mix.z * inv, mix.w * inv));
      continue;
    }
    const int64_t to = (static_cast<int64_t>(b) * p.Hq + hh) * p.splits + split;
    *reinterpret_cast<float4 *>(p.part + to * kFewDim + c) = make_float4(mix.x * vs, mix.y * vs, mix.z * vs, mix.w * vs);
    if (c == 0) *reinterpret_cast<float2 *>(p.ml + to * 2) = make_float2(top, sum);
  }
}

// One workgroup per (query head, sequence): eight teams of 32 lanes take every eighth share.
__global__ __launch_bounds__(256) void decode_few_merge_kernel(const FewArgs p) {
  constexpr int kEach = kFewMaxSplits / 8;
  __shared__ __attribute__((aligned(16))) float mixes[8][kFewDim];
  __shared__ float stats[8][2];
  const int b = blockIdx.y, h = blockIdx.x, tid = threadIdx.x, team = tid >> 5, c = (tid & 31) * 4;
  const int ctx = min(p.ctx[b], p.max_blocks * p.bs), share = few_share(ctx, p.splits), shares = (ctx + share - 1) / share;
  unsigned short *out = p.out + (static_cast<int64_t>(b) * p.Hq + h) * kFewDim + c;
  if (ctx <= 0) {                                            // an empty sequence gets zeros
    if (team == 0) *reinterpret_cast<uint2 *>(out) = make_uint2(0, 0);
    return;
  }
  if (shares == 1) return;
  const int64_t first = (static_cast<int64_t>(b) * p.Hq + h) * p.splits;
  float2 ml[kEach];
  float4 part[kEach];
#pragma unroll
  for (int i = 0; i < kEach; ++i) {
    const int s = team + i * 8;
    ml[i] = make_float2(-INFINITY, 0.f);
    part[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (s < shares) {
      ml[i] = *reinterpret_cast<const float2 *>(p.ml + (first + s) * 2);
      part[i] = *reinterpret_cast<const float4 *>(p.part + (first + s) * kFewDim + c);
    }
  }
  float top = ml[0].x, sum = 0.f;
#pragma unroll
  for (int i = 1; i < kEach; ++i) top = fmaxf(top, ml[i].x);
  auto add = [](float4 &to, float f, const float4 &x) __attribute__((always_inline)) { to.x += f * x.x; to.y += f * x.y; to.z += f * x.z; to.w += f * x.w; };
  float4 mix = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int i = 0; i < kEach; ++i) {
    const float f = ml[i].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[i].x - top);
    sum += f * ml[i].y;
    add(mix, f, part[i]);
  }
  *reinterpret_cast<float4 *>(&mixes[team][c]) = mix;
  if (c == 0) {
    stats[team][0] = top;
    stats[team][1] = sum;
  }
  __syncthreads();
  if (team) return;
#pragma unroll
  for (int i = 1; i < 8; ++i) top = fmaxf(top, stats[i][0]);
  sum = 0.f;
  mix = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float f = stats[i][0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(stats[i][0] - top);
    sum += f * stats[i][1];
    add(mix, f, *reinterpret_cast<const float4 *>(&mixes[i][c]));
  }
  const float inv = sum > 0.f ? 1.0f / sum : 0.f;
  *reinterpret_cast<uint2 *>(out) = make_uint2(pack_bf16x2(mix.x * inv, mix.y * inv), pack_bf16x2(mix.z * inv, mix.w * inv));
}

// Shares there may be: about 512 workgroups, which is what a context of thousands wants (8 sequences of up to 4096 tokens, 32 heads on 8, layer:
// 83 us with 16 shares, 95 with 32: what a workgroup ends with is a fifth of a share of 64).  With eight query heads per KV head a CU holds one workgroup
// and not two or more: as many as there are CUs, or those without a share to work on take a round of their own (attention block, 64 heads on 8, one sequence of 60 tokens,
// us: 33.0 with 31 shares, 36.3 with 64), but 16 at least (four of up to 4096 tokens: 67.6 with 7, 50.5 with 16).
// Where one share fewer keeps the workspace within 1 MiB (63 and not 64 for 32 heads), it is left out: an allocator has such a piece at hand, and a graph that
// is captured takes no memory of its own for it (a larger piece took 0.6 ms of a capture).
inline int64_t few_share_bytes(int batch, int q_heads) { return static_cast<int64_t>(batch) * q_heads * (kFewDim + 2) * 4; }
inline int few_splits(int batch, int q_heads, int kv_heads) {
  const int workgroups = q_heads / kv_heads == 8 ? 256 : 512;
  int splits = kFewMaxSplits;
  while (splits > 16 && splits * batch * kv_heads > workgroups) splits /= 2;
  return (1 << 20) / few_share_bytes(batch, q_heads) == splits - 1 ? splits - 1 : splits;
}

}  // namespace tlf

// Up to 8 sequences of one or two query heads per KV head, up to 4 of more, whose queries and mixes fill the registers (a workgroup of four heads has
// 130 to 160, three a CU).
extern "C" int tlf_decode_few_supported(int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size) {
  const int g = num_kv_heads;
  if (batch <= 0 || head_dim != tlf::kFewDim || block_size <= 0 || block_size % 16) return 0;
  if ((g != 1 && g != 2 && g != 4 && g != 8 && g != 16) || num_q_heads <= 0 || num_q_heads % g) return 0;
  const int group = num_q_heads / g;
  if (group != 1 && group != 2 && group != 4 && group != 8) return 0;
  return group <= 2 ? batch <= 8 && batch * g <= 64 : batch <= 4 && batch * g <= 32;
}

// Whether it is the faster one for all lengths that the tables can hold (a captured step has the tables' width and no lengths): it has a share's rows on their way
// when it has used those before, so where shares get long the kernel of decode_attn.hip overtakes it, and later with fewer sequences, which have more shares.
// Attention block with int8 projections of a width of 4096, us, preparation, paged_decode_kernel and merge / here, longest of contexts of up to a factor of eight:
//   32 heads on 8     1 sequence of 700 32.1 / 27.3, 4096 43.4 / 33.6, 16384 86.3 / 43.7, 65536 114 / 85, 131072 153 / 143;  2 of 700 32.7 / 27.6, 32768 87.6 / 78.1,
//                     65536 115 / 123;  3 of 700 33.3 / 29.5, 8192 59.8 / 48.2, 16384 72.4 / 76.5;  4 of 700 34.8 / 30.1, 8192 59.0 / 54.0, 16384 71.1 / 78.4
//   16 heads on 8     1 of 700 28.6 / 22.7, 65536 110 / 76;  2 of 32768 82.6 / 68.4;  4 of 8192 52.9 / 46.4, 16384 65.6 / 69.0;  8 of 700 32.1 / 27.3,
//                     8192 54.6 / 49.1, 16384 87.2 / 90.4
//   64 heads on 8     1 of 700 38.2 / 35.1, 32768 102 / 92;  2 of 700 39.1 / 35.8, 8192 67.2 / 64.5, 16384 80.9 / 93.8;  3 of 700 39.9 / 39.5, 4096 54.0 / 54.8;
//                     4 of 700 41.7 / 39.9, 4096 54.5 / 50.4, 8192 67.2 / 72.3 (32 on 4 34.4 / 33.9 of 1000, 43.6 / 45.4 of 4096: up to there it is as good either way)
//   16 heads on 16    1 of 700 40.1 / 25.0, 65536 171 / 132;  4 of 700 42.0 / 28.2, 8192 83.7 / 56.6, 32768 176 / 150 (8 on 8 91 / 109)
extern "C" int tlf_decode_few_preferred(int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size, int32_t max_blocks) {
  if (!tlf_decode_few_supported(batch, num_q_heads, num_kv_heads, head_dim, block_size)) return 0;
  const bool eight = num_q_heads / num_kv_heads == 8;
  const int64_t most = batch == 1 ? (eight ? 32768 : 65536) : batch == 2 ? (eight ? 8192 : 32768) : eight ? 4096 : 8192;
  return static_cast<int64_t>(max_blocks) * block_size <= most;
}

extern "C" size_t tlf_decode_few_workspace_bytes(int32_t batch, int32_t num_q_heads, int32_t num_kv_heads) {
  if (batch <= 0 || num_q_heads <= 0 || num_kv_heads <= 0) return 0;
  return static_cast<size_t>(tlf::few_splits(batch, num_q_heads, num_kv_heads) * tlf::few_share_bytes(batch, num_q_heads));
}

extern "C" int tlf_decode_few(const void *x, int64_t x_stride, const void *q_norm_weight, const void *k_norm_weight, float eps,
                              const int64_t *positions, const float *cos_sin, int32_t max_pos, const int32_t *slot_mapping, void *k_cache,
                              void *v_cache, int32_t kv_dtype, const float *k_scale, const float *v_scale, const int32_t *block_tables,
                              int64_t block_table_stride, const int32_t *context_lens, void *out, int32_t batch, int32_t num_q_heads,
                              int32_t num_kv_heads, int32_t head_dim, int32_t block_size, int32_t max_blocks, int64_t num_cache_blocks,
                              float scale, void *workspace, size_t workspace_bytes, void *stream) {
  using namespace tlf;
  if (batch == 0) return TLF_OK;
  if (!x || !k_cache || !v_cache || !block_tables || !context_lens || !out) return TLF_E_NULL;
  if (!tlf_decode_few_supported(batch, num_q_heads, num_kv_heads, head_dim, block_size)) return TLF_E_UNSUPPORTED;
  if (kv_dtype != TLF_KV_BF16 && kv_dtype != TLF_KV_FP8_E4M3) return TLF_E_UNSUPPORTED;
  const bool raw = q_norm_weight != nullptr, f8 = kv_dtype == TLF_KV_FP8_E4M3;
  if (raw && (!k_norm_weight || !positions || !cos_sin)) return TLF_E_NULL;
  if (f8 && (!k_scale || !v_scale)) return TLF_E_NULL;
  const int64_t width = static_cast<int64_t>(num_q_heads + (raw ? 2 * num_kv_heads : 0)) * head_dim;
  if (x_stride < width || max_blocks <= 0 || num_cache_blocks <= 0 || block_table_stride < max_blocks || (raw && max_pos <= 0)) return TLF_E_SHAPE;
  if (static_cast<int64_t>(max_blocks) * block_size > (1ll << 30)) return TLF_E_SHAPE;
  if (!aligned16(x) || x_stride % 8 || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out) || !aligned16(q_norm_weight) ||
      !aligned16(k_norm_weight) || !aligned16(cos_sin))
    return TLF_E_ALIGN;
  if (!workspace || workspace_bytes < tlf_decode_few_workspace_bytes(batch, num_q_heads, num_kv_heads) || !aligned16(workspace)) return TLF_E_WORKSPACE;
  FewArgs a{};
  if (raw) {
    a.prep = QkRopeStoreArgs{};
    a.prep.qw = static_cast<const unsigned short *>(q_norm_weight); a.prep.kw = static_cast<const unsigned short *>(k_norm_weight);
    a.prep.eps = eps; a.prep.positions = positions; a.prep.cos_sin = cos_sin; a.prep.max_pos = max_pos;
    a.prep.k_cache = static_cast<unsigned char *>(k_cache); a.prep.v_cache = static_cast<unsigned char *>(v_cache);
    a.prep.slot_mapping = slot_mapping; a.prep.num_slots = num_cache_blocks * block_size; a.prep.kv_dtype = kv_dtype;
    a.prep.num_q_heads = num_q_heads; a.prep.num_kv_heads = num_kv_heads;
  }
  a.x = static_cast<const unsigned short *>(x); a.ldx = x_stride;
  a.k_cache = static_cast<const unsigned char *>(k_cache); a.v_cache = static_cast<const unsigned char *>(v_cache);
  a.k_scale = k_scale; a.v_scale = v_scale; a.bt = block_tables; a.bt_stride = block_table_stride; a.ctx = context_lens;
  a.out = static_cast<unsigned short *>(out); a.blocks = num_cache_blocks; a.Hq = num_q_heads; a.Hkv = num_kv_heads; a.bs = block_size;
  a.max_blocks = max_blocks; a.scale_log2 = scale * kFewLog2e;
  const int most = (max_blocks * block_size + kFewShare - 1) / kFewShare, splits = few_splits(batch, num_q_heads, num_kv_heads);
  a.splits = splits < most ? splits : most;
  a.part = static_cast<float *>(workspace);
  a.ml = a.part + static_cast<int64_t>(batch) * num_q_heads * a.splits * kFewDim;
  const dim3 grid(a.splits, num_kv_heads, batch), block(256);
  hipStream_t s = static_cast<hipStream_t>(stream);
#define TLF_FEW_R(G, F8)                                                                                  \
  do {                                                                                                    \
    if (raw) TLF_LAUNCH((decode_few_kernel<G, F8, true>), grid, block, 0, s, a);                          \
    else TLF_LAUNCH((decode_few_kernel<G, F8, false>), grid, block, 0, s, a);                             \
  } while (0)
#define TLF_FEW(G)                  \
  case G:                           \
    if (f8) TLF_FEW_R(G, true);     \
    else TLF_FEW_R(G, false);       \
    break;
  switch (num_q_heads / num_kv_heads) {
    TLF_FEW(1) TLF_FEW(2) TLF_FEW(4) TLF_FEW(8)
  }
#undef TLF_FEW
#undef TLF_FEW_R
  if (int rc = launch_status()) return rc;
  TLF_LAUNCH(decode_few_merge_kernel, dim3(num_q_heads, batch), block, 0, s, a);
  return launch_status();
}
