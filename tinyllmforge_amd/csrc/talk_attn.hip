// In front of the attention of talk_attn.h: projection row [q | k | v] -> RMS norm over all of q and over all of k, rotation of
// the first rot_dims dimensions of every head in pairs (2 i, 2 i + 1), the score's constants (with a temperature per head) into
// q, keys and values into the paged caches.  One workgroup per token and part.  HBM bound: a row is read once and written once.
#include <algorithm>

#include "talk_attn.h"

namespace tlf {

struct TalkPrepArgs {
  const void *proj;            // [n, ld]: q heads, k heads, v heads
  Partials part;               // or its partial sums
  int64_t ld;
  const void *q_norm, *k_norm; // [H * D], [G * D]
  const void *temp;            // [H] or NULL
  const int64_t *positions;
  const float *cos_sin;        // [max_pos, rot_dims]: cos of the pairs, then sin
  int32_t max_pos, rot_dims;
  const int32_t *slots;        // cache slot per token, negative: no store
  void *q_out;                 // [n, H, Dp]
  SinkCache c;
  int32_t n, H, vec;
  float eps, q_scale;
};

// blockIdx.y 0: q, 1: k, 2: v; pieces of 8 elements of a head, MAXC per thread
template <typename T, int MAXC, bool PART>
__global__ __launch_bounds__(256) void talk_prep_kernel(const TalkPrepArgs a) {
  __shared__ float part[4];
  const SinkCache &c = a.c;
  const int64_t tok = blockIdx.x;
  const int kind = blockIdx.y, heads = kind == 0 ? a.H : c.G, dims = kind < 2 ? c.D : c.Dv, padded = kind < 2 ? c.Dp : c.Vp;
  const int col0 = kind == 0 ? 0 : kind == 1 ? a.H * c.D : (a.H + c.G) * c.D;
  const int nch = padded / 8, pieces = heads * nch;
  const int64_t pos = a.positions[tok], slot = a.slots[tok];
  float x[MAXC][8], ss = 0.f;
#pragma unroll
  for (int q = 0; q < MAXC; ++q) {
    const int piece = static_cast<int>(threadIdx.x) + q * 256, head = piece / nch, d = (piece - head * nch) * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[q][e] = 0.f;
    if (piece >= pieces || d >= dims) continue;
    const int col = col0 + head * dims + d;
    if (a.vec) {
      if constexpr (PART) a.part.ld8(tok, col, x[q]);
      else Elem<T>::ld8(static_cast<const T *>(a.proj) + tok * a.ld + col, x[q]);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (d + e < dims) x[q][e] = PART ? a.part.ld(tok, col + e) : Elem<T>::ld(static_cast<const T *>(a.proj) + tok * a.ld + col + e);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(x[q][e], x[q][e], ss);
  }
  float inv = 1.f;
  if (kind < 2) {
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = (part[0] + part[1]) + (part[2] + part[3]);
    inv = 1.0f / sqrtf(ss / static_cast<float>(heads * dims) + a.eps);
  }
  const bool store = slot >= 0 && slot < c.pages * c.bs;
  if (kind > 0 && !store) return;
  const int64_t page = store ? slot / c.bs : 0;
  const T *w = static_cast<const T *>(kind == 0 ? a.q_norm : a.k_norm);
  const int half = a.rot_dims / 2;
  const float *cs = pos >= 0 && pos < a.max_pos && half ? a.cos_sin + pos * a.rot_dims : nullptr;
#pragma unroll
  for (int q = 0; q < MAXC; ++q) {
    const int piece = static_cast<int>(threadIdx.x) + q * 256, head = piece / nch, d = (piece - head * nch) * 8;
    if (piece >= pieces) continue;
    if (kind < 2 && d < dims) {
      float wn[8];
      if (a.vec) Elem<T>::ld8(w + head * dims + d, wn);
      else
#pragma unroll
        for (int e = 0; e < 8; ++e) wn[e] = d + e < dims ? Elem<T>::ld(w + head * dims + d + e) : 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) x[q][e] = x[q][e] * inv * wn[e];
      if (cs && d < a.rot_dims) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const int i = (d + e) / 2;
          if (i < half) {
            const float co = cs[i], si = cs[half + i], u = x[q][e], v = x[q][e + 1];
            x[q][e] = __fmul_rn(u, co) - __fmul_rn(v, si);
            x[q][e + 1] = __fmul_rn(v, co) + __fmul_rn(u, si);
          }
        }
      }
    }
    if (kind == 0) {
      const float m = a.q_scale * (a.temp ? Elem<T>::ld(static_cast<const T *>(a.temp) + head) : 1.f);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[q][e] *= m;
      Elem<T>::st8(static_cast<T *>(a.q_out) + (tok * a.H + head) * c.Dp + d, x[q]);
    } else {
      const int64_t crow = (page * c.G + head) * c.bs + (slot - page * c.bs);
      T *dst = static_cast<T *>(const_cast<void *>(kind == 1 ? c.k : c.v));
      Elem<T>::st8(dst + crow * padded + d, x[q]);
    }
  }
}

// The same for rows of prompts: bf16 projections, head dimensions that are padded nowhere, q of 64, 128, 256 or 512 granules of 8 values, k and v
// of one of these.  A workgroup has eight rows of one part; WPR waves have a row, CH granules a lane, and NB rows each are on their way
// at once: the kernel above waits for a row, for its sum and then for norm weights, cosines and sines.
//
// HBM bound: 12237 rows of 16 + 2 x 8 heads of 128, 200 MB, 65 us a row and part a workgroup, 49 so (a large copy 39); 32 heads 111 and 70.
constexpr int kPrepRows = 8;

template <int WPR, int CH>
__device__ __forceinline__ void talk_prep_rows(const TalkPrepArgs &a, int kind, float (&part)[kPrepRows][4]) {
  typedef unsigned short T;
  constexpr int AT = 4 / WPR, NB = kPrepRows / AT < 4 / CH ? kPrepRows / AT : 4 / CH;   // rows at a time; of a thread
  const SinkCache &c = a.c;
  const int heads = kind == 0 ? a.H : c.G, dims = kind < 2 ? c.D : c.Dv, nch = dims / 8;
  const int col0 = kind == 0 ? 0 : kind == 1 ? a.H * c.D : (a.H + c.G) * c.D;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, own = wave / WPR, half = a.rot_dims / 2;
  uint4 x[NB][CH];
  int piece[CH];
#pragma unroll
  for (int q = 0; q < CH; ++q) piece[q] = (q * WPR + wave % WPR) * 64 + lane;
  for (int first = 0; first < kPrepRows; first += NB * AT) {
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kPrepRows + first + own;
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    const T *from = static_cast<const T *>(a.proj) + min(row0 + k * AT, static_cast<int64_t>(a.n) - 1) * a.ld + col0;
#pragma unroll
    for (int q = 0; q < CH; ++q) x[k][q] = *reinterpret_cast<const uint4 *>(from + piece[q] * 8);
  }
  int64_t pos[NB];
  int32_t slot[NB];
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    const int64_t row = min(row0 + k * AT, static_cast<int64_t>(a.n) - 1);
    pos[k] = a.positions[row];
    slot[k] = a.slots[row];
  }
  float inv[NB];
  uint4 w[CH];
  if (kind < 2) {
    const T *wp = static_cast<const T *>(kind == 0 ? a.q_norm : a.k_norm);
#pragma unroll
    for (int q = 0; q < CH; ++q) w[q] = *reinterpret_cast<const uint4 *>(wp + piece[q] * 8);
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      float ss = 0.f;
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        float f[8];
        unpack8(x[k][q], f);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(f[e], f[e], ss);
      }
      inv[k] = wave_sum(ss);
    }
    if constexpr (WPR > 1) {
      if (lane == 0)
#pragma unroll
        for (int k = 0; k < NB; ++k) part[first + own + k * AT][wave % WPR] = inv[k];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const float *s = part[first + own + k * AT];
        inv[k] = WPR == 2 ? s[0] + s[1] : (s[0] + s[1]) + (s[2] + s[3]);
      }
    }
#pragma unroll
    for (int k = 0; k < NB; ++k) inv[k] = 1.0f / sqrtf(inv[k] / static_cast<float>(heads * dims) + a.eps);
  }
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    const int64_t row = row0 + k * AT;
    const bool store = row < a.n && (kind == 0 || (slot[k] >= 0 && slot[k] < c.pages * c.bs));
    const int page = c.bs_shift >= 0 ? slot[k] >> c.bs_shift : slot[k] / c.bs;
    const bool turns = pos[k] >= 0 && pos[k] < a.max_pos && half;
    const float *cs = a.cos_sin + (turns ? pos[k] : 0) * a.rot_dims;
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      const int head = piece[q] / nch, d = (piece[q] - head * nch) * 8;
      uint4 out = x[k][q];
      if (kind < 2) {
        float f[8], wn[8];
        unpack8(x[k][q], f);
        unpack8(w[q], wn);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = f[e] * inv[k] * wn[e];
        if (turns && d < a.rot_dims) {                               // rotations end between granules
          const float4 co = *reinterpret_cast<const float4 *>(cs + d / 2), si = *reinterpret_cast<const float4 *>(cs + half + d / 2);
          const float cv[4] = {co.x, co.y, co.z, co.w}, sv[4] = {si.x, si.y, si.z, si.w};
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            const float u = f[e], v = f[e + 1];
            f[e] = __fmul_rn(u, cv[e / 2]) - __fmul_rn(v, sv[e / 2]);
            f[e + 1] = __fmul_rn(v, cv[e / 2]) + __fmul_rn(u, sv[e / 2]);
          }
        }
        if (kind == 0) {
          const float m = a.q_scale * (a.temp ? Elem<T>::ld(static_cast<const T *>(a.temp) + head) : 1.f);
#pragma unroll
          for (int e = 0; e < 8; ++e) f[e] *= m;
        }
        out = pack8(f);
      }
      if (!store) continue;
      T *to = kind == 0 ? static_cast<T *>(a.q_out) + (row * a.H + head) * dims + d
                        : static_cast<T *>(const_cast<void *>(kind == 1 ? c.k : c.v)) + ((static_cast<int64_t>(page) * c.G + head) * c.bs + (slot[k] - page * c.bs)) * dims + d;
      *reinterpret_cast<uint4 *>(to) = out;
    }
  }
  }
}

// WIDE: some part has 512 granules.  Without, its two granules a lane cost the others no registers: 52 -> 49 us above.
template <bool WIDE>
__global__ __launch_bounds__(256) void talk_prep_rows_kernel(const TalkPrepArgs a) {
  __shared__ float part[kPrepRows][4];
  const int kind = blockIdx.y, granules = (kind == 0 ? a.H * a.c.D : a.c.G * (kind == 1 ? a.c.D : a.c.Dv)) / 8;
  if (WIDE && granules == 512) talk_prep_rows<4, 2>(a, kind, part);
  else if (granules == 256) talk_prep_rows<4, 1>(a, kind, part);
  else if (granules == 128) talk_prep_rows<2, 1>(a, kind, part);
  else talk_prep_rows<1, 1>(a, kind, part);
}
// Sizes it takes, from 2048 rows on (4000 rows of 16 heads 26 and 20 us, 2100 of 32 heads 22 and 22); with fewer, a row a workgroup fills the chip.
inline bool talk_prep_takes_rows(const TalkPrepArgs &a) {
  auto whole = [](int64_t granules) { return granules == 64 || granules == 128 || granules == 256 || granules == 512; };
  const SinkCache &c = a.c;
  return a.vec && a.n >= 2048 && c.D == c.Dp && c.Dv == c.Vp && a.rot_dims % 8 == 0 && (!a.rot_dims || aligned16(a.cos_sin)) &&
         whole(static_cast<int64_t>(a.H) * c.D / 8) && whole(static_cast<int64_t>(c.G) * c.D / 8) && whole(static_cast<int64_t>(c.G) * c.Dv / 8);
}

template <typename T, bool PART>
int launch_talk_prep(const TalkPrepArgs &a, int pieces, hipStream_t s) {
  if constexpr (sizeof(T) == 2 && !PART)
    if (talk_prep_takes_rows(a)) {
      const dim3 grid((a.n + kPrepRows - 1) / kPrepRows, 3);
      const int most = std::max(a.H * a.c.D, a.c.G * std::max(a.c.D, a.c.Dv));
      if (most == 512 * 8) TLF_LAUNCH(talk_prep_rows_kernel<true>, grid, dim3(256), 0, s, a);
      else TLF_LAUNCH(talk_prep_rows_kernel<false>, grid, dim3(256), 0, s, a);
      return launch_status();
    }
  const dim3 grid(a.n, 3);
  if (pieces <= 256) TLF_LAUNCH((talk_prep_kernel<T, 1, PART>), grid, dim3(256), 0, s, a);
  else if (pieces <= 512) TLF_LAUNCH((talk_prep_kernel<T, 2, PART>), grid, dim3(256), 0, s, a);
  else if (pieces <= 1024) TLF_LAUNCH((talk_prep_kernel<T, 4, PART>), grid, dim3(256), 0, s, a);
  else TLF_LAUNCH((talk_prep_kernel<T, 16, PART>), grid, dim3(256), 0, s, a);
  return launch_status();
}

}  // namespace tlf

extern "C" int tlf_talk_prep(const void *proj, int64_t proj_stride, const float *partials, int32_t splits, const float *scale,
                             const void *q_norm, const void *k_norm, const void *temp, const int64_t *positions,
                             const float *cos_sin, int32_t max_pos, int32_t rot_dims, const int32_t *slot_mapping, void *q_out,
                             void *k_cache, void *v_cache, int32_t n, int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim,
                             int32_t block_size, int64_t num_pages, float eps, float score_scale, int32_t dtype, void *stream) {
  using namespace tlf;
  TalkPrepArgs a{};
  if (n < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || rot_dims < 0 || rot_dims % 2 || rot_dims > dim) return TLF_E_SHAPE;
  if (dtype != TLF_DT_BF16 && dtype != TLF_DT_F32) return TLF_E_UNSUPPORTED;
  if (n == 0) return TLF_OK;
  if (int rc = partials_check(partials, scale, splits, dtype)) return rc;
  if (int rc = sink_cache_make(a.c, k_cache, v_cache, nullptr, 0, block_size, kv_heads, dim, vdim, num_pages)) return rc;
  const int64_t cols = static_cast<int64_t>(heads + kv_heads) * dim + static_cast<int64_t>(kv_heads) * vdim;
  if (proj_stride < cols || proj_stride > (1 << 28)) return TLF_E_SHAPE;
  const int64_t pq = static_cast<int64_t>(heads) * (a.c.Dp / 8), pv = static_cast<int64_t>(kv_heads) * (a.c.Vp / 8), pieces = pq > pv ? pq : pv;
  if (pieces > 4096) return TLF_E_SHAPE;
  if ((!proj && splits <= 1) || !q_norm || !k_norm || !positions || !slot_mapping || !q_out || (rot_dims && !cos_sin)) return TLF_E_NULL;
  if (!aligned16(q_out)) return TLF_E_ALIGN;
  a.proj = proj; a.ld = proj_stride;
  a.part = Partials{partials, scale, n * proj_stride, static_cast<int32_t>(proj_stride), splits};
  a.q_norm = q_norm; a.k_norm = k_norm; a.temp = temp; a.positions = positions; a.cos_sin = cos_sin; a.max_pos = max_pos;
  a.rot_dims = rot_dims; a.slots = slot_mapping; a.q_out = q_out; a.n = n; a.H = heads; a.eps = eps;
  a.q_scale = score_scale * kSinkLog2e;
  a.vec = dim % 8 == 0 && vdim % 8 == 0 && proj_stride % 8 == 0 && (splits > 1 || aligned16(proj)) && aligned16(q_norm) && aligned16(k_norm);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (splits > 1) return launch_talk_prep<unsigned short, true>(a, static_cast<int>(pieces), s);
  return dtype == TLF_DT_BF16 ? launch_talk_prep<unsigned short, false>(a, static_cast<int>(pieces), s)
                              : launch_talk_prep<float, false>(a, static_cast<int>(pieces), s);
}
