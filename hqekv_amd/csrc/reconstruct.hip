// A hybrid cache back into dense fp16 K and V (B,Hkv,T,D) (KV_cache_reconstruct, quant/hybrid_quant.py:732-846, and
// KV_cache_reconstruct_hqe, quant/hqe_2.py:967-1084): every class dequantised with the reference's two fp16 roundings
// (quant/pack_unpack.py:331-332) and written to its tokens' positions, both sides in one launch.
//
// Bound: HBM -- the cache is read once and the dense tensors are written once, 16 bytes per lane.  A workgroup takes 128
// tokens of one class of one (b, kv head).  V classes and token-major fp16 rows are 16 lanes (8 channels each) per token
// as they lie.  K classes are channel-major, the result is token-major: a wave takes one 32-token group, a lane two
// channels of it (its codes are one short run of each row; the four waves read neighbouring runs of the same lines), and
// turns it in a corner of LDS of its own, sixteen tokens at a time -- 68 words per token row, so the channel-pair writes
// walk all banks and the 16-byte reads stay aligned.  17 KB of LDS and 67 registers: seven workgroups per CU, no barrier.
// Measured at B=1 of the fp16 / 8 / 4 / 2-bit mix, us a launch: 16k tokens (73 MB) 258 as dequantise launches, transposing copies
// and index_put scatters, 28.9 with the whole 128-token tile in LDS (four workgroups per CU, and 80 bytes of scratch memory
// per lane for what is a uint4 in an array), now 26.6; 512 tokens 7.0 -> 6.1, 64k 103 -> 88, 2 x 64k 197 -> 158.  Positions
// that are looked at for the first time cost two position checks and a wait for each on top (see cover_once_kernel).
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "quant_math.h"

#pragma clang fp contract(off)

namespace hq {

struct RcSeg {
  const void *data;
  const half_t *scale;
  const half_t *zero;
  const int64_t *idx;
  half_t *out;          // the dense tensor of this segment's side
  int64_t pos_base;
  int64_t slab_tokens;  // token rows between two (b, kv head) slabs of a token-major segment
  int32_t n_tokens;
  int16_t bits;
  int16_t kind;         // 0: channel-major K, 1: token-major; + 2: 1-bit normal-quantile coding
};
typedef uint32_t rc_words_t __attribute__((ext_vector_type(4)));   // (uint4 in an array went through scratch memory)
constexpr int RC_SEGS = 2 * HQEKV_MAX_SEGS;
struct RcTable {
  RcSeg seg[RC_SEGS];
  int32_t begin[RC_SEGS];   // first tile of every segment, counted from grid.y = 0 of the launch; INT32_MAX past the last
};

constexpr int RC_THREADS = 256;
constexpr int RC_TOK = 128;    // tokens per workgroup
constexpr int RC_CH = 128;     // channels turned in LDS at a time
constexpr int RC_ROW = 68;     // 32-bit words per token row in LDS
constexpr int RC_HALF = 16;    // tokens a wave turns at a time
constexpr int64_t RC_GRID_Y = 65535;

// keep LDS traffic of one wave in program order (the hardware does; this holds the compiler to it)
__device__ __forceinline__ void rc_wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// where token t of the segment goes; -1: outside the dense tensor (an index counts from the end when negative, as in
// torch; one that names no row is dropped)
__device__ __forceinline__ int64_t rc_position(const RcSeg &s, int64_t t, int64_t T) {
  int64_t p = s.idx ? s.idx[t] : s.pos_base + t;
  if (p < 0) p += T;
  return p >= 0 && p < T ? p : -1;
}

// the value of a code pair: rnd16(rnd16(c * scale) + zero), or rnd16(rnd16(+-k * std) + mean)
template <bool NORMAL>
__device__ __forceinline__ half2_t rc_value(uint32_t c0, uint32_t c1, half2_t s2, half2_t z2) {
  half2_t c;
  if (NORMAL) {
    c[0] = c0 ? (half_t)0.67431640625f : (half_t)-0.67431640625f;
    c[1] = c1 ? (half_t)0.67431640625f : (half_t)-0.67431640625f;
  } else {
    c[0] = (half_t)(unsigned short)c0;
    c[1] = (half_t)(unsigned short)c1;
  }
  const half2_t m = c * s2;
  return m + z2;
}

// 8 adjacent channels of one token: BITS bytes of codes in the low bits of w0 (and w1)
template <int BITS, bool NORMAL>
__device__ __forceinline__ rc_words_t rc_piece(uint32_t w0, uint32_t w1, half_t s, half_t z) {
  const half2_t s2 = {s, s}, z2 = {z, z};
  uint32_t r[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t w = BITS == 8 && j >= 2 ? w1 : w0;
    const int k = BITS == 8 ? 2 * (j & 1) : 2 * j;
    r[j] = h2_bits(rc_value<NORMAL>(code_at<BITS>(w, k), code_at<BITS>(w, k + 1), s2, z2));
  }
  return (rc_words_t){r[0], r[1], r[2], r[3]};
}

// `dim`: head_dim where it is known (128: the pieces of a row are counted by shifts)
template <int BITS, bool NORMAL, typename Dim>
__device__ __forceinline__ void rc_token_major_of(const RcSeg &s, int64_t bh, int t0, Dim dim, int64_t T) {
  const int D = dim;
  const int P = D >> 3, items = RC_TOK * P;   // pieces of 8 channels
  constexpr int U = 4;
  for (int i0 = threadIdx.x; i0 < items; i0 += U * RC_THREADS) {
    rc_words_t v[U];
    half_t sc[U], zr[U];
    int64_t pos[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {   // the requests of U pieces together
      const int i = i0 + u * RC_THREADS;
      const int t = t0 + i / P, cp = i % P;
      const bool in = i < items && t < s.n_tokens;
      const int64_t row = bh * s.slab_tokens + (in ? t : t0);
      const char *src = (const char *)s.data + (row * D + cp * 8) * BITS / 8;
      pos[u] = in ? rc_position(s, t, T) : -1;
      if (BITS == 16) {
        v[u] = *reinterpret_cast<const rc_words_t *>(src);
      } else {
        if (BITS == 8) {
          v[u].x = reinterpret_cast<const uint32_t *>(src)[0];
          v[u].y = reinterpret_cast<const uint32_t *>(src)[1];
        } else if (BITS == 4) {
          v[u].x = *reinterpret_cast<const uint32_t *>(src);
        } else if (BITS == 2) {
          v[u].x = *reinterpret_cast<const unsigned short *>(src);
        } else {
          v[u].x = *reinterpret_cast<const unsigned char *>(src);
        }
        const int64_t g = row * (D >> 5) + (cp >> 2);
        sc[u] = s.scale[g];
        zr[u] = s.zero[g];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int cp = (i0 + u * RC_THREADS) % P;
      if constexpr (BITS != 16) v[u] = rc_piece<BITS, NORMAL>(v[u].x, v[u].y, sc[u], zr[u]);
      if (pos[u] >= 0) *reinterpret_cast<rc_words_t *>(s.out + (bh * T + pos[u]) * D + cp * 8) = v[u];
    }
  }
}
template <int BITS, bool NORMAL>
__device__ __forceinline__ void rc_token_major(const RcSeg &s, int64_t bh, int t0, int D, int64_t T) {
  if (D == 128) rc_token_major_of<BITS, NORMAL>(s, bh, t0, std::integral_constant<int, 128>{}, T);
  else rc_token_major_of<BITS, NORMAL>(s, bh, t0, D, T);
}

template <int BITS, bool NORMAL>
__device__ __forceinline__ void rc_channel_major(const RcSeg &s, int64_t bh, int t0, int D, int64_t T, uint32_t *tiles) {
  const int dp = threadIdx.x & 63, g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // channel pair, 32-token group
  const int n = s.n_tokens, tg = t0 + 32 * g;              // the group's first token
  if (tg >= n) return;                                      // (whole waves; nothing below is shared between them)
  uint32_t *tile = tiles + g * (RC_HALF * RC_ROW);
  // where the lane's 16-byte pieces go: a piece of token dp / P + ... of each half.  Asked for ahead of the codes.
  const int P = min(RC_CH, D) >> 3;                         // pieces of a token row
  int64_t pos[2][RC_HALF / 4];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < RC_HALF / 4; ++j) {
      const int k = RC_HALF * h + 4 * j + (dp >> 4);        // (for rows of 128 channels; others ask again below)
      pos[h][j] = tg + k < n ? rc_position(s, tg + k, T) : -1;
    }
  for (int c0 = 0; c0 < D; c0 += RC_CH) {
    const int d = min(c0 + 2 * dp, D - 2);                  // (past the last channel: that one again, not stored)
    uint32_t a[BITS], b[BITS];   // the group's words of both channels
    half2_t s2 = {}, z2 = {};
    {
      if constexpr (BITS == 16) {
        const half_t *ra = (const half_t *)s.data + (bh * D + d) * (int64_t)n + tg, *rb = ra + n;
        if ((n & 7) == 0) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int at = tg + 8 * q < n ? q : 0;          // (past the class's end: the first eight again, not stored)
            const uint4 x = reinterpret_cast<const uint4 *>(ra)[at], y = reinterpret_cast<const uint4 *>(rb)[at];
            a[4 * q] = x.x; a[4 * q + 1] = x.y; a[4 * q + 2] = x.z; a[4 * q + 3] = x.w;
            b[4 * q] = y.x; b[4 * q + 1] = y.y; b[4 * q + 2] = y.z; b[4 * q + 3] = y.w;
          }
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int k0 = min(2 * i, n - 1 - tg), k1 = min(2 * i + 1, n - 1 - tg);
            a[i] = h2_bits((half2_t){ra[k0], ra[k1]});
            b[i] = h2_bits((half2_t){rb[k0], rb[k1]});
          }
        }
      } else {   // (the class holds whole groups of 32 tokens)
        const int64_t ga = (bh * D + d) * (int64_t)(n >> 5) + (tg >> 5), gb = ga + (n >> 5);
        const uint32_t *wa = (const uint32_t *)s.data + ga * BITS, *wb = (const uint32_t *)s.data + gb * BITS;
#pragma unroll
        for (int i = 0; i < BITS; ++i) {
          a[i] = wa[i];
          b[i] = wb[i];
        }
        s2 = (half2_t){s.scale[ga], s.scale[gb]};
        z2 = (half2_t){s.zero[ga], s.zero[gb]};
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      {
        uint32_t *col = tile + dp;
#pragma unroll
        for (int i = 0; i < RC_HALF; ++i) {
          const int k = RC_HALF * h + i;
          if constexpr (BITS == 16) {
            col[i * RC_ROW] = __builtin_amdgcn_perm(b[k / 2], a[k / 2], k & 1 ? 0x07060302u : 0x05040100u);
          } else {
            constexpr int PF = 32 / BITS;
            col[i * RC_ROW] = h2_bits(rc_value<NORMAL>(code_at<BITS>(a[k / PF], k % PF), code_at<BITS>(b[k / PF], k % PF), s2, z2));
          }
        }
      }
      rc_wave_fence();
      if (P == 16 && c0 + RC_CH <= D) {
#pragma unroll
        for (int j = 0; j < RC_HALF / 4; ++j)
          if (pos[h][j] >= 0)
            *reinterpret_cast<uint4 *>(s.out + (bh * T + pos[h][j]) * D + c0 + (dp & 15) * 8) =
                *reinterpret_cast<const uint4 *>(tile + (4 * j + (dp >> 4)) * RC_ROW + (dp & 15) * 4);
      } else {   // other head sizes, and the last channels of one that is no multiple of 128
        const int pieces = min(RC_CH, D - c0) >> 3;
        for (int i = dp; i < RC_HALF * pieces; i += 64) {
          const int k = i / pieces, cp = i % pieces, t = tg + RC_HALF * h + k;
          const int64_t p = t < n ? rc_position(s, t, T) : -1;
          if (p >= 0) *reinterpret_cast<uint4 *>(s.out + (bh * T + p) * D + c0 + cp * 8) = *reinterpret_cast<const uint4 *>(tile + k * RC_ROW + cp * 4);
        }
      }
      rc_wave_fence();
    }
  }
}

__global__ __launch_bounds__(RC_THREADS, 7) void cache_reconstruct_kernel(RcTable tb, int D, int64_t T) {
  __shared__ __align__(16) uint32_t tile[RC_THREADS / 64 * RC_HALF * RC_ROW];
  int si = -1, first = 0;
#pragma unroll
  for (int k = 0; k < RC_SEGS; ++k) {
    const bool in = (int)blockIdx.y >= tb.begin[k];
    si += in ? 1 : 0;
    first = in ? tb.begin[k] : first;
  }
  const RcSeg s = tb.seg[si];
  const int64_t bh = blockIdx.x;
  const int t0 = ((int)blockIdx.y - first) * RC_TOK;
#define HQ_RC(B_, N_) \
  if (s.kind & 1) rc_token_major<B_, N_>(s, bh, t0, D, T); else rc_channel_major<B_, N_>(s, bh, t0, D, T, tile)
  switch (s.bits) {
    case 16: HQ_RC(16, false); break;
    case 8: HQ_RC(8, false); break;
    case 4: HQ_RC(4, false); break;
    case 2: HQ_RC(2, false); break;
    default:
      if (s.kind & 2) { HQ_RC(1, true); } else { HQ_RC(1, false); }
  }
#undef HQ_RC
}

// One bit per position: a position outside [0, n) or whose bit is set already raises status.  With as many indices as
// positions, no complaint means every position is named once.
struct CoverArgs {
  const int64_t *idx[HQEKV_MAX_SEGS];
  int64_t begin[HQEKV_MAX_SEGS];   // first of the back-to-back numbering; INT64_MAX past the last array
};
__global__ __launch_bounds__(256) void cover_once_kernel(CoverArgs a, int64_t n, uint32_t *status, uint32_t *bits) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int64_t *src = a.idx[0];
  int64_t first = 0;
#pragma unroll
  for (int k = 1; k < HQEKV_MAX_SEGS; ++k) {
    const bool in = i >= a.begin[k];
    src = in ? a.idx[k] : src;
    first = in ? a.begin[k] : first;
  }
  const int64_t at = i - first, p = src[at];
  const uint32_t bit = 1u << (p & 31);
  uint32_t bad = p < 0 || p >= n || (atomicOr(bits + (p >> 5), bit) & bit) ? 1u : 0u;
  if (p != src[at & ~31LL] + (at & 31)) bad |= 2u;
  if (bad) atomicOr(status, bad);
}

}  // namespace hq

using namespace hq;

extern "C" int hqekv_cover_once(const int64_t *const *idx, const int64_t *counts, int n_arrays, void *scratch, int64_t scratch_bytes,
                                void *stream) {
  if (n_arrays <= 0 || n_arrays > HQEKV_MAX_SEGS || !idx || !counts || !scratch) return fail(HQEKV_E_ARG, "cover_once: bad arrays");
  CoverArgs a{};
  int64_t n = 0;
  for (int k = 0; k < HQEKV_MAX_SEGS; ++k) {
    if (k < n_arrays && (counts[k] < 0 || (counts[k] > 0 && !idx[k]))) return fail(HQEKV_E_ARG, "cover_once: bad array %d", k);
    a.idx[k] = k < n_arrays ? idx[k] : nullptr;
    a.begin[k] = k < n_arrays ? n : 0x7fffffffffffffffLL;
    if (k < n_arrays) n += counts[k];
  }
  if (n == 0) return HQEKV_OK;
  if (n > (1LL << 38)) return fail(HQEKV_E_UNSUPPORTED, "cover_once: too many positions");
  if ((uintptr_t)scratch & 3) return fail(HQEKV_E_ALIGN, "cover_once: scratch not 4-byte aligned");
  if (scratch_bytes < 4 * (1 + (n + 31) / 32)) return fail(HQEKV_E_WORKSPACE, "cover_once: scratch too small");
  hipLaunchKernelGGL(cover_once_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, a, n,
                     (uint32_t *)scratch, (uint32_t *)scratch + 1);
  return check_launch("cover_once_kernel");
}

extern "C" int hqekv_cache_reconstruct(const hqekv_seg *k_segs, int n_k, const hqekv_seg *v_segs, int n_v, void *K, void *V,
                                       int64_t BH, int64_t D, int64_t T, void *stream) {
  if (n_k < 0 || n_k > HQEKV_MAX_SEGS || n_v < 0 || n_v > HQEKV_MAX_SEGS || (n_k && (!k_segs || !K)) || (n_v && (!v_segs || !V)))
    return fail(HQEKV_E_ARG, "cache_reconstruct: bad segment tables");
  if (BH <= 0 || BH > 0x7fffffffLL || D <= 0 || D % 32 != 0 || D > 4096 || T < 0)
    return fail(HQEKV_E_ARG, "cache_reconstruct: need B*H > 0 and head_dim a multiple of 32 up to 4096");
  if (((uintptr_t)K | (uintptr_t)V) & 15) return fail(HQEKV_E_ALIGN, "cache_reconstruct: dense tensors must be 16-byte aligned");
  RcTable tb{};
  int m = 0;
  int64_t tiles = 0;
  for (int k = 0; k < n_k + n_v; ++k) {
    const bool is_k = k < n_k;
    const hqekv_seg &s = is_k ? k_segs[k] : v_segs[k - n_k];
    if (s.n_tokens < 0 || s.n_tokens >= (1LL << 30)) return fail(HQEKV_E_ARG, "cache_reconstruct: segment %d: bad n_tokens", k);
    if (s.n_tokens == 0) continue;
    if (!(s.bits == 16 || s.bits == 8 || s.bits == 4 || s.bits == 2 || s.bits == 1))
      return fail(HQEKV_E_ARG, "cache_reconstruct: segment %d bits=%d", k, s.bits);
    if (!s.data || (s.bits != 16 && (!s.scale || !s.zero))) return fail(HQEKV_E_ARG, "cache_reconstruct: segment %d lacks data / scale / zero", k);
    if ((uintptr_t)s.data & (s.bits == 16 ? 15 : 3)) return fail(HQEKV_E_ALIGN, "cache_reconstruct: segment %d data misaligned", k);
    const bool tm = !is_k || (s.bits == 16 && (s.layout & 3) == HQEKV_LAYOUT_TOKEN_MAJOR);
    if (!tm && s.bits != 16 && s.n_tokens % 32) return fail(HQEKV_E_ARG, "cache_reconstruct: segment %d n_tokens not a multiple of 32", k);
    if (s.slab_tokens != 0 && (s.slab_tokens < s.n_tokens || !tm))
      return fail(HQEKV_E_ARG, "cache_reconstruct: segment %d: slab_tokens applies to token-major segments and must be >= n_tokens", k);
    RcSeg &r = tb.seg[m];
    r.data = s.data;
    r.scale = (const half_t *)s.scale;
    r.zero = (const half_t *)s.zero;
    r.idx = s.idx;
    r.out = (half_t *)(is_k ? K : V);
    r.pos_base = s.pos_base;
    r.slab_tokens = s.slab_tokens > 0 ? s.slab_tokens : s.n_tokens;
    r.n_tokens = (int32_t)s.n_tokens;
    r.bits = (int16_t)s.bits;
    r.kind = (int16_t)((tm ? 1 : 0) | (s.bits == 1 && (s.layout & 3) == HQEKV_LAYOUT_NORMAL1 ? 2 : 0));
    tb.begin[m++] = (int32_t)tiles;
    tiles += (s.n_tokens + RC_TOK - 1) / RC_TOK;
  }
  for (int k = m; k < RC_SEGS; ++k) tb.begin[k] = 0x7fffffff;
  // More tiles than grid.y holds (4.2 million tokens on both sides together): another launch, whose begins are counted from
  // its first tile.  (At most 16 segments of 2^30 tokens: fewer than 2^28 tiles.)
  for (int64_t first = 0; first < tiles; first += RC_GRID_Y) {
    hipLaunchKernelGGL(cache_reconstruct_kernel, dim3((unsigned)BH, (unsigned)std::min(tiles - first, RC_GRID_Y)), dim3(RC_THREADS), 0,
                       (hipStream_t)stream, tb, (int)D, T);
    const int rc = check_launch("cache_reconstruct_kernel");
    if (rc) return rc;
    for (int k = 0; k < m; ++k) tb.begin[k] -= (int32_t)RC_GRID_Y;
  }
  return HQEKV_OK;
}
