// What the cache policy ranks blocks by, on the device: a token's importance from the ring of recent attention rows,
// the mean importance of every 32-token block (K ranking), the same weighted with the V token ranges (V ranking), and
// the ranges of new V tokens -- the reference's short chains of torch reductions (model/public_func.py:58-106,217-221;
// quant/hqe_2.py:510-518), one launch each.  The results decide rankings, so every fp16 rounding and every order of
// additions is torch's own on the GPU, measured with order-sensitive inputs and checked against torch on the device:
//   * a sum over the ROWS of a matrix (the 20 ring rows, the batch, the KV heads) is taken by one thread per column
//     with four interleaved fp32 accumulators -- row k goes to accumulator k mod 4 -- added as ((a0 + a1) + a2) + a3;
//   * a sum over 32 CONTIGUOUS values is a balanced tree over adjacent pairs in fp32;
//   * every intermediate tensor is fp16: each step rounds to nearest even; a division by 32 is a multiplication by
//     its (exact) reciprocal; tensor / tensor is the correctly rounded fp32 quotient.
#include <algorithm>

#include "common.h"

#pragma clang fp contract(off)

namespace hq {

constexpr int IMP_THREADS = 256;

template <typename Load>
__device__ __forceinline__ float sum_rows_like_torch(int n_rows, Load &&load) {
  float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
  int r = 0;
  for (; r + 3 < n_rows; r += 4) {
    a0 += load(r);
    a1 += load(r + 1);
    a2 += load(r + 2);
    a3 += load(r + 3);
  }
  if (r < n_rows) a0 += load(r);
  if (r + 1 < n_rows) a1 += load(r + 1);
  if (r + 2 < n_rows) a2 += load(r + 2);
  return ((a0 + a1) + a2) + a3;
}

// lane 0 of every group of 32 lanes ends up with the adjacent-pairs tree sum of the group's values
__device__ __forceinline__ float tree_sum_32(float v) {
#pragma unroll
  for (int off = 1; off < 32; off <<= 1) v += __shfl_down(v, off, 32);
  return v;
}

// importance[c] = rnd16(rnd16(sum of ring column c) / min(rows, n - c)), divided by 32 in place as the ranking helper
// does (model/public_func.py:94-96); block score = sum of the block's 32 divided values.
__global__ __launch_bounds__(IMP_THREADS) void importance_scores_kernel(const half_t *__restrict__ ring, int rows,
                                                                       int64_t max_len, int64_t n, int64_t total,
                                                                       half_t *__restrict__ imp_out,
                                                                       half_t *__restrict__ scores) {
  const int64_t c = (int64_t)blockIdx.x * IMP_THREADS + threadIdx.x;
  float v = 0.f;
  if (c < total) {
    const half_t *col = ring + c;
    const half_t s = (half_t)sum_rows_like_torch(rows, [&](int r) { return (float)col[(int64_t)r * max_len]; });
    const int64_t seen_i = n - c < (int64_t)rows ? n - c : (int64_t)rows;
    const half_t seen = (half_t)(float)seen_i;
    const half_t imp = (half_t)((float)s / (float)seen);
    const half_t d = (half_t)((float)imp * 0.03125f);
    imp_out[c] = d;
    v = (float)d;
  }
  v = tree_sum_32(v);
  if ((threadIdx.x & 31) == 0 && c < total) scores[c >> 5] = (half_t)v;
}

// block scores of x[c] (* w[c]) / 32
__global__ __launch_bounds__(IMP_THREADS) void weighted_scores_kernel(const half_t *__restrict__ x,
                                                                     const half_t *__restrict__ w, int64_t total,
                                                                     half_t *__restrict__ scores) {
  const int64_t c = (int64_t)blockIdx.x * IMP_THREADS + threadIdx.x;
  float v = 0.f;
  if (c < total) {
    half_t t = x[c];
    if (w) t = (half_t)((float)t * (float)w[c]);
    v = (float)(half_t)((float)t * 0.03125f);
  }
  v = tree_sum_32(v);
  if ((threadIdx.x & 31) == 0 && c < total) scores[c >> 5] = (half_t)v;
}

// out[t] = sum over heads of rnd16(sum over batch of rnd16(max_d - min_d)), one workgroup per token
constexpr int RANGE_MAX_ROWS = 1024;
__global__ __launch_bounds__(IMP_THREADS) void token_range_kernel(const half_t *__restrict__ v, int B, int H, int64_t T,
                                                                 int D, int64_t slab_tokens, half_t *__restrict__ out) {
  __shared__ half_t r[RANGE_MAX_ROWS];
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int row = wave; row < B * H; row += IMP_THREADS / 64) {
    const half_t *p = v + ((int64_t)row * slab_tokens + t) * D;
    float mx = -INFINITY, mn = INFINITY;
    for (int d = lane; d < D; d += 64) {
      const float x = (float)p[d];
      mx = fmaxf(mx, x);
      mn = fminf(mn, x);
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      mx = fmaxf(mx, xor_f(mx, m));
      mn = fminf(mn, xor_f(mn, m));
    }
    if (lane == 0) r[row] = (half_t)(mx - mn);   // both are fp16 numbers: the fp32 difference rounded once
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const float s = sum_rows_like_torch(H, [&](int h) {
      if (B == 1) return (float)r[h];
      return (float)(half_t)sum_rows_like_torch(B, [&](int b) { return (float)r[b * H + h]; });
    });
    out[t] = (half_t)s;
  }
}

__device__ __forceinline__ void block_score(half_t x, half_t w, bool weighted, half_t *score) {
  const half_t t = weighted ? (half_t)((float)x * (float)w) : x;
  const float v = tree_sum_32((float)(half_t)((float)t * 0.03125f));
  if ((threadIdx.x & 31) == 0) *score = (half_t)v;
}

// The same for rows of whole 16-byte pieces: 16 lanes per (token, slab) row, 32 tokens per workgroup, so a token's rows
// are a handful of independent 16-byte loads per lane and a reduction stays inside a row of 16 lanes (four DPP steps).
// Bound by latency at 32 tokens (the later compressions: 8.0 us as one workgroup per token with 2-byte loads and trips
// through the LDS crossbar; 4.9 us now) and by HBM at a whole prompt's.  Workgroups past the tokens copy the `n_prev` older
// ranges that the new ones follow.  With `x`, the scores of the blocks go with them (T and n_prev are multiples of 32 then):
// one launch for two of 4.0 and 2.3 us.
constexpr int RANGE_TOK = 32, RANGE_THREADS = 16 * RANGE_TOK;
__global__ __launch_bounds__(RANGE_THREADS) void token_range_rows_kernel(const half_t *__restrict__ v, int B, int H, int64_t T,
                                                                        int D, int64_t slab_tokens, half_t *__restrict__ out,
                                                                        const half_t *__restrict__ prev, int64_t n_prev,
                                                                        int token_blocks, const half_t *__restrict__ x, int weighted,
                                                                        half_t *__restrict__ scores) {
  if ((int)blockIdx.x >= token_blocks) {
    half_t *dst = out - n_prev;
    for (int64_t i = ((int64_t)blockIdx.x - token_blocks) * RANGE_THREADS + threadIdx.x; i < n_prev; i += ((int64_t)gridDim.x - token_blocks) * RANGE_THREADS) {
      const half_t r = prev[i];
      dst[i] = r;
      if (x) block_score(x[i], r, weighted, scores + (i >> 5));   // (whole groups of 32 lanes come this far)
    }
    return;
  }
  extern __shared__ half_t range_rows[];   // B * H rows of RANGE_TOK
  half_t (*r)[RANGE_TOK] = reinterpret_cast<half_t (*)[RANGE_TOK]>(range_rows);
  const int cp = threadIdx.x & 15, tl = threadIdx.x >> 4;
  const int64_t t = (int64_t)blockIdx.x * RANGE_TOK + tl, tc = t < T ? t : T - 1;
  const int rows = B * H;
  constexpr int U = 4;   // rows in flight per lane
  for (int row0 = 0; row0 < rows; row0 += U) {
    float mxs[U], mns[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      mxs[u] = -INFINITY;
      mns[u] = INFINITY;
    }
    for (int d = cp * 8; d < D; d += 128) {
      uint4 raw[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        raw[u] = *reinterpret_cast<const uint4 *>(v + ((int64_t)min(row0 + u, rows - 1) * slab_tokens + tc) * D + d);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        half_t x[8];
        __builtin_memcpy(x, &raw[u], 16);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          mxs[u] = fmaxf(mxs[u], (float)x[i]);
          mns[u] = fminf(mns[u], (float)x[i]);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float mx = mxs[u], mn = mns[u];
      mx = fmaxf(mx, dpp_f<0xB1>(mx));
      mn = fminf(mn, dpp_f<0xB1>(mn));
      mx = fmaxf(mx, dpp_f<0x4E>(mx));
      mn = fminf(mn, dpp_f<0x4E>(mn));
      mx = fmaxf(mx, dpp_f<0x141>(mx));
      mn = fminf(mn, dpp_f<0x141>(mn));
      mx = fmaxf(mx, dpp_f<0x140>(mx));
      mn = fminf(mn, dpp_f<0x140>(mn));
      if (cp == 0 && row0 + u < rows) r[row0 + u][tl] = (half_t)(mx - mn);
    }
  }
  __syncthreads();
  const int64_t to = (int64_t)blockIdx.x * RANGE_TOK + threadIdx.x;
  if (threadIdx.x < RANGE_TOK && to < T) {
    const float s = sum_rows_like_torch(H, [&](int h) {
      if (B == 1) return (float)r[h][threadIdx.x];
      return (float)(half_t)sum_rows_like_torch(B, [&](int b) { return (float)r[b * H + h][threadIdx.x]; });
    });
    out[to] = (half_t)s;
    if (x) block_score(x[n_prev + to], (half_t)s, weighted, scores + ((n_prev + to) >> 5));
  }
}

// Stable descending order of every row of scores, NaN first (what torch.sort(descending=True, stable=True) returns): a
// block's place is the number of blocks that precede it.  A workgroup places 64 blocks; its 16 waves count over a
// sixteenth of all keys each, read from LDS four at a time (every lane the same ones).  A key is the score's order-
// preserving 16 bits above the complement of its index, so no two are equal.  Bound by latency: 2 x 1025 scores take
// 5.8 us (written to host memory), a stack launch and a radix sort of both rows 15 us and their copy to the host 20 more.
constexpr int RANK_THREADS = 1024, RANK_ITEMS = 64, RANK_MAX = 32768;
__device__ __forceinline__ uint32_t rank_key(half_t x, int i) {
  uint32_t u = (uint32_t)__builtin_bit_cast(unsigned short, x);
  if ((u & 0x7fffu) == 0) u = 0;                     // -0 and +0 are equal
  u = (u & 0x8000u) ? ~u & 0xffffu : u | 0x8000u;
  if (x != x) u = 0xffffu;
  return u << 16 | (0xffffu - (uint32_t)i);
}
struct RankRows {
  const half_t *row[HQEKV_MAX_SEGS];
};
__global__ __launch_bounds__(RANK_THREADS) void rank_blocks_kernel(RankRows rows, int n, int32_t *__restrict__ order) {
  extern __shared__ __align__(16) uint32_t keys[];   // n keys, padded with zeros (below every key) to a multiple of 64
  __shared__ int counts[RANK_THREADS / 64][RANK_ITEMS];
  const half_t *row = rows.row[blockIdx.y];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, padded = (n + 63) / 64 * 64;
  for (int i = threadIdx.x; i < padded; i += RANK_THREADS) keys[i] = i < n ? rank_key(row[i], i) : 0u;
  __syncthreads();
  const int i = (int)blockIdx.x * RANK_ITEMS + lane;
  const uint32_t mine = i < n ? keys[i] : 0xffffffffu;
  int c = 0;
  for (int j = 4 * w; j < padded; j += 4 * (RANK_THREADS / 64)) {
    const uint4 k = *reinterpret_cast<const uint4 *>(keys + j);
    c += (k.x > mine ? 1 : 0) + (k.y > mine ? 1 : 0) + (k.z > mine ? 1 : 0) + (k.w > mine ? 1 : 0);
  }
  counts[w][lane] = c;
  __syncthreads();
  if (w == 0 && i < n) {
    int place = 0;
#pragma unroll
    for (int k = 0; k < RANK_THREADS / 64; ++k) place += counts[k][lane];
    order[(int64_t)blockIdx.y * n + place] = i;
  }
}

}  // namespace hq

using namespace hq;

extern "C" int hqekv_importance_scores(const void *ring, int32_t rows, int64_t max_len, int64_t n, int64_t total,
                                       void *importance_out, void *scores_out, void *stream) {
  if (!ring || !importance_out || !scores_out) return fail(HQEKV_E_ARG, "importance_scores: null pointer");
  if (rows <= 0 || total <= 0 || total > n || n > max_len || total % 32)
    return fail(HQEKV_E_ARG, "importance_scores: need 0 < total <= n <= max_len, total a multiple of 32, rows > 0");
  const int64_t blocks = (total + IMP_THREADS - 1) / IMP_THREADS;
  if (blocks > 0x7fffffffLL) return fail(HQEKV_E_UNSUPPORTED, "importance_scores: too many columns");
  hipLaunchKernelGGL(importance_scores_kernel, dim3((unsigned)blocks), dim3(IMP_THREADS), 0, (hipStream_t)stream,
                     (const half_t *)ring, (int)rows, max_len, n, total, (half_t *)importance_out, (half_t *)scores_out);
  return check_launch("importance_scores");
}

extern "C" int hqekv_weighted_block_scores(const void *x, const void *weights, int64_t total, void *scores_out,
                                           void *stream) {
  if (!x || !scores_out) return fail(HQEKV_E_ARG, "weighted_block_scores: null pointer");
  if (total <= 0 || total % 32) return fail(HQEKV_E_ARG, "weighted_block_scores: total must be a positive multiple of 32");
  const int64_t blocks = (total + IMP_THREADS - 1) / IMP_THREADS;
  if (blocks > 0x7fffffffLL) return fail(HQEKV_E_UNSUPPORTED, "weighted_block_scores: too many columns");
  hipLaunchKernelGGL(weighted_scores_kernel, dim3((unsigned)blocks), dim3(IMP_THREADS), 0, (hipStream_t)stream,
                     (const half_t *)x, (const half_t *)weights, total, (half_t *)scores_out);
  return check_launch("weighted_block_scores");
}

static int range_launch(const void *v, int64_t B, int64_t H, int64_t T, int64_t D, int64_t slab_tokens, const void *prev, int64_t n_prev,
                        void *out, const void *x, int weighted, void *scores, void *stream) {
  if (n_prev < 0 || (n_prev > 0 && !prev)) return fail(HQEKV_E_ARG, "token_range: bad older ranges");
  if (!v || !out) return fail(HQEKV_E_ARG, "token_range: null pointer");
  if (B <= 0 || H <= 0 || T <= 0 || D <= 0 || slab_tokens < T)
    return fail(HQEKV_E_ARG, "token_range: empty shape or slab_tokens < T");
  if (B * H > RANGE_MAX_ROWS) return fail(HQEKV_E_UNSUPPORTED, "token_range: B * H = %lld > %d", (long long)(B * H), RANGE_MAX_ROWS);
  if (T > 0x7fffffffLL || D > 0x7fffffffLL) return fail(HQEKV_E_UNSUPPORTED, "token_range: T or D too large");
  if (D % 8 == 0 && ((uintptr_t)v & 15) == 0) {
    const int token_blocks = (int)((T + RANGE_TOK - 1) / RANGE_TOK);
    const int64_t copy_blocks = std::min<int64_t>((n_prev + RANGE_THREADS - 1) / RANGE_THREADS, 1024);
    hipLaunchKernelGGL(token_range_rows_kernel, dim3((unsigned)(token_blocks + copy_blocks)), dim3(RANGE_THREADS),
                       (size_t)(B * H * RANGE_TOK) * sizeof(half_t), (hipStream_t)stream, (const half_t *)v, (int)B, (int)H, T, (int)D, slab_tokens,
                       (half_t *)out + n_prev, (const half_t *)prev, n_prev, token_blocks, (const half_t *)x, weighted, (half_t *)scores);
    return check_launch("token_range");
  }
  if (n_prev > 0 || x) return fail(HQEKV_E_UNSUPPORTED, "token_range_append: rows of 16-byte aligned pieces only");
  hipLaunchKernelGGL(token_range_kernel, dim3((unsigned)T), dim3(IMP_THREADS), 0, (hipStream_t)stream, (const half_t *)v,
                     (int)B, (int)H, T, (int)D, slab_tokens, (half_t *)out);
  return check_launch("token_range");
}

extern "C" int hqekv_token_range_append(const void *v, int64_t B, int64_t H, int64_t T, int64_t D, int64_t slab_tokens,
                                        const void *prev, int64_t n_prev, void *out, void *stream) {
  return range_launch(v, B, H, T, D, slab_tokens, prev, n_prev, out, nullptr, 0, nullptr, stream);
}

extern "C" int hqekv_range_block_scores(const void *v, int64_t B, int64_t H, int64_t T, int64_t D, int64_t slab_tokens, const void *prev,
                                        int64_t n_prev, const void *x, int weighted, void *range_out, void *scores_out, void *stream) {
  if (!x || !scores_out) return fail(HQEKV_E_ARG, "range_block_scores: null pointer");
  if (T % 32 || n_prev % 32) return fail(HQEKV_E_ARG, "range_block_scores: whole blocks of 32 tokens only");
  return range_launch(v, B, H, T, D, slab_tokens, prev, n_prev, range_out, x, weighted, scores_out, stream);
}

extern "C" int hqekv_token_range(const void *v, int64_t B, int64_t H, int64_t T, int64_t D, int64_t slab_tokens,
                                 void *out, void *stream) {
  return hqekv_token_range_append(v, B, H, T, D, slab_tokens, nullptr, 0, out, stream);
}

extern "C" int hqekv_rank_blocks(const void *const *scores, int rows, int64_t n, int32_t *order, void *stream) {
  if (!scores || !order || rows <= 0 || rows > HQEKV_MAX_SEGS || n <= 0) return fail(HQEKV_E_ARG, "rank_blocks: null pointer or bad shape");
  if (n > RANK_MAX) return fail(HQEKV_E_UNSUPPORTED, "rank_blocks: more than %d scores per row", RANK_MAX);
  RankRows rr{};
  for (int r = 0; r < rows; ++r) {
    if (!scores[r]) return fail(HQEKV_E_ARG, "rank_blocks: row %d is null", r);
    rr.row[r] = (const half_t *)scores[r];
  }
  const size_t lds = (size_t)((n + 63) / 64 * 64) * sizeof(uint32_t);
  if (lds > 48 * 1024) {   // beyond the default limit of a launch (128 KB of the CU's 160 at most)
    const hipError_t e = hipFuncSetAttribute((const void *)rank_blocks_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, RANK_MAX * (int)sizeof(uint32_t));
    if (e != hipSuccess) return fail((int)e, "rank_blocks: %s", hipGetErrorString(e));
  }
  hipLaunchKernelGGL(rank_blocks_kernel, dim3((unsigned)((n + RANK_ITEMS - 1) / RANK_ITEMS), (unsigned)rows), dim3(RANK_THREADS), lds,
                     (hipStream_t)stream, rr, (int)n, order);
  return check_launch("rank_blocks_kernel");
}
