// The prompt side of the attention layer (model/llama_hqe.py:141-188): causal attention over the whole prompt, and the
// probabilities of its last rows, which seed the importance ring.  The reference calls flash-attention for the first
// and a dense matmul + softmax over the last 20 query rows for the second; here both are matrix-core kernels for
// head_dim 128 in fp16 with fp32 accumulation, reading K and V once per query head through the caches (the query
// heads of one KV head are neighbours in the grid), without `repeat_kv` copies.
//
// Both kernels compute S^T = K . Q^T -- keys along M, queries along N of v_mfma_f32_32x32x16_f16 -- so that a lane
// owns ONE query (column lane % 32): the running maximum, the sum and the rescaling of the output are per-lane
// scalars, and the exponentials a lane holds (keys 8 g + 4 (lane / 32) + j of a 32-key tile, g = 0..3, j = 0..3) are
// already laid out as the B operand of the second product, O^T = V^T . P^T.  That product needs, per lane, eight
// KEYS of one channel (4 h + j and 8 + 4 h + j of a 16-key step, for lane half h): V stays row-major in LDS and the
// operand comes out of two transposing reads (ds_read_b64_tr_b16: a group of 16 lanes names four key rows x 32 bytes,
// every lane receives four consecutive keys of one channel).
#include "common.h"

namespace hq {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef float f16_t __attribute__((ext_vector_type(16)));
typedef __fp16 h4raw_t __attribute__((__vector_size__(4 * sizeof(__fp16))));
typedef __attribute__((address_space(3))) h4raw_t lds_h4_t;

constexpr int PA_D = 128;
constexpr int PA_WAVES = 4;
constexpr int PA_THREADS = 64 * PA_WAVES;
constexpr int PA_BC = 32;              // keys per score tile
constexpr float PA_SLACK = 8.f;        // powers of two
// (powers of two, by the keys that a row block walks; the reason beside its use)
__device__ __forceinline__ int pa_share(int keys) {
  const int lg = 32 - __builtin_clz(keys);
  return keys <= 8192 ? max(5, lg - 7) : lg - 6;
}
// How the four waves of a workgroup share its work, and how many keys a wave takes at a time.
// <1, 1>: 32 query rows each, 128 per workgroup, every wave walks all key tiles (154 registers, 32 KB of LDS: three
// workgroups per CU).  For long prompts, which are bound by the chip's power: no order of the same instructions is faster.
// <1, 2>: the same with 64 keys per step, two workgroups per CU.  A short prompt waits for its longest walk: a lone wave needs
// 0.63 us for 32 keys and 1.15 us for 64 (one barrier, one maximum across the lane halves, one test of the rescale; the second
// tile's products run beside the first one's exponentials).
// <2, 1>: the two waves of 32 query rows deal the key tiles among themselves and merge their maxima, sums and outputs at the
// end: walks of half the length in twice as many workgroups.  A step stages two tiles, so LDS holds two workgroups per CU.
template <int KS_, int NB_, bool REVERSED_>
struct PaShape {
  static constexpr bool REVERSED = REVERSED_;   // the second 256 workgroups come in the opposite order
  static constexpr int KS = KS_, NB = NB_, WGS = KS_ * NB_ == 1 ? 3 : 2;
  static constexpr int ROWS = 128 / KS;            // query rows per workgroup
  static constexpr int STEP = PA_BC * NB * KS;     // keys staged per step
  static constexpr int TILE = STEP * PA_D;         // fp16 elements of one staged K (or V) step
};

struct PromptArgs {
  const half_t *q, *k, *v;
  half_t *out;
  int64_t q_b, q_h, q_t;   // strides in elements; the channel stride is 1
  int64_t k_b, k_h, k_t;
  int64_t v_b, v_h, v_t;
  int64_t o_b, o_h, o_t;
  int32_t Hq, Hkv, T;
  int32_t BH, by_xcd;      // B * Hq; by_xcd: B * Hkv is a multiple of 8
  float scale;
};

// A tile of keys goes from memory to LDS without passing through registers (`buffer_load_dwordx4 ... lds`: lane l's
// 16 bytes land at M0 + 16 l, so one wave instruction fills four 256-byte rows).  K and V are both row-major in LDS,
// [key][128 channels], unpadded; banks are spread by a swizzle of the 16-byte pieces inside a row, applied on the
// memory side: the lane that fills piece slot c of a row fetches piece c ^ (row % 16) of K, c ^ 4 (row % 4) of V.
// These loads are inline asm (the compiler makes every LDS access after the builtin form wait for all of them), so the
// wait -- vmcnt(0), once per tile, right before the barrier -- is explicit.
typedef int desc_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ desc_t make_desc(const void *base, uint32_t bytes) {   // `base` and `bytes` wave-uniform
  const uint64_t a = (uint64_t)(uintptr_t)base;
  desc_t d;
  d.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  d.y = __builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu));
  d.z = __builtin_amdgcn_readfirstlane((int)bytes);
  d.w = 0x00020000;
  return d;
}
__device__ __forceinline__ uint32_t lds_offset_of(const void *p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char *)p;
}
__device__ __forceinline__ void dma_1k(uint32_t lds, desc_t d, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(lds), "v"(voff), "s"(d), "s"(soff) : "memory");
}
__device__ __forceinline__ void wait_all_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
struct PaSource {
  desc_t k, v;
  uint32_t k_lane, v_lane;   // this thread's byte offsets inside a tile (row tid / 16, swizzled piece)
  uint32_t k_row, v_row;     // bytes between two keys
};
// rows tid / 16 + 16 i of the step; wave w's instruction i fills rows 16 i + 4 w .. + 3
template <int KEYS>
__device__ __forceinline__ void pa_tile_dma(const PaSource &src, int k0, const half_t *ks, const half_t *vs, int w) {
  const uint32_t kb = lds_offset_of(ks) + (uint32_t)w * 1024u, vb = lds_offset_of(vs) + (uint32_t)w * 1024u;
#pragma unroll
  for (int i = 0; i < KEYS / 16; ++i) {
    dma_1k(kb + 4096u * i, src.k, src.k_lane, (uint32_t)(k0 + 16 * i) * src.k_row);
    dma_1k(vb + 4096u * i, src.v, src.v_lane, (uint32_t)(k0 + 16 * i) * src.v_row);
  }
}

// S^T of one key tile for the wave's 32 queries: 16 fp32 values per lane
__device__ __forceinline__ f16_t pa_scores(const half_t *ks, const h8_t (&qreg)[8], int n, int h) {
  f16_t sc = (f16_t)(0.f);
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const h8_t kk = *reinterpret_cast<const h8_t *>(ks + n * PA_D + ((2 * s + h) ^ (n & 15)) * 8);
    sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kk, qreg[s], sc, 0, 0, 0);
  }
  return sc;
}
template <bool CAUSAL, typename S>
__global__ __launch_bounds__(PA_THREADS, S::WGS) void prompt_attn_kernel(PromptArgs a) {
  constexpr int KS = S::KS, NB = S::NB;
  __shared__ __align__(16) half_t tiles[2][2][S::TILE];   // K, V: two steps each
  half_t (&ks_all)[2][S::TILE] = tiles[0];
  half_t (&vs_all)[2][S::TILE] = tiles[1];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int rg = w / KS, sp = w % KS;   // this wave's 32 rows of the workgroup, its share of the key tiles
  // The grid is one-dimensional, longest rows first over ALL heads (a causal walk's length grows with its row: the short
  // ones fill the gaps at the end).  Workgroup i runs on XCD i mod 8: where the KV heads divide evenly among the XCDs,
  // the query heads of a KV head share one and meet in its L2.  With the rows of one head after the other (a head's row
  // blocks dealt to all XCDs): T = 32768 9.35 -> 8.04 ms, 8192 0.73 -> 0.57 ms, 4099 196 -> 165 us (32 heads over 8).
  const int nrep = a.Hq / a.Hkv;
  // Two workgroups per CU: the second 256 come in the opposite order (eight by eight, so that a KV head stays on its XCD), and a
  // CU that began with a long walk is given a short one: T = 2048 54.4 -> 53.2 us, 3500 130 -> 124, 4099 171.6 -> 165.9.
  int item = (int)blockIdx.x;
  if (S::REVERSED && item >> 8 == 1) {
    const int m = min((int)gridDim.x - 256, 256), g = a.by_xcd ? 8 : 1, p = item - 256;
    item = 256 + m - g - p / g * g + p % g;
  }
  const int qi = item / a.BH, slot = item % a.BH;
  const int bh = a.by_xcd ? ((slot / 8 / nrep) * 8 + slot % 8) * nrep + slot / 8 % nrep : slot;
  const int q0 = ((int)gridDim.x / a.BH - 1 - qi) * S::ROWS;
  const int b = bh / a.Hq, hq = bh % a.Hq, hkv = hq / nrep;
  const int T = a.T;
  const half_t *qp = a.q + b * a.q_b + hq * a.q_h;
  const half_t *kp = a.k + b * a.k_b + hkv * a.k_h;
  const half_t *vp = a.v + b * a.v_b + hkv * a.v_h;
  const int my_q = q0 + 32 * rg + n;
  // the lane's query row: 8 steps of 16 channels, of which it supplies 8 (by lane half)
  h8_t qreg[8];
  {
    const half_t *qr = qp + (int64_t)min(my_q, T - 1) * a.q_t + 8 * h;
#pragma unroll
    for (int s = 0; s < 8; ++s) qreg[s] = *reinterpret_cast<const h8_t *>(qr + 16 * s);
  }
  f16_t o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = (f16_t)(0.f);
  float m = -INFINITY, limit = -INFINITY, lsum = 0.f;
  const float sl2 = a.scale * 1.4426950408889634f;
  const int kend = CAUSAL ? min(T, q0 + S::ROWS) : T;
  const int n_steps = (kend + S::STEP - 1) / S::STEP, share = pa_share(kend);
  PaSource src;
  src.k = make_desc(kp, (uint32_t)((int64_t)T * a.k_t * 2));   // (below 4 GiB: checked by the host)
  src.v = make_desc(vp, (uint32_t)((int64_t)T * a.v_t * 2));
  src.k_row = (uint32_t)a.k_t * 2u;
  src.v_row = (uint32_t)a.v_t * 2u;
  {
    const uint32_t row = threadIdx.x >> 4, slot16 = threadIdx.x & 15;
    src.k_lane = row * src.k_row + ((slot16 ^ (row & 15)) * 16u);
    src.v_lane = row * src.v_row + ((slot16 ^ (4 * (row & 3))) * 16u);
  }
  // Two steps' tiles in LDS, one barrier per step: iteration j waits for its own requests of step j (made an iteration
  // ago), passes the barrier -- now every wave's part of step j is there and every wave has finished step j - 1 --
  // requests step j + 1 into the buffer that step j - 1 was read from, and works on its tile of step j.
  // where this lane points the transposing reads of V: lane r of a group of 16 names key row 4h + r / 4 of a step and
  // the 8 bytes of channels 32 dt + 16 (n / 16) + 4 (r % 4) ..; the row's pieces are swizzled by 4 (row % 4) = 4 (r / 4)
  int v_off[4];
  {
    const int r = lane & 15, key = 4 * h + (r >> 2);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      const int piece = 4 * dt + 2 * (n >> 4) + ((r & 3) >> 1);
      v_off[dt] = key * PA_D + ((piece ^ (4 * (r >> 2))) * 8) + 4 * (r & 1);
    }
  }
  // (rows past the end of the prompt are outside the buffer descriptors: whatever such a row holds in LDS -- zeros from
  // this fill or an older tile's finite values -- meets an exponential that is exactly zero)
  if (n_steps * S::STEP > T) {
#pragma unroll
    for (int i = 0; i < 4 * KS * NB; ++i) *reinterpret_cast<uint4 *>(&vs_all[0][0] + (threadIdx.x + PA_THREADS * i) * 8) = make_uint4(0, 0, 0, 0);
    __syncthreads();
  }
  const int odd = n_steps & 1;
  pa_tile_dma<S::STEP>(src, 0, ks_all[odd], vs_all[odd], w);   // (a step past the last one is fetched and never used)
  // The query is waited for here, with the first step.  Left to its first use, the compiler waits for it inside the loop, by a
  // count that knows nothing of the requests above: every other step then waited for the one it had just asked for.
#pragma unroll
  for (int s = 0; s < 8; ++s) asm volatile("" : "+v"(qreg[s]));
  auto step = [&](int j, const half_t *ks, const half_t *vs, half_t *ks_nxt, half_t *vs_nxt) {
    const int k0 = j * S::STEP + sp * PA_BC * NB;
    wait_all_loads();   // this wave's part of step j, requested an iteration ago
    __syncthreads();
    pa_tile_dma<S::STEP>(src, (j + 1) * S::STEP, ks_nxt, vs_nxt, w);   // in flight across the products
    ks += sp * PA_BC * NB * PA_D;
    vs += sp * PA_BC * NB * PA_D;
    // (a tile that lies after every query of this wave is worked through like any other: all its elements are masked,
    // the maximum stays and the exponentials are zeros; skipping it would cost a copy of the accumulators per tile)
    f16_t s[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) s[i] = pa_scores(ks + i * PA_BC * PA_D, qreg, n, h);
    const bool edge = (k0 + PA_BC * NB > T) || (CAUSAL && k0 + PA_BC * NB - 1 > q0 + 32 * rg);   // some element of the tile is masked
    // the running maximum is kept in units of the scaled logit (base-2 exponent); a raw score enters as s * sl2
    if (edge) {   // (uniform per wave; one branch around all selects)
      const int last_key = (CAUSAL ? min(my_q, T - 1) : T - 1) - k0 - 4 * h;   // the last visible key, relative to element r's base
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (32 * i + 8 * (r >> 2) + (r & 3) > last_key) s[i][r] = -INFINITY;
    }
    float raw = -INFINITY;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) raw = fmaxf(raw, s[i][r]);
    // m is what the exponents are taken relative to: the maximum so far, or a little less.  The 64 products of a rescale (and the
    // exchange between the lane halves) are left out while what passes m does so by less than 2^PA_SLACK and holds less than
    // 2^-share of the lane's sum: a maximum's own weight is exactly one and has no rounding error, which shows where it
    // dominates its row -- and in a long walk at a smaller share, since the others are smaller, too (pa_share).  Relative error
    // (2-norm) against 64 bits, 32 heads over 8, N(0, 1): a rescale each time and the sum taken before the rounding to fp16 / this /
    // 2^-4 throughout: T = 1003 2.535e-4 / 2.518 / 2.521, 4099 2.589 / 2.582 / 2.595; <1, 1>: 8192 2.520 / 2.518 / 2.535, 16384 2.357 /
    // 2.353 / 2.370, 32768 2.0737 / 2.0726 / 2.0883; two channels of K ten times as large, 4099 2.357 / 2.347 / 2.352, 32768 2.261 / 2.250 /
    // 2.269.  Time of the three, us, on one card: T = 2048 50.8 / 49.9 / 48.6, 4099 159.3 / 157.6 / 155.5, 8192 553 / 547 / 532, 32768
    // 8175 / 8100 / 7960.  (sl2 > 0; KS = 1: the first tile always holds key 0, which no query masks: m is finite from then on.)
    // Per lane on purpose: a divergent branch keeps the accumulators where they are (inactive lanes must keep their
    // values, so the products are in place under the execution mask, skipped when no lane needs them); a wave-uniform
    // branch made the compiler copy all 64 accumulators per tile.
    raw *= sl2;
    auto bound = [&](int share_of) { return m + fminf(fmaxf((float)(__builtin_amdgcn_frexp_expf(lsum) - share_of), 0.f), PA_SLACK); };
    if constexpr (KS * NB > 1) limit = bound(share);   // (<1, 1>: by the sum at the last rescale, a smaller one)
    const uint64_t over = __builtin_amdgcn_ballot_w64(raw > limit), both = over | over >> 32 | over << 32;   // a query's two lanes agree
    if (both >> lane & 1) {
      const float mx = fmaxf(m, fmaxf(raw, __shfl_xor(raw, 32, 64)));
      const float alpha = __builtin_amdgcn_exp2f(m - mx);   // (the bare instruction: results below 2^-126 may flush to zero)
      lsum *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;
      m = mx;
      if constexpr (KS * NB == 1) limit = bound(share - 1);
    }
    const float base = KS > 1 && m == -INFINITY ? 0.f : m;   // nothing but masked keys so far: exponentials of -inf are zero
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      // What is added up is what is multiplied: exponentials as fp16 numbers, their sum in fp32.  A weight's rounding then
      // cancels against its share of the sum (and two are added per instruction).
      h8_t p[2];
      float part[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int r = 0; r < 8; ++r) p[t][r] = (half_t)__builtin_amdgcn_exp2f(__builtin_fmaf(s[i][8 * t + r], sl2, -base));
        part[t] = 0.f;
#pragma unroll
        for (int r = 0; r < 8; r += 2) part[t] = __builtin_amdgcn_fdot2((half2_t){p[t][r], p[t][r + 1]}, (half2_t){(half_t)1, (half_t)1}, part[t], false);
      }
      lsum += part[0] + part[1];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
          // V^T operand through the transposing LDS read: a group of 16 lanes names four key rows x 32 bytes and each
          // lane receives four consecutive keys of one channel; two reads (keys 4h + j, 8 + 4h + j) make the operand
          const half_t *src_lo = vs + v_off[dt] + (32 * i + 16 * t) * PA_D;
          const h4raw_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h4_t *)(src_lo));
          const h4raw_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h4_t *)(src_lo + 8 * PA_D));
          h8_t av;
          __builtin_memcpy(&av, &lo, 8);
          __builtin_memcpy(reinterpret_cast<char *>(&av) + 8, &hi, 8);
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, p[t], o[dt], 0, 0, 0);
        }
    }
  };
  // two steps per round, so that each half works on fixed buffers; the odd one first (leaving the loop between the two costs
  // copies of the accumulators)
  if (odd) step(0, ks_all[1], vs_all[1], ks_all[0], vs_all[0]);
  for (int j = odd; j < n_steps; j += 2) {
    step(j, ks_all[0], vs_all[0], ks_all[1], vs_all[1]);
    step(j + 1, ks_all[1], vs_all[1], ks_all[0], vs_all[0]);
  }
  wait_all_loads();   // the last request (a step nobody reads) must have landed before this workgroup's LDS can go to another
  lsum += __shfl_xor(lsum, 32, 64);
  constexpr int OWN = 4 / KS;   // of the four 32-channel parts of the output, those that a wave brings together and stores
  if constexpr (KS > 1) {
    // The waves of a row group exchange bounds, sums and outputs through LDS, each for its own channels.  A lane's 16 outputs of
    // a part go to words 64 apart, lanes adjacent: no bank conflicts.
    static_assert(KS == 2 && PA_WAVES / KS * 4096 * 4 + PA_WAVES * 512 <= (int)sizeof(tiles), "one sender per part");
    float *pool_o = reinterpret_cast<float *>(&tiles[0][0][0]) + rg * 4096;
    float2 *pool_ml = reinterpret_cast<float2 *>(reinterpret_cast<float *>(&tiles[0][0][0]) + PA_WAVES / KS * 4096) + rg * KS * 64;
    __syncthreads();   // the tiles are no longer read
    pool_ml[sp * 64 + lane] = make_float2(m, lsum);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      if (dt / OWN != sp) {
#pragma unroll
        for (int i = 0; i < 16; ++i) pool_o[1024 * dt + 64 * i + lane] = o[dt][i];
      }
    __syncthreads();
    const float2 ml = pool_ml[(sp ^ 1) * 64 + lane];
    const float mx = fmaxf(m, ml.x), ca = __builtin_amdgcn_exp2f(m - mx), cb = __builtin_amdgcn_exp2f(ml.x - mx);   // (the first wave's tiles start with key 0: its m is finite)
    lsum = lsum * ca + ml.y * cb;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      if (dt / OWN == sp) {
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] = o[dt][i] * ca + pool_o[1024 * dt + 64 * i + lane] * cb;
      }
  }
  if (my_q < T) {
    const float inv = 1.0f / lsum;
    half_t *orow = a.out + b * a.o_b + hq * a.o_h + (int64_t)my_q * a.o_t;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      if (KS == 1 || dt / OWN == sp) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          h4_t y;
#pragma unroll
          for (int j = 0; j < 4; ++j) y[j] = (half_t)(o[dt][4 * g + j] * inv);
          *reinterpret_cast<h4_t *>(orow + 32 * dt + 8 * g + 4 * h) = y;
        }
      }
  }
}

// ---- probabilities of the last R <= 32 query rows, with the reference's roundings (model/llama_hqe.py:156-168):
// the product rounded to fp16, times the scale rounded to fp16, plus the mask rounded to fp16, floored at the most
// negative fp16, softmax in fp32, rounded to fp16.  One workgroup per (b, query head); its four waves deal the
// 32-key tiles round-robin and walk them twice: maximum and sum, then the probabilities.
struct LastRowsArgs {
  const half_t *q, *k;
  const half_t *mask;   // additive, (B, 1, R, T) with strides, or nullptr: causal
  half_t *probs;        // (B, Hq, R, T) contiguous
  int64_t q_b, q_h, q_t;
  int64_t k_b, k_h, k_t;
  int64_t m_b, m_r;
  int32_t Hq, Hkv, T, R;
  float scale;
  float2 *partial;      // (B * Hq, R, slices) (maximum, sum) of a slice of the keys, or nullptr: one workgroup per head does it all
  int32_t slices;
};

struct __attribute__((packed, aligned(2))) lr_quad_t { uint64_t v; };    // four fp16 at an element's alignment
struct __attribute__((packed, aligned(2))) lr_oct_t { uint64_t v[2]; };  // eight

// One score tile's 16 values per lane, as the reference's fp16 chain leaves them: query column `my_q` (its mask row
// `mrow`, or the causal rule) against keys 32 * tile + 8 (r / 4) + 4 h + r % 4; -inf where no key is visible.
__device__ __forceinline__ void lr_logits(const LastRowsArgs &a, f16_t s, const half_t *mrow, int tile, int h, int my_q, half_t (&x)[16]) {
  const half_t none = (half_t)-INFINITY;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int key = 32 * tile + 8 * (r >> 2) + 4 * h + (r & 3);
    half_t v = (half_t)((float)(half_t)s[r] * a.scale);
    if (mrow) {
      v = (half_t)((float)v + (float)mrow[min(key, a.T - 1)]);
      v = (half_t)fmaxf((float)v, -65504.f);
      x[r] = key < a.T ? v : none;
    } else {
      x[r] = (key < a.T && key <= my_q) ? v : none;
    }
  }
}
__device__ __forceinline__ void lr_load_keys(const half_t *kp, int64_t k_t, int T, int tile, int n, int h, h8_t (&k)[8]) {
  const half_t *kr = kp + (int64_t)min(32 * tile + n, T - 1) * k_t + 8 * h;
#pragma unroll
  for (int st = 0; st < 8; ++st) k[st] = *reinterpret_cast<const h8_t *>(kr + 16 * st);
}
// running (maximum, sum) over one tile
__device__ __forceinline__ void lr_tile_stats(const half_t (&x)[16], float &m, float &l) {
  float mx = m;
#pragma unroll
  for (int r = 0; r < 16; ++r) mx = fmaxf(mx, (float)x[r]);
  if (mx == -INFINITY) return;   // nothing but masked keys so far
  float part = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) part += __expf((float)x[r] - mx);
  l = l * __expf(m - mx) + part;
  m = mx;
}
// over the two halves of every wave, then the waves: afterwards every thread holds column n's pair
// (`at(k)`: 32 pairs of LDS for wave k)
template <int WAVES, typename At>
__device__ __forceinline__ void lr_merge(float &m, float &l, int n, int h, int w, At at) {
  const float mo = __shfl_xor(m, 32, 64), lo = __shfl_xor(l, 32, 64);
  const float mx = fmaxf(m, mo);
  l = (m == -INFINITY ? 0.f : l * __expf(m - mx)) + (mo == -INFINITY ? 0.f : lo * __expf(mo - mx));
  if (h == 0) at(w)[n] = make_float2(mx, l);
  __syncthreads();
  float2 v[WAVES];
#pragma unroll
  for (int k = 0; k < WAVES; ++k) v[k] = at(k)[n];
  m = -INFINITY;
#pragma unroll
  for (int k = 0; k < WAVES; ++k) m = fmaxf(m, v[k].x);
  l = 0.f;
#pragma unroll
  for (int k = 0; k < WAVES; ++k) l += v[k].x == -INFINITY ? 0.f : v[k].y * __expf(v[k].x - m);
}

// Without room for the slices' statistics: one workgroup per (b, query head) walks all keys twice.
__global__ __launch_bounds__(PA_THREADS, 2) void prompt_last_rows_kernel(LastRowsArgs a) {
  __shared__ float2 sh_ml[PA_WAVES][32];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int b = (int)blockIdx.x / a.Hq, hq = (int)blockIdx.x % a.Hq, hkv = hq / (a.Hq / a.Hkv);
  const int T = a.T, R = a.R;
  const half_t *kp = a.k + b * a.k_b + hkv * a.k_h;
  const int row = min(n, R - 1);         // lanes past the last row repeat it and store nothing
  const int my_q = T - R + row;
  h8_t qreg[8];
  {
    const half_t *qr = a.q + b * a.q_b + hq * a.q_h + (int64_t)my_q * a.q_t + 8 * h;
#pragma unroll
    for (int s = 0; s < 8; ++s) qreg[s] = *reinterpret_cast<const h8_t *>(qr + 16 * s);
  }
  const half_t *mrow = a.mask ? a.mask + b * a.m_b + (int64_t)row * a.m_r : nullptr;
  const int n_tiles = (T + 31) / 32;
  auto tile_logits = [&](int tile, half_t (&x)[16]) {
    h8_t k[8];
    lr_load_keys(kp, a.k_t, T, tile, n, h, k);
    f16_t s = (f16_t)(0.f);
#pragma unroll
    for (int st = 0; st < 8; ++st) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(k[st], qreg[st], s, 0, 0, 0);
    lr_logits(a, s, mrow, tile, h, my_q, x);
  };
  float m = -INFINITY, l = 0.f;
  for (int tile = w; tile < n_tiles; tile += PA_WAVES) {
    half_t x[16];
    tile_logits(tile, x);
    lr_tile_stats(x, m, l);
  }
  lr_merge<PA_WAVES>(m, l, n, h, w, [&](int k) { return sh_ml[k]; });
  const float inv = 1.0f / l;
  half_t *prow = a.probs + (((int64_t)b * a.Hq + hq) * R + row) * (int64_t)T;
  for (int tile = w; tile < n_tiles; tile += PA_WAVES) {
    half_t x[16];
    tile_logits(tile, x);
    if (n >= R) continue;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int key = 32 * tile + 8 * g + 4 * h;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (key + j < T) prow[key + j] = (half_t)(__expf((float)x[4 * g + j] - m) * inv);
    }
  }
}

// Short prompts in one launch: the R rows of a KV head's query heads as columns of 32-column tiles, a workgroup per column
// tile, one of its waves per 32 keys; the logits stay in registers until the row's statistics are there.  Bound: one chain --
// K rows -> LDS -> products -> statistics across the waves -> stores -- and, with sixteen waves on a CU, their vector
// instructions (a second tile per wave costs 6 us: 1003 keys 14.6 us against 10.1 in two launches).  K and the query rows are
// fetched whole rows at a time and turned in LDS: as fragments straight from memory, 32 lines per load, a CU's address unit
// alone took 4 us per sixteen tiles.
// (a wave's own LDS traffic in order, without a barrier)
__device__ __forceinline__ void lr_wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ int ls_piece(int row, int piece) { return row * PA_D + ((piece ^ (row & 15)) << 3); }   // 16-byte pieces, in halves
template <int WAVES>
__global__ __launch_bounds__(WAVES * 64, 1) void prompt_last_short_kernel(LastRowsArgs a) {
  __shared__ __align__(16) half_t sh_k[WAVES][32 * PA_D];
  __shared__ __align__(16) half_t sh_q[32 * PA_D];
  __shared__ float2 sh_ml[WAVES][32];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5, r4 = lane >> 4, piece = lane & 15;   // (a load takes four rows)
  const int b = (int)blockIdx.x / a.Hkv, hkv = (int)blockIdx.x % a.Hkv;
  const int T = a.T, R = a.R, nrep = a.Hq / a.Hkv;
  half_t *ks = sh_k[w];
  {
    const half_t *kp = a.k + b * a.k_b + hkv * a.k_h + 8 * piece;
    const half_t *qp = a.q + b * a.q_b + hkv * nrep * a.q_h + 8 * piece;
    h8_t k[8], q[(7 + WAVES) / WAVES];
#pragma unroll
    for (int j = 0; j < 8; ++j) k[j] = *reinterpret_cast<const h8_t *>(kp + (int64_t)min(32 * w + 4 * j + r4, T - 1) * a.k_t);
#pragma unroll
    for (int j = 0; 4 * WAVES * j < 32; ++j) {
      const int c = min(32 * (int)blockIdx.y + ((4 * (WAVES * j + w) + r4) & 31), nrep * R - 1);   // (columns past the last one repeat it)
      q[j] = *reinterpret_cast<const h8_t *>(qp + (c / R) * a.q_h + (int64_t)(T - R + c % R) * a.q_t);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) *reinterpret_cast<h8_t *>(ks + ls_piece(4 * j + r4, piece)) = k[j];
#pragma unroll
    for (int j = 0; 4 * WAVES * j < 32; ++j)
      if (4 * (WAVES * j + w) < 32) *reinterpret_cast<h8_t *>(sh_q + ls_piece(4 * (WAVES * j + w) + r4, piece)) = q[j];
  }
  const int col = 32 * (int)blockIdx.y + n;                    // (query head of the group, row)
  const bool live = col < nrep * R;                            // lanes past the last column store nothing
  const int hq = hkv * nrep + (live ? col : nrep * R - 1) / R, row = (live ? col : nrep * R - 1) % R;
  const half_t *mrow = a.mask ? a.mask + b * a.m_b + (int64_t)row * a.m_r : nullptr;
  __syncthreads();
  f16_t s = (f16_t)(0.f);
#pragma unroll
  for (int st = 0; st < 8; ++st)
    s = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const h8_t *>(ks + ls_piece(n, 2 * st + h)),
                                               *reinterpret_cast<const h8_t *>(sh_q + ls_piece(n, 2 * st + h)), s, 0, 0, 0);
  half_t x[16];
  float m = -INFINITY, l = 0.f;
  lr_logits(a, s, mrow, w, h, T - R + row, x);   // (a tile past the last one: no key is visible)
  lr_tile_stats(x, m, l);
  lr_merge<WAVES>(m, l, n, h, w, [&](int k) { return sh_ml[k]; });
  if (!live) return;
  const float inv = 1.0f / l;
  half_t *prow = a.probs + (((int64_t)b * a.Hq + hq) * R + row) * (int64_t)T;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int key = 32 * w + 8 * g + 4 * h;
    half_t p[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) p[j] = (half_t)(__expf((float)x[4 * g + j] - m) * inv);
    if (key + 3 < T) {
      lr_quad_t y;
      __builtin_memcpy(&y, p, 8);
      *reinterpret_cast<lr_quad_t *>(prow + key) = y;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (key + j < T) prow[key + j] = p[j];
    }
  }
}

// With room for the slices' statistics and many keys, two launches.  Bound: HBM (K once, the rows' probabilities twice through the memory-side cache).
// prompt_last_logits_kernel: the R rows of all query heads of a KV head lie side by side as columns of 32-column tiles
// (4 heads x 20 rows: three tiles instead of four that are 3/8 empty); a workgroup takes one column tile and one slice of
// the keys, leaves the logits where the probabilities will be -- four keys of a row per 8-byte store -- and the slice's
// (maximum, sum) per row.  prompt_last_probs_kernel turns rows of logits into probabilities, 16 bytes per lane.  Walking
// the keys a second time instead of the stored logits, with slices of 2048 keys and more: 38.8 us at T = 1003 (one slice),
// 175 us at T = 32768 (32 heads over 8); now 9 us and 53 us.  K and the query rows are fetched whole rows at a time and turned in
// LDS, in a wave's own corner: as fragments straight from memory, 32 lines per load, T = 4099 19.0 us against 15.4, B = 2 29.0 /
// 22.3, 8192 27.9 / 21.0, 32768 65.9 / 52.6.
__global__ __launch_bounds__(PA_THREADS, 3) void prompt_last_logits_kernel(LastRowsArgs a) {
  __shared__ __align__(16) half_t sh_k[PA_WAVES][32 * PA_D];
  __shared__ __align__(16) half_t sh_q[32 * PA_D];
  __shared__ float2 sh_ml[PA_WAVES][32];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5, r4 = lane >> 4, piece = lane & 15;   // (a load takes four rows)
  const int b = (int)blockIdx.x / a.Hkv, hkv = (int)blockIdx.x % a.Hkv;
  const int T = a.T, R = a.R, nrep = a.Hq / a.Hkv;
  const int all_tiles = (T + 31) / 32, per_slice = (all_tiles + a.slices - 1) / a.slices;
  const int tile0 = (int)blockIdx.y * per_slice, n_tiles = min(all_tiles, tile0 + per_slice);
  const half_t *kp = a.k + b * a.k_b + hkv * a.k_h + 8 * piece;
  half_t *ks = sh_k[w];
  h8_t k[8];
  auto fetch = [&](int tile) {   // (rows past the last one repeat it)
#pragma unroll
    for (int j = 0; j < 8; ++j) k[j] = *reinterpret_cast<const h8_t *>(kp + (int64_t)min(32 * tile + 4 * j + r4, T - 1) * a.k_t);
  };
  fetch(min(tile0 + w, all_tiles - 1));
  {
    const half_t *qp = a.q + b * a.q_b + hkv * nrep * a.q_h + 8 * piece;
    h8_t q[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c = min(32 * (int)blockIdx.z + 4 * (PA_WAVES * j + w) + r4, nrep * R - 1);   // (columns past the last one repeat it)
      q[j] = *reinterpret_cast<const h8_t *>(qp + (c / R) * a.q_h + (int64_t)(T - R + c % R) * a.q_t);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) *reinterpret_cast<h8_t *>(sh_q + ls_piece(4 * (PA_WAVES * j + w) + r4, piece)) = q[j];
  }
  const int col = 32 * (int)blockIdx.z + n;                    // (query head of the group, row)
  const bool live = col < nrep * R;                            // lanes past the last column store nothing
  const int hq = hkv * nrep + (live ? col : nrep * R - 1) / R, row = (live ? col : nrep * R - 1) % R, my_q = T - R + row;
  const half_t *mrow = a.mask ? a.mask + b * a.m_b + (int64_t)row * a.m_r : nullptr;
  half_t *prow = a.probs + (((int64_t)b * a.Hq + hq) * R + row) * (int64_t)T;
  float m = -INFINITY, l = 0.f;
  __syncthreads();
  h8_t qreg[8];
#pragma unroll
  for (int st = 0; st < 8; ++st) qreg[st] = *reinterpret_cast<const h8_t *>(sh_q + ls_piece(n, 2 * st + h));
#pragma unroll 1
  for (int tile = tile0 + w; tile < n_tiles; tile += PA_WAVES) {
#pragma unroll
    for (int j = 0; j < 8; ++j) *reinterpret_cast<h8_t *>(ks + ls_piece(4 * j + r4, piece)) = k[j];
    fetch(min(tile + PA_WAVES, all_tiles - 1));   // (past the last one: read, not used)
    lr_wave_fence();   // (a wave's own corner: no other wave waits for it)
    f16_t s = (f16_t)(0.f);
#pragma unroll
    for (int st = 0; st < 8; ++st)
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const h8_t *>(ks + ls_piece(n, 2 * st + h)), qreg[st], s, 0, 0, 0);
    lr_wave_fence();
    half_t x[16];
    lr_logits(a, s, mrow, tile, h, my_q, x);
    lr_tile_stats(x, m, l);
    if (live) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int key = 32 * tile + 8 * g + 4 * h;
        if (key + 3 < T) {
          lr_quad_t y;
          __builtin_memcpy(&y, x + 4 * g, 8);
          *reinterpret_cast<lr_quad_t *>(prow + key) = y;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (key + j < T) prow[key + j] = x[4 * g + j];
        }
      }
    }
  }
  lr_merge<PA_WAVES>(m, l, n, h, w, [&](int k) { return sh_ml[k]; });
  if (threadIdx.x < 32 && live) a.partial[((int64_t)b * a.Hq + hq) * R * a.slices + (int64_t)row * a.slices + blockIdx.y] = make_float2(m, l);
}

// The same in one launch where a slice is one tile for each wave: the logits stay in registers, and a workgroup takes the rows'
// statistics from the records that its slices' workgroups leave beside the launch's number (as in decode_step.hip: nothing has
// to be cleared, memory without this number is not ready).  A workgroup that has looked `patience` times leaves every record of
// its column tile itself -- the same instructions on the same operands, hence the same bits -- so that nobody depends on being
// scheduled beside others; workgroups that wait for one another are neighbours in the grid, within 8 * 48 of each other.  The same
// bits as in two launches, too: slices, tiles and sums are theirs.
// Bound: one chain of 6 us at 1003 keys (8.3 in two launches) -- entry, K and query rows, products, statistics across the waves,
// records written and seen, probabilities -- and for longer prompts what its looks read past the L2.  The records of 32 columns
// lie side by side: one store per workgroup, one load per thread and eight slices (rows' records apart, a slice per lane: 8.1 us
// at 1003 keys, 24.5 instead of 12.2 at 4099).  A longer sleep between looks costs 0.3 us and more at 1003 keys and gains nothing.
struct LastOnceArgs {
  u32x4 *records;       // (B * Hkv, column tiles, slices, 32): (maximum, number, sum, number)
  uint32_t lo, hi;      // the launch's number
  int32_t patience;
  int32_t near;         // slabs side by side in the grid, then slices
};
// A wave's corner of LDS: its keys, then statistics (40 KB in all: four workgroups per CU).
union LastOnceCorner {
  half_t __attribute__((aligned(16))) k[32 * PA_D];
  struct {
    float2 wave[32], row[8];   // of its tile; of columns 8 w ... + 7, (maximum, 1 / sum)
    int seen;
  } after;
  __device__ LastOnceCorner() {}
};
template <int G>   // up to 8 G slices
__global__ __launch_bounds__(PA_THREADS, 4) void prompt_last_once_kernel(LastRowsArgs a, LastOnceArgs o) {
  __shared__ LastOnceCorner corner[PA_WAVES];
  __shared__ __align__(16) half_t sh_q[32 * PA_D];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5, r4 = lane >> 4, piece = lane & 15;   // (a load takes four rows)
  const int own = (int)blockIdx.x / o.near, bh = (int)blockIdx.y * o.near + (int)blockIdx.x % o.near;
  const int b = bh / a.Hkv, hkv = bh % a.Hkv;
  const int T = a.T, R = a.R, nrep = a.Hq / a.Hkv, slices = a.slices;
  const int all_tiles = (T + 31) / 32, per_slice = (all_tiles + slices - 1) / slices;   // (up to PA_WAVES)
  const int col0 = 32 * (int)blockIdx.z, columns = nrep * R;
  const half_t *kp = a.k + b * a.k_b + hkv * a.k_h + 8 * piece;
  const int64_t row0 = ((int64_t)b * a.Hq + hkv * nrep) * R;   // column c of the KV head is row row0 + c of (B * Hq, R)
  const rsrc_t records = make_rsrc(o.records + (int64_t)(bh * (int)gridDim.z + (int)blockIdx.z) * slices * 32, (uint32_t)slices * 512u);
  half_t *ks = corner[w].k;
  const int col = min(col0 + n, columns - 1);                  // (query head of the group, row); columns past the last one repeat it
  const bool live = col0 + n < columns;                        // and store nothing
  const int row = col % R;
  const half_t *mrow = a.mask ? a.mask + b * a.m_b + (int64_t)row * a.m_r : nullptr;
  bool q_there = false;
  half_t x[16];
  auto slice = [&](int i, half_t (&y)[16]) {   // the logits of this wave's tile of a slice; the slice's record
    const int tile = w < per_slice ? i * per_slice + w : all_tiles;   // (past the last one: no key is visible)
    h8_t k[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) k[j] = *reinterpret_cast<const h8_t *>(kp + (int64_t)min(32 * tile + 4 * j + r4, T - 1) * a.k_t);
    if (!q_there) {
      const half_t *qp = a.q + b * a.q_b + hkv * nrep * a.q_h + 8 * piece;
      h8_t q[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int c = min(col0 + 4 * (PA_WAVES * j + w) + r4, columns - 1);
        q[j] = *reinterpret_cast<const h8_t *>(qp + (c / R) * a.q_h + (int64_t)(T - R + c % R) * a.q_t);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) *reinterpret_cast<h8_t *>(sh_q + ls_piece(4 * (PA_WAVES * j + w) + r4, piece)) = q[j];
      q_there = true;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) *reinterpret_cast<h8_t *>(ks + ls_piece(4 * j + r4, piece)) = k[j];
    __syncthreads();
    f16_t s = (f16_t)(0.f);
#pragma unroll
    for (int st = 0; st < 8; ++st)
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const h8_t *>(ks + ls_piece(n, 2 * st + h)),
                                                 *reinterpret_cast<const h8_t *>(sh_q + ls_piece(n, 2 * st + h)), s, 0, 0, 0);
    float m = -INFINITY, l = 0.f;
    lr_logits(a, s, mrow, tile, h, T - R + row, y);
    lr_tile_stats(y, m, l);
    lr_merge<PA_WAVES>(m, l, n, h, w, [&](int k) { return corner[k].after.wave; });
    if (threadIdx.x < 32)
      __builtin_amdgcn_raw_buffer_store_b128((u32x4){__builtin_bit_cast(uint32_t, m), o.lo, __builtin_bit_cast(uint32_t, l), o.hi}, records, (32 * i + n) * 16, 0,
                                             HQ_THROUGH);
  };
  // Eight lanes merge a column's records, in the order of wave_sum, which prompt_last_probs_kernel takes.
  auto merge = [&](int patience) {
    const int c = (int)threadIdx.x >> 3, l8 = lane & 7;
    u32x4 rec[G];
    for (int look = 0;; ++look) {
      bool ready = true;
#pragma unroll
      for (int g = 0; g < G; ++g)
        if (g == 0 || 8 * g < slices)
          rec[g] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(records, (32 * min(l8 + 8 * g, slices - 1) + c) * 16, 0, HQ_THROUGH));
#pragma unroll
      for (int g = 0; g < G; ++g)
        if (g == 0 || 8 * g < slices) ready = ready && rec[g][1] == o.lo && rec[g][3] == o.hi;
      if (__builtin_amdgcn_ballot_w64(!ready) == 0) break;
      if (look >= patience) return false;
      __builtin_amdgcn_s_sleep(2);
    }
    float vm[G], m = -INFINITY, part[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const uint32_t rm = g == 0 || 8 * g < slices ? rec[g][0] : 0u;   // (bit_cast of a vector's element reads its first)
      vm[g] = l8 + 8 * g < slices ? __builtin_bit_cast(float, rm) : -INFINITY;
      m = fmaxf(m, vm[g]);
    }
#pragma unroll
    for (int k = 1; k < 8; k *= 2) m = fmaxf(m, __shfl_xor(m, k, 64));
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (g && 8 * g >= slices) break;
      const uint32_t rl = rec[g][2];
      part[g] = vm[g] == -INFINITY ? 0.f : __builtin_bit_cast(float, rl) * __expf(vm[g] - m);
#pragma unroll
      for (int k = 1; k < 8; k *= 2) part[g] += __shfl_xor(part[g], k, 64);
    }
    const float l = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
    if (l8 == 0) corner[w].after.row[lane >> 3] = make_float2(m, 1.0f / l);
    return true;
  };
  slice(own, x);
  {
    const bool there = merge(o.patience);
    if (lane == 0) corner[w].after.seen = there;
  }
  __syncthreads();
  if (!(corner[0].after.seen && corner[1].after.seen && corner[2].after.seen && corner[3].after.seen)) {
#pragma unroll 1
    for (int i = 0; i < slices; ++i) {
      half_t y[16];
      __syncthreads();   // (the last slice's tiles and statistics have been read)
      slice(i, y);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    merge(0);   // (its own records, in memory by now)
    __syncthreads();
  }
  if (!live) return;
  const float m = corner[n >> 3].after.row[n & 7].x, inv = corner[n >> 3].after.row[n & 7].y;
  const int key0 = 32 * (own * per_slice + w);
  if (w >= per_slice) return;
  half_t *prow = a.probs + (row0 + col) * (int64_t)T;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int key = key0 + 8 * g + 4 * h;
    half_t p[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) p[j] = (half_t)(__expf((float)x[4 * g + j] - m) * inv);
    if (key + 3 < T) {
      lr_quad_t y;
      __builtin_memcpy(&y, p, 8);
      *reinterpret_cast<lr_quad_t *>(prow + key) = y;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (key + j < T) prow[key + j] = p[j];
    }
  }
}

constexpr int LR_SPAN = 2048;   // probabilities of one row per workgroup: 256 lanes x 8
__global__ __launch_bounds__(PA_THREADS) void prompt_last_probs_kernel(LastRowsArgs a) {
  __shared__ float sh[2];
  const int lane = threadIdx.x & 63;
  half_t *prow = a.probs + (int64_t)blockIdx.y * a.T;
  const int e0 = (int)blockIdx.x * LR_SPAN + (int)threadIdx.x * 8;
  const bool whole = e0 + 8 <= a.T;
  half_t x[8];
  if (whole) {
    const lr_oct_t v = *reinterpret_cast<const lr_oct_t *>(prow + e0);
    __builtin_memcpy(x, &v, 16);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = e0 + i < a.T ? prow[e0 + i] : (half_t)0;
  }
  if (threadIdx.x < 64) {   // the slices' statistics of this row
    const float2 *ps = a.partial + (int64_t)blockIdx.y * a.slices;
    const float2 v = lane < a.slices ? ps[lane] : make_float2(-INFINITY, 0.f);   // (at most 64 slices)
    const float m = wave_max(v.x);
    const float l = wave_sum(v.x == -INFINITY ? 0.f : v.y * __expf(v.x - m));
    if (lane == 0) {
      sh[0] = m;
      sh[1] = 1.0f / l;
    }
  }
  __syncthreads();
  const float m = sh[0], inv = sh[1];
  half_t y[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) y[i] = (half_t)(__expf((float)x[i] - m) * inv);
  if (whole) {
    lr_oct_t v;
    __builtin_memcpy(&v, y, 16);
    *reinterpret_cast<lr_oct_t *>(prow + e0) = v;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (e0 + i < a.T) prow[e0 + i] = y[i];
  }
}

}  // namespace hq

using namespace hq;

static bool rows_16_byte_aligned(const void *p, int64_t s0, int64_t s1, int64_t s2) {
  return ((uintptr_t)p & 15) == 0 && s0 % 8 == 0 && s1 % 8 == 0 && s2 % 8 == 0;
}

// Which form, by the number of 128-row workgroups, us (the forms compared on one card).  Up to 400 (B = 1 and 32 heads: T up to
// 1600) two waves per row group: 128 (T = 500) 12.2 against 15.3 of <1, 2> and 17.6 of <1, 1>, 256 (1003) 22.1 / 24.4 / 27.5, 384
// (1500) 35.9 / 35.7 / 39.2; at 480 (1800) 49.1 / 44.9 / 49.7.  Up to 1500 64 keys per step: 512 (2048) 50.8 against 56.7 of <1, 1>,
// 672 (28 heads over 4, 3000) 84.8 / 90.9, 1056 (4099) 169.0 / 172.8, 1376 (5500) 279 / 290; beyond it is even or behind: 2048
// (8192) 586 / 584, 4096 (16384) 2255 / 2203.
// The opposite order of the second 256 workgroups, us without / with it: of the 64-key form always, 416 workgroups (T = 1632)
// 39.6 / 38.7, from 512 even; of walks of half the length past two and a half rounds, 608 (1200) 26.2 / 26.0, 728 (777, B = 2, 28
// heads) 25.1 / 23.5, 768 (1500) 36.0 / 35.6.
namespace hq {
PromptForm prompt_form(int64_t T, int64_t BH) {
  const int64_t wgs = (T + 127) / 128 * BH;
  if (wgs <= 400) return PromptForm{2, 1, (T + 63) / 64 * BH > 640};
  return wgs <= 1500 ? PromptForm{1, 2, true} : PromptForm{1, 1, false};
}
}  // namespace hq

extern "C" int hqekv_prompt_attn(const void *q, const int64_t *q_strides, const void *k, const int64_t *k_strides,
                                 const void *v, const int64_t *v_strides, void *out, const int64_t *out_strides, int64_t B,
                                 int64_t Hq, int64_t Hkv, int64_t T, int64_t D, float scale, int causal, void *stream) {
  if (!q || !k || !v || !out || !q_strides || !k_strides || !v_strides || !out_strides)
    return fail(HQEKV_E_ARG, "prompt_attn: null pointer");
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || T <= 0 || Hq % Hkv) return fail(HQEKV_E_ARG, "prompt_attn: need B, T > 0 and Hq %% Hkv == 0");
  if (!(scale > 0.f)) return fail(HQEKV_E_ARG, "prompt_attn: the scale must be positive");
  if (D != PA_D) return fail(HQEKV_E_UNSUPPORTED, "prompt_attn: head_dim %lld (supported: 128)", (long long)D);
  if (T > 0x7fffff00LL || B * Hq > 65535) return fail(HQEKV_E_UNSUPPORTED, "prompt_attn: T or B * Hq too large");
  if (!rows_16_byte_aligned(q, q_strides[0], q_strides[1], q_strides[2]) || !rows_16_byte_aligned(k, k_strides[0], k_strides[1], k_strides[2]) ||
      !rows_16_byte_aligned(v, v_strides[0], v_strides[1], v_strides[2]) || ((uintptr_t)out & 7) || out_strides[0] % 4 || out_strides[1] % 4 || out_strides[2] % 4)
    return fail(HQEKV_E_ALIGN, "prompt_attn: rows of q, k, v must be 16-byte aligned (of out: 8-byte)");
  // (the tiles of K and V are fetched through 32-bit buffer offsets from each head's first row)
  if (T * k_strides[2] * 2 >= (1LL << 32) || T * v_strides[2] * 2 >= (1LL << 32) || k_strides[2] <= 0 || v_strides[2] <= 0)
    return fail(HQEKV_E_UNSUPPORTED, "prompt_attn: a head's K or V rows must span less than 4 GiB (T * token stride * 2 bytes)");
  PromptArgs a;
  a.q = (const half_t *)q; a.k = (const half_t *)k; a.v = (const half_t *)v; a.out = (half_t *)out;
  a.q_b = q_strides[0]; a.q_h = q_strides[1]; a.q_t = q_strides[2];
  a.k_b = k_strides[0]; a.k_h = k_strides[1]; a.k_t = k_strides[2];
  a.v_b = v_strides[0]; a.v_h = v_strides[1]; a.v_t = v_strides[2];
  a.o_b = out_strides[0]; a.o_h = out_strides[1]; a.o_t = out_strides[2];
  a.Hq = (int32_t)Hq; a.Hkv = (int32_t)Hkv; a.T = (int32_t)T; a.scale = scale;
  a.BH = (int32_t)(B * Hq); a.by_xcd = (B * Hkv) % 8 == 0;
  const PromptForm form = prompt_form(T, B * Hq);
  const int64_t rows = form.key_shares == 2 ? 64 : 128, wgs = (T + rows - 1) / rows * B * Hq;
  if (wgs > 0x7fffffffLL) return fail(HQEKV_E_UNSUPPORTED, "prompt_attn: T * B * Hq too large");
#define LAUNCH(C_, KS_, NB_, REV_)                                                                                                                \
  hipLaunchKernelGGL((prompt_attn_kernel<C_, PaShape<KS_, NB_, REV_>>), dim3((unsigned)wgs), dim3(PA_THREADS), 0, (hipStream_t)stream, a)
#define LAUNCH_K(C_)                    \
  if (form.key_shares == 2 && form.reversed) LAUNCH(C_, 2, 1, true); \
  else if (form.key_shares == 2) LAUNCH(C_, 2, 1, false);            \
  else if (form.tiles == 2) LAUNCH(C_, 1, 2, true);                  \
  else LAUNCH(C_, 1, 1, false)
  if (causal) { LAUNCH_K(true); } else { LAUNCH_K(false); }
#undef LAUNCH_K
#undef LAUNCH
  return check_launch("prompt_attn");
}

// Up to 512 keys one launch, a wave per 32 keys.  One launch against two, us (32 heads over 8, 20 rows, host included): 128 keys
// 6.2 / 7.1 (one workgroup of four waves per head then), 256 7.1 / 9.3, 512 8.2 / 9.4; B = 4 500 8.0 / 14.2, B = 64 64 / 126;
// 1003 keys at two tiles per wave 14.6 / 10.1, B = 4 15.3 / 17.6.
// Waves without a key cost time in the exchange of statistics: up to 384 keys on 12 waves against 16, 257 keys 6.7 / 7.6, 384 6.4 /
// 7.5, B = 64 300 43.0 / 47.9.
constexpr int64_t LS_KEYS = 512;
// Beyond, slices of the keys: about 48 (b, query head) slices per column tile's 32 give the chip four to six workgroups per CU;
// a slice keeps a tile for each of its four waves.
static int last_rows_slices(int64_t B, int64_t Hq, int64_t T) {
  int64_t s = (1536 + B * Hq - 1) / (B * Hq);
  const int64_t most = (T + 127) / 128;
  if (s > most) s = most;
  if (s > 64) s = 64;
  if (s < 2) s = 2;
  return T <= LS_KEYS || B * Hq * 32 > 65535 ? 1 : (int)s;
}

// One launch where a slice is a tile per wave, up to 30 000 (workgroup, slice) pairs: each time all of them look, that is 15 MB of
// records past the L2, and by then workgroups that wait keep others from beginning.  Two launches / one, us (20 rows, back to back;
// heads over KV heads, tokens, pairs in thousands): 32/8 600 0.6 7.8 / 5.6, 1003 1.5 8.3 / 5.9, 2048 6 9.6 / 7.4, 3000 14 11.8 / 8.7,
// 4099 26 15.0 / 12.2, 5460 44 16.7 / 17.3, 6144 55 16.2 / 18.5; 32/32 4099 35 16.3 / 18.2; 40/8 4099 35 17.5 / 17.2; 64/64 3000 37
// 19.7 / 20.0; 40/8 3800 29 15.4 / 12.3; B = 2 32/8 1003 3 10.2 / 7.1, 3000 28 16.9 / 14.9; B = 4 1003 6 13.4 / 8.7; B = 8 768 7
// 18.4 / 12.5.
constexpr int LO_SLICES = 48, LO_PAIRS = 30000;
static bool last_rows_once(int64_t T, int sl) { return sl > 1 && sl <= LO_SLICES && (T + 31) / 32 <= (int64_t)PA_WAVES * sl; }

extern "C" int64_t hqekv_prompt_last_rows_workspace_bytes(int64_t B, int64_t Hq, int64_t T) {
  if (B <= 0 || Hq <= 0 || T <= 0) return -1;
  const int sl = last_rows_slices(B, Hq, T);
  return sl > 1 ? B * Hq * sl * 32 * (int64_t)(last_rows_once(T, sl) ? sizeof(u32x4) : sizeof(float2)) : 0;
}

static int last_rows(const void *q, const int64_t *q_strides, const void *k, const int64_t *k_strides, const void *mask,
                     const int64_t *mask_strides, void *probs, int64_t B, int64_t Hq, int64_t Hkv, int64_t T, int64_t D, int64_t R, float scale,
                     void *workspace, int64_t workspace_bytes, int patience, void *stream) {
  if (!q || !k || !probs || !q_strides || !k_strides || (mask && !mask_strides)) return fail(HQEKV_E_ARG, "prompt_last_rows: null pointer");
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || T <= 0 || Hq % Hkv || R <= 0 || R > 32 || R > T)
    return fail(HQEKV_E_ARG, "prompt_last_rows: need B > 0, Hq %% Hkv == 0 and 0 < R <= min(32, T)");
  if (D != PA_D) return fail(HQEKV_E_UNSUPPORTED, "prompt_last_rows: head_dim %lld (supported: 128)", (long long)D);
  if (T > 0x7fffff00LL || B * Hq > 0x7fffffffLL) return fail(HQEKV_E_UNSUPPORTED, "prompt_last_rows: T or B * Hq too large");
  if (!rows_16_byte_aligned(q, q_strides[0], q_strides[1], q_strides[2]) || !rows_16_byte_aligned(k, k_strides[0], k_strides[1], k_strides[2]))
    return fail(HQEKV_E_ALIGN, "prompt_last_rows: rows of q and k must be 16-byte aligned");
  LastRowsArgs a;
  a.q = (const half_t *)q; a.k = (const half_t *)k; a.mask = (const half_t *)mask; a.probs = (half_t *)probs;
  a.q_b = q_strides[0]; a.q_h = q_strides[1]; a.q_t = q_strides[2];
  a.k_b = k_strides[0]; a.k_h = k_strides[1]; a.k_t = k_strides[2];
  a.m_b = mask ? mask_strides[0] : 0; a.m_r = mask ? mask_strides[1] : 0;
  a.Hq = (int32_t)Hq; a.Hkv = (int32_t)Hkv; a.T = (int32_t)T; a.R = (int32_t)R; a.scale = scale;
  const int64_t columns = (Hq / Hkv * R + 31) / 32;
  if (T <= LS_KEYS && B * Hkv <= 0x7fffffffLL && columns <= 65535) {
    const dim3 grid((unsigned)(B * Hkv), (unsigned)columns);
    a.partial = nullptr;
    a.slices = 1;
#define LAUNCH(W_) hipLaunchKernelGGL(prompt_last_short_kernel<W_>, grid, dim3(W_ * 64), 0, (hipStream_t)stream, a)
    if (T <= 64) LAUNCH(2);
    else if (T <= 128) LAUNCH(4);
    else if (T <= 256) LAUNCH(8);
    else if (T <= 384) LAUNCH(12);
    else LAUNCH(16);
#undef LAUNCH
    return check_launch("prompt_last_rows");
  }
  // the keys in slices when the caller brought room for the slices' statistics; else one workgroup per head
  const int sl = last_rows_slices(B, Hq, T);
  const int64_t need = B * Hq * sl * 32 * (int64_t)sizeof(float2);
  if (sl > 1 && workspace && workspace_bytes >= need) {
    if ((uintptr_t)workspace & 7) return fail(HQEKV_E_ALIGN, "prompt_last_rows: workspace not 8-byte aligned");
    a.slices = sl;
    const dim3 grid((unsigned)(B * Hkv), (unsigned)sl, (unsigned)columns);
    bool once = last_rows_once(T, sl) && B * Hkv * columns * sl * sl <= LO_PAIRS && patience >= 0 && workspace_bytes >= 2 * need &&
                ((uintptr_t)workspace & 15) == 0;
    if (once) {   // (a captured launch would bear the same number in every replay)
      hipStreamCaptureStatus capture = hipStreamCaptureStatusActive;
      once = hipStreamIsCapturing((hipStream_t)stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone;
    }
    if (once) {
      a.partial = nullptr;
      const int near = B * Hkv % 8 ? 1 : 8;
      const dim3 by_slice((unsigned)(sl * near), (unsigned)(B * Hkv / near), (unsigned)columns);
      const uint64_t number = launch_number();
      const LastOnceArgs o{(u32x4 *)workspace, (uint32_t)number, (uint32_t)(number >> 32), patience, near};
#define LAUNCH(G_) hipLaunchKernelGGL(prompt_last_once_kernel<G_>, by_slice, dim3(PA_THREADS), 0, (hipStream_t)stream, a, o)
      if (sl <= 8) LAUNCH(1);
      else if (sl <= 16) LAUNCH(2);
      else if (sl <= 24) LAUNCH(3);
      else LAUNCH(6);
#undef LAUNCH
      return check_launch("prompt_last_rows");
    }
    a.partial = (float2 *)workspace;
    hipLaunchKernelGGL(prompt_last_logits_kernel, grid, dim3(PA_THREADS), 0, (hipStream_t)stream, a);
    hipLaunchKernelGGL(prompt_last_probs_kernel, dim3((unsigned)((T + LR_SPAN - 1) / LR_SPAN), (unsigned)(B * Hq * R)), dim3(PA_THREADS), 0,
                       (hipStream_t)stream, a);
  } else {
    a.partial = nullptr;
    a.slices = 1;
    hipLaunchKernelGGL(prompt_last_rows_kernel, dim3((unsigned)(B * Hq)), dim3(PA_THREADS), 0, (hipStream_t)stream, a);
  }
  return check_launch("prompt_last_rows");
}

extern "C" int hqekv_prompt_last_rows(const void *q, const int64_t *q_strides, const void *k, const int64_t *k_strides,
                                      const void *mask, const int64_t *mask_strides, void *probs, int64_t B, int64_t Hq,
                                      int64_t Hkv, int64_t T, int64_t D, int64_t R, float scale, void *workspace,
                                      int64_t workspace_bytes, void *stream) {
  return last_rows(q, q_strides, k, k_strides, mask, mask_strides, probs, B, Hq, Hkv, T, D, R, scale, workspace, workspace_bytes, STEP_PATIENCE, stream);
}
extern "C" int hqekv_selftest_last_rows(const void *q, const int64_t *q_strides, const void *k, const int64_t *k_strides,
                                        const void *mask, const int64_t *mask_strides, void *probs, int64_t B, int64_t Hq,
                                        int64_t Hkv, int64_t T, int64_t D, int64_t R, float scale, void *workspace,
                                        int64_t workspace_bytes, int patience, void *stream) {
  return last_rows(q, q_strides, k, k_strides, mask, mask_strides, probs, B, Hq, Hkv, T, D, R, scale, workspace, workspace_bytes, patience, stream);
}
