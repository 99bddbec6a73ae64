// What the decode-attention kernels share: the segment table, the arguments of the fused softmax, and the dequantiser's
// arithmetic on pairs of codes.
#pragma once

#include <stdlib.h>

#include <type_traits>
#include <utility>

#include "common.h"

#pragma clang fp contract(off)  // the two fp16 roundings of the dequantiser must stay separate


namespace hq {

struct SegDev {
  const void *data;
  const half_t *scale;
  const half_t *zero;
  const int64_t *idx;
  int64_t pos_base;
  int64_t n_tokens;
  int32_t bits;
  int32_t layout;      // HQEKV_LAYOUT_*: 1 = fp16 K stored token-major, 2 = 1-bit normal-quantile coding
  int32_t unit_begin;  // first chunk of this segment in the p.V partial buffer
  int32_t n_units;     // tiles (q.K^T) or chunks (p.V) of this segment
  int64_t slab_tokens; // token rows between two (b, kv head) slabs of a token-major segment (>= n_tokens)
};

struct SegTable {
  SegDev seg[HQEKV_MAX_SEGS];
  int32_t nseg;
  int32_t total_units;
  int32_t max_units;   // the largest n_units of any segment
  int32_t per_unit;    // tiles or blocks per unit of the matrix-core launches (decode_tiles.h); 0 = the older forms
  int32_t begin[HQEKV_MAX_SEGS];  // first grid.y index of every segment (INT32_MAX past nseg): one scalar load finds a workgroup's segment
};

// grid.y enumerates the units of all segments back to back (no idle workgroups): unit u belongs to the last
// segment whose first unit is <= u.  Branch-free on the eight begins, which arrive in one scalar load.
__device__ __forceinline__ int seg_of_unit(const SegTable &tb, int u) {
  int s = -1;
#pragma unroll
  for (int k = 0; k < HQEKV_MAX_SEGS; ++k) s += (u >= tb.begin[k]) ? 1 : 0;
  return s;
}
// begin[s] without a second, dependent load from the argument segment
__device__ __forceinline__ int begin_of_seg(const SegTable &tb, int s) {
  int b = 0;
#pragma unroll
  for (int k = 0; k < HQEKV_MAX_SEGS; ++k) b += (k == s) ? tb.begin[k] : 0;
  return b;
}

// A running maximum starts at SM_FLOOR, below every finite fp16 logit but finite: a logit of -inf (a score beyond fp16's
// range) then adds exp(-inf) = 0 wherever it meets other logits or none, where exp(-inf - -inf) would be NaN.  A row of
// nothing but -inf still sums to zero and becomes NaN, as in torch.
constexpr float SM_FLOOR = -3.0e38f;

// Optional fusion of the softmax into the two GEMV launches (valid when no mask is added and the K
// classes as well as the V classes each cover every position exactly once):
//   q.K^T stores the scaled fp16 logit instead of the raw score and one (max, sum exp) pair per tile and
//   head; p.V turns a logit into its probability while staging it and writes it back for the caller.
// The split-K partials are summed by the LAST p.V workgroup of each (b, kv head) to finish, when there are few
// enough of them; otherwise by a small launch of their own.  Nobody waits for anybody: a workgroup stores its
// partial rows write-through (agent-scope relaxed stores go past the per-XCD L2), waits for the stores to be
// acknowledged, and bumps one relaxed agent-scope counter; whoever reads the final count adds the rows up with
// loads that bypass the L2 as well, in the fixed order of the separate launch.  No release / acquire fences are
// involved: those write back and invalidate the whole L2 on this chip (the step went from 39 to 146 us with them).
struct FuseArgs {
  float2 *stats;       // (B*Hq, n_stat) pairs (m, l); nullptr = unfused
  int32_t n_stat;      // tiles per row of stats = number of q.K^T tiles per (b, kv head)
  float inv_sqrt_d;
  // Folded combine (independent of the softmax fusion): one arrival counter per (b, kv head), zeroed by the q.K^T
  // launch of the same call; nullptr = the split-K partials are summed by a launch of their own.
  uint32_t *arrive;
  half_t *out;         // (B*Hq, D) attention output, written by the last workgroup of each (b, kv head)
  int32_t two_step;    // never fold the bias removal of a code into its multiply (HQEKV_TWO_STEP_DEQUANT)
};
// More than eight query heads per KV head are served in slices of at most eight, one launch each: the launch's NREP
// heads are heads `off` .. `off` + NREP - 1 of the `group` query heads of their KV head (a launch that covers all
// heads: group = NREP, off = 0).  Group and offset ride in the upper half of the kernels' head-count argument,
// hq_slice = Hq | group << 16 | off << 24, and are used without a branch: as two members at the end of FuseArgs, or
// behind a test for "no slices", the kernel's other scalar loads ended up behind a first, dependent one -- half a
// microsecond in every workgroup -- and even one more plain argument moved the launches by a quarter.
// -> first query head (inside its batch row) that a workgroup of KV head `hkv` works on
__device__ __forceinline__ int first_head(int hq_slice, int hkv) { return hkv * ((hq_slice >> 16) & 0xff) + (int)((uint32_t)hq_slice >> 24); }
__host__ __device__ constexpr int hq_with_slice(int Hq, int group, int off) { return Hq | group << 16 | off << 24; }

// What the caller of a decode step does next to the attention (model/llama_hqe.py:131-133, 200), folded into the
// step's last launch: the row of the importance ring -- the probabilities summed over the batch, rounded to fp16,
// then summed over the heads and rounded again (model/public_func.py:243-257: attn_weights.sum(0).sum(0)) -- and
// the copies that append the step's key and value rows to the fp16 residual.
struct StepEpilogue {
  const half_t *weights;   // (B, Hq, Tall) probabilities
  half_t *ring_line;       // (Tall) or nullptr
  int64_t Tall;
  int32_t B, Hq;
  int32_t ring_by;         // threads torch's reduction deals the head rows to for this shape: 1 or 2
  int64_t ring_tokens;     // several rows at once (Tall = rows * ring_tokens, ring_stride columns apart in the store); 0 = one
  int64_t ring_stride;
  int32_t ring_fill_rows;  // rows of the store to zero where nothing else is written
  int32_t app_rows;        // token rows to append per (b, kv head); 0 = none
  int32_t app_row_elems;   // head_dim
  int32_t app_bh;          // B * Hkv
  const half_t *app_src[2];
  half_t *app_dst[2];          // first destination row of slab 0
  int64_t app_src_slab[2];     // elements between two (b, kv head) slabs
  int64_t app_dst_slab[2];
  // a row per (b, kv head) that is quantised on the way (hqekv_step_extra.leave_*); slabs in elements of each array
  int32_t leave_bits, leave_groups;   // groups of 32 per row
  const half_t *leave_src;
  uint32_t *leave_code;
  half_t *leave_scale, *leave_zero;
  int64_t leave_slab, leave_rows;     // elements / destination token rows between two slabs
};

// A workgroup learns its segment and its tile/chunk from its block id with two scalar loads at the top of
// the kernel: the eight unit begins, then the segment's 64-byte entry (a scalar load that misses costs about
// a microsecond; walking the table entry by entry would chain several of them).

// Workgroups are handed to the 8 XCDs round-robin in launch order, and each XCD has its own L2.
// Neighbouring tiles of one (b, kv head) slab share cache lines (a tile's row segment is shorter than a
// line, its scale/zero rows are a quarter of one), so the (b, kv head) index is the FASTEST grid
// dimension: with B*Hkv a multiple of 8, every tile of a slab runs on the same XCD, neighbours meet in
// one L2, and the eight XCDs get equal work.  (Tile-fastest order fetched every line 2x on average.)

// keep every load issued above this point ahead of the arithmetic below it (the scheduler would
// otherwise sink loads next to their uses to save registers, serialising the memory latency)
#define HQ_LOADS_ABOVE()                     \
  do {                                       \
    asm volatile("" ::: "memory");           \
    __builtin_amdgcn_sched_barrier(0);       \
  } while (0)

__device__ __forceinline__ half2_t as_h2(uint32_t u) {
  half2_t h;
  __builtin_memcpy(&h, &u, 4);
  return h;
}
__device__ __forceinline__ uint32_t as_u32(half2_t h) {
  uint32_t u;
  __builtin_memcpy(&u, &h, 4);
  return u;
}
__device__ __forceinline__ half2_t pack_h2(half_t a, half_t b) {
  half2_t h;
  h[0] = a;
  h[1] = b;
  return h;
}

// [lo.byte_k, 0, hi.byte_k, 0]: byte k of two packed words side by side in the 16-bit halves
template <int K>
__device__ __forceinline__ uint32_t byte_pair(uint32_t lo, uint32_t hi) {
  return __builtin_amdgcn_perm(hi, lo, 0x0c040c00u + (uint32_t)K * 0x00010001u);
}
// (lo.half_H, hi.half_H) of two registers holding fp16 pairs
template <int H>
__device__ __forceinline__ half2_t half_pair(uint32_t lo, uint32_t hi) {
  return as_h2(__builtin_amdgcn_perm(hi, lo, H == 0 ? 0x05040100u : 0x07060302u));
}

// Field I (of 8/BITS) of the byte pair `u` as two exact fp16 integers.
template <int BITS, int I>
__device__ __forceinline__ half2_t field_pair(uint32_t u) {
  constexpr int POS = I * BITS;                         // bit position inside the byte
  constexpr uint32_t FMASK = ((1u << BITS) - 1u) << POS;
  constexpr uint32_t MASK = FMASK | (FMASK << 16);
  constexpr uint32_t EXPO = (uint32_t)(10 - POS + 15) << 10;  // fp16 bits of 2^(10-POS)
  constexpr uint32_t MAGIC = EXPO | (EXPO << 16);
  // (u & MASK) | MAGIC in one VALU op; the mask rides in a scalar register, the magic in a vector one
  uint32_t r;
  const uint32_t magic_v = MAGIC;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(u), "s"(MASK), "v"(magic_v));
  const half2_t biased = as_h2(r);                      // 2^(10-POS) + c, exact
  const half2_t bias = as_h2(MAGIC);
  return biased - bias;                                 // c, exact
}

// The same field still carrying its bias: 2^(10-POS) + c.
template <int BITS, int I>
__device__ __forceinline__ half2_t field_pair_biased(uint32_t u) {
  constexpr int POS = I * BITS;
  constexpr uint32_t FMASK = ((1u << BITS) - 1u) << POS;
  constexpr uint32_t MASK = FMASK | (FMASK << 16);
  constexpr uint32_t EXPO = (uint32_t)(10 - POS + 15) << 10;
  constexpr uint32_t MAGIC = EXPO | (EXPO << 16);
  uint32_t r;
  const uint32_t magic_v = MAGIC;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(u), "s"(MASK), "v"(magic_v));
  return as_h2(r);
}
// -2^(10-POS) * s for field I: with it rnd16(c * s) is ONE fused multiply-add on the biased field,
// (2^(10-POS) + c) * s - 2^(10-POS) * s = c * s before the single rounding -- exactly the product the reference
// rounds -- provided 2^(10-POS) * s is itself an fp16 number, i.e. |s| < 64 at POS = 0 (scaling by a power of two
// is exact short of overflow).  Callers take this route only after checking the scales of the whole tile.
template <int BITS, int I>
__device__ __forceinline__ half2_t bias_times_scale(half2_t s2) {
  constexpr _Float16 NB = (_Float16)(-(float)(1 << (10 - I * BITS)));
  return s2 * (half2_t){NB, NB};
}

// the reference dequantiser's two roundings (quant/pack_unpack.py:331-332) on a pair of codes
__device__ __forceinline__ half2_t dequant_pair(half2_t c, half2_t s2, half2_t z2) {
  const half2_t m = c * s2;
  return m + z2;
}

// 1-bit normal-quantile coding (quant/pack_unpack.py:371-375): x = rnd16(rnd16(centre[c] * std) + mean)
// with centre = -+k, k = fp16(0.6745).  rnd16(-+k * std) = -+a with a = rnd16(k * std), so with a2 formed
// once per group the value is the single rounding of (2c - 1) * a + mean: two packed fused ops.
#define HQ_NORMAL1_CENTER ((_Float16)0.67431640625f)  // fp16(norm.ppf(0.75))
__device__ __forceinline__ half2_t normal1_spread(half2_t std2) {
  return std2 * (half2_t){HQ_NORMAL1_CENTER, HQ_NORMAL1_CENTER};
}
__device__ __forceinline__ half2_t dequant_pair_normal1(half2_t c, half2_t a2, half2_t mean2) {
  const half2_t t = __builtin_elementwise_fma(c, (half2_t){(_Float16)2, (_Float16)2}, (half2_t){(_Float16)-1, (_Float16)-1});
  return __builtin_elementwise_fma(t, a2, mean2);
}

// Consume one byte pair: 8/BITS dequantised pairs, each dotted with NREP operand pairs.
// NORMAL (1 bit only): s2 is the spread a2 = rnd16(k * std), z2 the mean.
template <int BITS, int NREP, int PF, bool NORMAL = false, int NFIELD = 8 / BITS>
__device__ __forceinline__ void consume_byte(uint32_t u, half2_t s2, half2_t z2, const half2_t (&a2)[NREP],
                                             float (&acc)[NREP][PF], int tok0) {
  constexpr int FPB = NFIELD;   // fields taken, from the low end of the byte
#define HQ_FIELD(I_)                                                                     \
  if constexpr (I_ < FPB) {                                                                      \
    const half2_t c2_ = field_pair<BITS, (I_ < FPB ? I_ : 0)>(u);                        \
    const half2_t x2 = NORMAL ? dequant_pair_normal1(c2_, s2, z2) : dequant_pair(c2_, s2, z2);  \
    _Pragma("unroll") for (int h = 0; h < NREP; ++h)                                     \
        acc[h][tok0 + I_] = __builtin_amdgcn_fdot2(x2, a2[h], acc[h][tok0 + I_], false); \
  }
  HQ_FIELD(0)
  HQ_FIELD(1)
  HQ_FIELD(2)
  HQ_FIELD(3)
  HQ_FIELD(4)
  HQ_FIELD(5)
  HQ_FIELD(6)
  HQ_FIELD(7)
#undef HQ_FIELD
}

// The same with the bias removal folded into the multiply (see bias_times_scale): nb[I] = -2^(10-POS_I) * s2.
template <int BITS, int NREP, int PF, int NFIELD>
__device__ __forceinline__ void consume_byte_fused_bias(uint32_t u, half2_t s2, half2_t z2, const half2_t (&nb)[8 / BITS],
                                                        const half2_t (&a2)[NREP], float (&acc)[NREP][PF], int tok0) {
#define HQ_FIELD(I_)                                                                      \
  if constexpr (I_ < NFIELD) {                                                            \
    const half2_t b2_ = field_pair_biased<BITS, (I_ < NFIELD ? I_ : 0)>(u);               \
    const half2_t m2_ = __builtin_elementwise_fma(b2_, s2, nb[I_ < NFIELD ? I_ : 0]);     \
    const half2_t x2 = m2_ + z2;                                                          \
    _Pragma("unroll") for (int h = 0; h < NREP; ++h)                                      \
        acc[h][tok0 + I_] = __builtin_amdgcn_fdot2(x2, a2[h], acc[h][tok0 + I_], false);  \
  }
  HQ_FIELD(0)
  HQ_FIELD(1)
  HQ_FIELD(2)
  HQ_FIELD(3)
  HQ_FIELD(4)
  HQ_FIELD(5)
  HQ_FIELD(6)
  HQ_FIELD(7)
#undef HQ_FIELD
}

template <int BITS, int NREP, int PF>
__device__ __forceinline__ void consume_words(uint32_t w0, uint32_t w1, half2_t s2, half2_t z2,
                                              const half2_t (&a2)[NREP], float (&acc)[NREP][PF]) {
  constexpr int FPB = 8 / BITS;
  consume_byte<BITS, NREP, PF>(byte_pair<0>(w0, w1), s2, z2, a2, acc, 0 * FPB);
  consume_byte<BITS, NREP, PF>(byte_pair<1>(w0, w1), s2, z2, a2, acc, 1 * FPB);
  consume_byte<BITS, NREP, PF>(byte_pair<2>(w0, w1), s2, z2, a2, acc, 2 * FPB);
  consume_byte<BITS, NREP, PF>(byte_pair<3>(w0, w1), s2, z2, a2, acc, 3 * FPB);
}

// ------------------------------------------------------------------------------- matrix-core form of the dot products
// With four query heads per KV head the inner product is a 4 x 4 x 4 matrix product per lane group: heads x
// (four elements of the reduction axis) x (the four lanes' tokens or channels).  v_mfma_f32_4x4x4_16b_f16 runs sixteen
// such blocks per wave, a block per four consecutive lanes: lane l supplies row l % 4 of its block's A (four fp16) and
// column l % 4 of its block's B, and receives column l % 4 of D (four fp32).  A holds the query (or the probabilities)
// of head l % 4, B the lane's own dequantised values -- bit for bit the ones the vector-ALU form feeds to its
// dot products -- so D is (4 heads) x (this lane's token or channel): one instruction on the matrix pipe in place of
// eight two-element dot products on the vector ALU.  Products are exact in fp32, accumulation is fp32; only the order
// of the additions differs from the vector-ALU form.
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f4_t mfma_4x4x4(half2_t a01, half2_t a23, half2_t b01, half2_t b23, f4_t c) {
  const half4_t a = __builtin_shufflevector(a01, a23, 0, 1, 2, 3);
  const half4_t b = __builtin_shufflevector(b01, b23, 0, 1, 2, 3);
  return __builtin_amdgcn_mfma_f32_4x4x4f16(a, b, c, 0, 0, 0);
}

template <typename F, int... Is>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, Is...>) {
  (f(std::integral_constant<int, Is>{}), ...);
}
// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// field I of a byte pair, dequantised with the reference's two roundings
template <int BITS, int I, bool NORMAL>
__device__ __forceinline__ half2_t dequant_field(uint32_t u, half2_t s2, half2_t z2) {
  const half2_t c2 = field_pair<BITS, I>(u);
  return NORMAL ? dequant_pair_normal1(c2, s2, z2) : dequant_pair(c2, s2, z2);
}
// the same with the bias removal folded into the multiply: nb = bias_times_scale<BITS, I>(s2)
template <int BITS, int I>
__device__ __forceinline__ half2_t dequant_field_fused_bias(uint32_t u, half2_t s2, half2_t z2, half2_t nb) {
  const half2_t m2 = __builtin_elementwise_fma(field_pair_biased<BITS, I>(u), s2, nb);
  return m2 + z2;
}

// Matrix-core form of consume_byte: byte pair `ua` belongs to elements 0, 1 of the reduction axis (a row pair of K, a
// token pair of V), `ub` to elements 2, 3; (a01, a23) is the A operand for those four elements.
template <int BITS, bool NORMAL, int NFIELD, int N>
__device__ __forceinline__ void consume_bytes_mfma(uint32_t ua, uint32_t ub, half2_t sa, half2_t za, half2_t sb, half2_t zb,
                                                   half2_t a01, half2_t a23, f4_t (&acc)[N], int tok0) {
  static_for<NFIELD>([&](auto I_) {
    constexpr int I = decltype(I_)::value;
    const half2_t xa = dequant_field<BITS, I, NORMAL>(ua, sa, za);
    const half2_t xb = dequant_field<BITS, I, NORMAL>(ub, sb, zb);
    acc[tok0 + I] = mfma_4x4x4(a01, a23, xa, xb, acc[tok0 + I]);
  });
}
template <int BITS, int NFIELD, int N>
__device__ __forceinline__ void consume_bytes_mfma_fused_bias(uint32_t ua, uint32_t ub, half2_t sa, half2_t za, half2_t sb,
                                                              half2_t zb, const half2_t (&nba)[8 / BITS],
                                                              const half2_t (&nbb)[8 / BITS], half2_t a01, half2_t a23,
                                                              f4_t (&acc)[N], int tok0) {
  static_for<NFIELD>([&](auto I_) {
    constexpr int I = decltype(I_)::value;
    const half2_t xa = dequant_field_fused_bias<BITS, I>(ua, sa, za, nba[I]);
    const half2_t xb = dequant_field_fused_bias<BITS, I>(ub, sb, zb, nbb[I]);
    acc[tok0 + I] = mfma_4x4x4(a01, a23, xa, xb, acc[tok0 + I]);
  });
}
__device__ __forceinline__ uint32_t byte_pair_at(uint32_t lo, uint32_t hi, int k) {  // byte_pair<k>, k known after unrolling
  return k == 0 ? byte_pair<0>(lo, hi) : k == 1 ? byte_pair<1>(lo, hi) : k == 2 ? byte_pair<2>(lo, hi) : byte_pair<3>(lo, hi);
}

}  // namespace hq
