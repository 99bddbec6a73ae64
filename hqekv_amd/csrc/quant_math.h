// Arithmetic shared by the quantise / dequantise kernels and the cache-migration kernel (gfx950): every routine
// here evaluates one step of the reference's fp16 chains with its roundings made explicit, so that any kernel
// built from them produces the same bits.  Include after "common.h", with fp contraction off.
#pragma once

#include "common.h"

#pragma clang fp contract(off)

namespace hq {

typedef float float2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t h2_bits(half2_t h) {
  uint32_t u;
  __builtin_memcpy(&u, &h, 4);
  return u;
}
__device__ __forceinline__ half2_t bits_h2(uint32_t u) {
  half2_t h;
  __builtin_memcpy(&h, &u, 4);
  return h;
}

// How the element-wise part of the chain is evaluated (results are those of the chain above, bit for bit):
//  * u = rnd16(x - mn) is one packed fp16 subtraction.  Rounding an fp16 sum first to fp32 (24-bit
//    significand >= 2*11+2) and then to fp16 gives the directly rounded fp16 sum, so there is nothing
//    to gain from the detour through fp32 that the op-by-op evaluation takes.
//  * v = rnd16(f32(u) / f32(scale)) is rnd16(f32(u) * r) with r the fp32 reciprocal of the group's
//    scale after one Newton step.  A quotient of two 11-bit significands is never closer than
//    1/(2047*4095) (relative) to a midpoint of the fp16 grid, which is more than the error of the
//    rounded product; hqekv_selftest_quant_division compares the two over all 2^32 operand pairs.
//    scale == 0 (constant group, or a range that underflows) and a non-finite scale keep the hardware
//    reciprocal (inf / 0 / NaN), which reproduces x/0 = inf, 0/0 = NaN and x/inf = 0.
//  * rne(clamp(v, 0, qmax)) is read from the significand of rnd16(clamp(v) + 1024): the fp16 grid has
//    spacing 1 on [1024, 2048) and 1024 is even, so the sum is 1024 + rne(v) exactly.  max() drops a
//    NaN operand, which turns the 0/0 of a constant group into code 0.
__device__ __forceinline__ float group_recip(float s) {
  const float r0 = __builtin_amdgcn_rcpf(s);
  const float e = __builtin_fmaf(-s, r0, 1.0f);
  const float r = __builtin_fmaf(e, r0, r0);
  // +-normal or +-denormal: classes 3, 4, 7, 8
  return __builtin_amdgcn_classf(s, 0x198) ? r : r0;
}

// fp16 bit patterns of 1024 + code for the pair (a, b) of already centred (x - mn) fp32 values
template <int BITS>
__device__ __forceinline__ uint32_t code_pair_biased(float ua, float ra, float ub, float rb) {
  constexpr _Float16 QMAX = (_Float16)((1 << BITS) - 1);
  const float2_t q = {ua * ra, ub * rb};
  half2_t v = __builtin_convertvector(q, half2_t);
  v = __builtin_elementwise_max(v, (half2_t){(_Float16)0, (_Float16)0});
  v = __builtin_elementwise_min(v, (half2_t){QMAX, QMAX});
  v = v + (half2_t){(_Float16)1024, (_Float16)1024};
  return h2_bits(v);
}

// z[i] holds (1024 + code[i], 1024 + code[i + N]) for i < N, N * BITS <= 16:
// returns code[i] at bit i*BITS and code[i + N] at bit 16 + i*BITS.
template <int BITS, int N>
__device__ __forceinline__ uint32_t horner_pack(const uint32_t *z) {
  constexpr uint32_t MASK = ((1u << BITS) - 1u) * 0x00010001u;
  uint32_t w = z[N - 1] & MASK;
#pragma unroll
  for (int i = N - 2; i >= 0; --i) w = (z[i] & MASK) | (w << BITS);
  return w;
}

// torch.min / torch.max over a group return the element with the LOWEST INDEX among equal ones (ATen's
// MinOps / MaxOps break ties by index), which decides the sign of a minimum or maximum that is zero when the group
// holds both +0 and -0.  The hardware minimum prefers -0 and the maximum +0, so groups whose minimum or maximum is
// a zero look the sign up: the bit pattern of the first zero among N values in index order, or 1 if there is none.
template <int N>
__device__ __forceinline__ uint32_t first_zero_bits(const half_t (&x)[N]) {
  uint32_t r = 1u;
#pragma unroll
  for (int i = N - 1; i >= 0; --i) {
    const uint32_t b = (uint32_t)__builtin_bit_cast(unsigned short, x[i]);
    if ((b & 0x7fffu) == 0u) r = b;
  }
  return r;
}

// One group of 32 contiguous values by four neighbouring lanes, `sub` = 0 .. 3, of which each holds eight: they store the codes.
struct QuantScale {
  half_t scale, zero;   // the same in all four lanes
};
template <int BITS>
__device__ __forceinline__ QuantScale quant_group_of_4(uint4 raw, uint32_t sub, uint32_t *crow) {
  constexpr float INV_QMAX = 1.0f / (float)((1 << BITS) - 1);
  const half2_t p[4] = {bits_h2(raw.x), bits_h2(raw.y), bits_h2(raw.z), bits_h2(raw.w)};

  half2_t lo2 = __builtin_elementwise_min(__builtin_elementwise_min(p[0], p[1]), __builtin_elementwise_min(p[2], p[3]));
  half2_t hi2 = __builtin_elementwise_max(__builtin_elementwise_max(p[0], p[1]), __builtin_elementwise_max(p[2], p[3]));
  // (min, -max) in one register: one packed min per butterfly step serves both
  half2_t mm = {(half_t)__builtin_fminf((float)lo2[0], (float)lo2[1]), (half_t)(-__builtin_fmaxf((float)hi2[0], (float)hi2[1]))};
  mm = __builtin_elementwise_min(mm, bits_h2(quad_xor_u<1>(h2_bits(mm))));
  mm = __builtin_elementwise_min(mm, bits_h2(quad_xor_u<2>(h2_bits(mm))));
  half_t mn_h = mm[0];
  float mn = (float)mn_h, mx = -(float)mm[1];
  // A zero extreme takes the sign of the group's first zero (torch's tie rule, see first_zero_bits).  The wave
  // branches around this as a whole (a scalar branch on the ballot): groups with a zero extreme are rare, and a
  // predicated copy of the block in every lane's path cost the kernel 5-10 %.
  const bool zero_extreme = __builtin_fminf(__builtin_fabsf(mn), __builtin_fabsf(mx)) == 0.0f;   // mn == 0 or mx == 0
  if (__builtin_amdgcn_ballot_w64(zero_extreme) != 0 && zero_extreme) {
    // (the condition is the same for the four lanes of a group: they hold its minimum and maximum)
    const half_t mine[8] = {p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
    const uint32_t own = first_zero_bits(mine);
    const uint32_t x1 = quad_xor_u<1>(own), x2 = quad_xor_u<2>(own), x3 = quad_xor_u<1>(x2);  // lanes sub^1, sub^2, sub^3
    uint32_t by_lane[4];
#pragma unroll
    for (int l = 0; l < 4; ++l) by_lane[l] = (sub == (uint32_t)l) ? own : (sub == (uint32_t)(l ^ 1)) ? x1 : (sub == (uint32_t)(l ^ 2)) ? x2 : x3;
    uint32_t first = 1u;
#pragma unroll
    for (int l = 3; l >= 0; --l)
      if (by_lane[l] != 1u) first = by_lane[l];
    const half_t z = __builtin_bit_cast(half_t, (unsigned short)first);   // (a zero extreme implies a zero element)
    if (mn == 0.0f) {
      mn_h = z;
      mn = (float)z;
    }
    if (mx == 0.0f) mx = (float)z;
  }

  const half_t d = (half_t)(mx - mn);
  const half_t sc = (half_t)((float)d * INV_QMAX);
  const float rcp = group_recip((float)sc);

  const half2_t mn2 = {mn_h, mn_h};
  float u[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const half2_t c = p[i] - mn2;
    u[2 * i] = (float)c[0];
    u[2 * i + 1] = (float)c[1];
  }

  if (BITS == 8) {
    uint32_t z[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      z[0] = code_pair_biased<8>(u[4 * h + 0], rcp, u[4 * h + 2], rcp);
      z[1] = code_pair_biased<8>(u[4 * h + 1], rcp, u[4 * h + 3], rcp);
      crow[sub * 2 + h] = horner_pack<8, 2>(z);
    }
  } else {
    uint32_t z[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) z[i] = code_pair_biased<BITS>(u[i], rcp, u[i + 4], rcp);
    if (BITS == 4) {
      crow[sub] = horner_pack<4, 4>(z);
    } else if (BITS == 1) {
      const uint32_t w = horner_pack<1, 4>(z);             // codes 0-3 in bits 0-3, codes 4-7 in bits 16-19
      const uint32_t b8 = (w & 0xfu) | ((w >> 12) & 0xf0u);  // this lane's 8 codes
      const uint32_t b16 = b8 | (quad_xor_u<1>(b8) << 8);        // even lanes: two lanes' codes in order
      const uint32_t other = quad_xor_u<2>(b16);
      if (sub == 0) crow[0] = b16 | (other << 16);
    } else {
      const uint32_t w = horner_pack<2, 4>(z);             // codes 0-3 in byte 0, codes 4-7 in byte 2
      const uint32_t h = __builtin_amdgcn_perm(0u, w, 0x0c0c0200u);   // 16 bits: this lane's 8 codes
      const uint32_t other = quad_xor_u<1>(h);
      if ((sub & 1) == 0) crow[sub >> 1] = h | (other << 16);
    }
  }
  return {sc, mn_h};
}
// the same from memory (16-byte aligned), scale and zero stored, too
template <int BITS>
__device__ __forceinline__ void quant_group_of_4(const half_t *x, uint32_t sub, uint32_t *crow, half_t *scale, half_t *zero) {
  const QuantScale q = quant_group_of_4<BITS>(*reinterpret_cast<const uint4 *>(x + sub * 8u), sub, crow);
  if (sub == 0) {
    *scale = q.scale;
    *zero = q.zero;
  }
}

struct Normal1Stats {
  half_t mean_h, std_h;
  float thr;  // std * 2^-25
};
struct Welford {
  float mean, m2;
};
// merge of two adjacent halves of n_half elements each (n_half a power of two, so every factor is exact)
__device__ __forceinline__ Welford welford_merge(Welford a, Welford b, float n_half) {
  const float delta = b.mean - a.mean;
  Welford r;
  r.mean = a.mean + delta * 0.5f;
  r.m2 = (a.m2 + b.m2) + ((delta * delta) * n_half) * 0.5f;
  return r;
}
// the tree over N = 2^k adjacent values held by one lane
template <int N>
__device__ __forceinline__ Welford welford_tree(const float (&x)[N]) {
  Welford w[N];
#pragma unroll
  for (int i = 0; i < N; ++i) w[i] = Welford{x[i], 0.f};
#pragma unroll
  for (int span = 1; span < N; span *= 2)
#pragma unroll
    for (int i = 0; i < N; i += 2 * span) w[i] = welford_merge(w[i], w[i + span], (float)span);
  return w[0];
}
__device__ __forceinline__ Normal1Stats normal1_finish(Welford w) {
  Normal1Stats st;
  st.mean_h = (half_t)w.mean;
  st.std_h = (half_t)__builtin_sqrtf(w.m2 / 31.0f);
  st.thr = (float)st.std_h * 0x1p-25f;
  return st;
}
__device__ __forceinline__ uint32_t normal1_code(half_t u, float thr) {
  const float uf = (float)u;
  return (uf > 0.0f && uf > thr) ? 1u : 0u;
}

}  // namespace hq
