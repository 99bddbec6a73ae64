// Cache maintenance on the device: one launch rebuilds every precision class of both sides (K and V) of a layer's
// cache from the old classes and the new fp16 tokens, following a block-level plan the host worked out.
//
// What the reference does per compression (quant/hqe_2.py:552-836) is a sequence of boolean-mask gathers,
// dequantise / re-quantise calls and torch.cat re-copies, one group of launches per (source, target) pair.  All of
// it moves whole blocks of 32 tokens, and every block ends in exactly one place, so the whole compression is a
// gather: destination block u of class c comes from block v of source s.  A unit of work is one quantisation
// group of one block -- K: (block, channel), the 32 tokens of a channel; V: (token, 32 channels) -- held by one
// lane as 32 fp16 values:
//   same width            copy of the packed words, scale and zero (a survivor keeps its bytes)
//   fp16 -> b bits        the quantiser of quant/pack_unpack.py:156-193 (or :218-253 for the 1-bit normal class)
//   a bits -> b < a bits  dequantise with the reference's two fp16 roundings (quant/pack_unpack.py:331-332), then
//                         quantise: what K_high_2_low / V_high_2_low do (quant/hqe_2.py:88-170)
//   fp16 -> fp16          copy (new K arrives token-major and is stored channel-major)
// Evicted blocks are simply in nobody's plan.  The arithmetic is the one of the stand-alone kernels (quant_math.h),
// so the bytes equal those of the step-by-step path.
#include <stddef.h>

#include "common.h"
#include "quant_math.h"

#pragma clang fp contract(off)

namespace hq {

struct MigClass {
  void *data;
  half_t *scale;
  half_t *zero;
  int64_t *idx;
  int64_t n_tokens;
  int64_t slab_tokens;  // tokens between (b, h) slabs of a token-major fp16 source (>= n_tokens)
  int32_t bits;
  int32_t layout;
  int32_t begin;        // destination: its first plan entry
  int32_t pad;
};

struct MigSide {
  MigClass src[HQEKV_MAX_SEGS];
  MigClass dst[HQEKV_MAX_SEGS];
  int32_t dst_begin[HQEKV_MAX_SEGS + 1];  // first plan entry of every destination class; [n_dst] = total
  int32_t n_dst;
  int32_t n_src;
  int32_t wgs;              // workgroups that serve the side
  const int32_t *plan_src;  // (source slot << 24) | source block, per destination block
  const int32_t *plan_pos;  // new position of the block's first token / 32
};

struct MigArgs {
  MigSide side[2];   // K, V
  hqekv_migrate_extra x;
  int32_t *status;   // optional: set to non-zero when a plan entry is refused
  int32_t BH, D;
};

// The plan lives in device memory and is read by the kernel only, so the kernel is what checks it: an entry must name
// a populated source class, a block inside it and a position inside the new sequence.  An entry that does not is
// skipped (its destination block keeps whatever the buffer held) and flagged; nothing is read or written out of range.
__device__ __forceinline__ bool plan_entry_ok(const MigClass *src, int n_src, int32_t code, int32_t pos, int total) {
  const uint32_t slot = (uint32_t)code >> 24, blk = (uint32_t)code & 0xffffffu;
  if (slot >= (uint32_t)n_src) return false;
  const int64_t n = src[slot].n_tokens;
  return n > 0 && src[slot].data != nullptr && (int64_t)blk < (n >> 5) && pos >= 0 && pos < total;
}
__device__ __forceinline__ void plan_refused(const MigArgs &a) {
  if (a.status) atomicOr(a.status, 1);
}

// where one lane's group lives: 32 adjacent fp16 values or packed words + scale + zero (blocks of token-major keys, whose
// groups are strided, are read by load_token_major_pair)
struct GroupRef {
  half_t *f16;
  uint32_t *words;
  half_t *s, *z;
};

template <bool IS_K>
__device__ __forceinline__ GroupRef group_ref(const MigClass &c, int64_t bh, int64_t block, int lane, int D) {
  GroupRef r{};
  const int64_t n = c.n_tokens;
  if (IS_K) {
    const int d = lane;  // channel
    if (c.bits == 16) {
      r.f16 = (half_t *)c.data + ((bh * D + d) * n + block * 32);   // (B,H,D,T)
    } else {
      const int64_t g = (bh * D + d) * (n >> 5) + block;
      r.words = (uint32_t *)c.data + g * c.bits;  // 32 codes of b bits = b words
      r.s = c.scale + g;
      r.z = c.zero + g;
    }
  } else {
    const int ng = D >> 5;
    const int k = lane / ng, cg = lane % ng;  // token of the block, channel group
    if (c.bits == 16) {
      const int64_t t = bh * c.slab_tokens + block * 32 + k;
      r.f16 = (half_t *)c.data + (t * D + cg * 32);
    } else {
      const int64_t g = (bh * n + block * 32 + k) * ng + cg;
      r.words = (uint32_t *)c.data + g * c.bits;
      r.s = c.scale + g;
      r.z = c.zero + g;
    }
  }
  return r;
}

// 32 fp16 values as 16 registers: xp[j] = (x[2j], x[2j+1])
__device__ __forceinline__ void load_f16(const GroupRef &r, uint32_t (&xp)[16]) {
  const uint4 *p = reinterpret_cast<const uint4 *>(r.f16);  // block starts are 64-byte aligned
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint4 v = p[i];
    xp[4 * i] = v.x;
    xp[4 * i + 1] = v.y;
    xp[4 * i + 2] = v.z;
    xp[4 * i + 3] = v.w;
  }
}
__device__ __forceinline__ void store_f16(const GroupRef &r, const uint32_t (&xp)[16]) {
  uint4 *p = reinterpret_cast<uint4 *>(r.f16);  // fp16 classes are stored with unit stride
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] = make_uint4(xp[4 * i], xp[4 * i + 1], xp[4 * i + 2], xp[4 * i + 3]);
}

// out = rnd16(rnd16(c * scale) + zero); NORMAL: rnd16(rnd16(+-k * std) + mean)
template <int BITS, bool NORMAL>
__device__ __forceinline__ void dequant_group(const GroupRef &r, uint32_t (&xp)[16]) {
  constexpr int PF = 32 / BITS;
  uint32_t w[BITS];
#pragma unroll
  for (int i = 0; i < BITS; ++i) w[i] = r.words[i];
  const half_t s = *r.s, z = *r.z;
  // fp16 multiply and add, each one rounding of the exact result (through fp32 the compiler's mixed-precision fma
  // with a +0 addend would lose the sign of a -0 product)
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    half2_t v;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int k = 2 * j + e;
      const uint32_t ci = code_at<BITS>(w[k / PF], k % PF);
      const half_t m = NORMAL ? (ci != 0u ? (half_t)0.67431640625f : (half_t)-0.67431640625f) * s : (half_t)(float)ci * s;
      v[e] = m + z;
    }
    xp[j] = h2_bits(v);
  }
}

template <int BITS>
__device__ __forceinline__ void quant_group(const GroupRef &r, const uint32_t (&xp)[16]) {
  constexpr int PF = 32 / BITS;
  constexpr int HALF = PF / 2;
  constexpr float INV_QMAX = 1.0f / (float)((1 << BITS) - 1);
  half2_t lo2 = bits_h2(xp[0]), hi2 = lo2;
#pragma unroll
  for (int j = 1; j < 16; ++j) {
    lo2 = __builtin_elementwise_min(lo2, bits_h2(xp[j]));
    hi2 = __builtin_elementwise_max(hi2, bits_h2(xp[j]));
  }
  half_t mn_h = (half_t)__builtin_fminf((float)lo2[0], (float)lo2[1]);
  float mn = (float)mn_h, mx = __builtin_fmaxf((float)hi2[0], (float)hi2[1]);
  // a zero extreme takes the sign of the group's first zero (torch's tie rule); rare, so the wave branches around it
  if (__builtin_amdgcn_ballot_w64(mn == 0.0f || mx == 0.0f) != 0 && (mn == 0.0f || mx == 0.0f)) {
    half_t v[32];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const half2_t h = bits_h2(xp[j]);
      v[2 * j] = h[0];
      v[2 * j + 1] = h[1];
    }
    const half_t z = __builtin_bit_cast(half_t, (unsigned short)first_zero_bits(v));
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
  float u[32];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const half2_t c = bits_h2(xp[j]) - mn2;
    u[2 * j] = (float)c[0];
    u[2 * j + 1] = (float)c[1];
  }
#pragma unroll
  for (int wj = 0; wj < BITS; ++wj) {
    uint32_t zz[HALF];
#pragma unroll
    for (int i = 0; i < HALF; ++i) zz[i] = code_pair_biased<BITS>(u[wj * PF + i], rcp, u[wj * PF + i + HALF], rcp);
    r.words[wj] = horner_pack<BITS, HALF>(zz);
  }
  *r.s = sc;
  *r.z = mn_h;
}

// the 1-bit normal-quantile quantiser: statistics in the order of torch's GPU reduction, code = [x > mean]
__device__ __forceinline__ void quant_group_normal1(const GroupRef &r, const uint32_t (&xp)[16]) {
  float xf[32];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const half2_t v = bits_h2(xp[j]);
    xf[2 * j] = (float)v[0];
    xf[2 * j + 1] = (float)v[1];
  }
  const Normal1Stats st = normal1_finish(welford_tree<32>(xf));
  uint32_t w = 0;
#pragma unroll
  for (int k = 0; k < 32; ++k) w |= normal1_code((half_t)(xf[k] - (float)st.mean_h), st.thr) << k;
  r.words[0] = w;
  *r.s = st.std_h;
  *r.z = st.mean_h;
}

// a group's values into the destination's form
__device__ __forceinline__ void quantize_to(const MigClass &dc, const GroupRef &dr, const uint32_t (&xp)[16]) {
  switch (dc.bits) {
    case 16: store_f16(dr, xp); break;
    case 8: quant_group<8>(dr, xp); break;
    case 4: quant_group<4>(dr, xp); break;
    case 2: quant_group<2>(dr, xp); break;
    default:
      if (dc.layout == HQEKV_LAYOUT_NORMAL1) quant_group_normal1(dr, xp);
      else quant_group<1>(dr, xp);
  }
}

// The packed words, scale and zero of N groups, all requested before the first is stored; a group's words start at a
// multiple of their own size, so they move as vectors where the planes are 16-byte aligned (every plane this package
// allocates is).
template <int BITS, int N>
__device__ __forceinline__ void copy_groups(const GroupRef (&sr)[N], const GroupRef (&dr)[N]) {
  constexpr int V = BITS < 4 ? BITS : 4;
  typedef uint32_t vec_t __attribute__((ext_vector_type(V)));
  half_t s[N], z[N];
#pragma unroll
  for (int g = 0; g < N; ++g) {
    s[g] = *sr[g].s;
    z[g] = *sr[g].z;
  }
  if ((((uintptr_t)sr[0].words | (uintptr_t)dr[0].words) & (4 * V - 1)) == 0) {   // (the same for all groups of a class)
    vec_t w[N][BITS / V];
#pragma unroll
    for (int g = 0; g < N; ++g)
#pragma unroll
      for (int i = 0; i < BITS / V; ++i) w[g][i] = reinterpret_cast<const vec_t *>(sr[g].words)[i];
#pragma unroll
    for (int g = 0; g < N; ++g)
#pragma unroll
      for (int i = 0; i < BITS / V; ++i) reinterpret_cast<vec_t *>(dr[g].words)[i] = w[g][i];
  } else {
    uint32_t w[N][BITS];
#pragma unroll
    for (int g = 0; g < N; ++g)
#pragma unroll
      for (int i = 0; i < BITS; ++i) w[g][i] = sr[g].words[i];
#pragma unroll
    for (int g = 0; g < N; ++g)
#pragma unroll
      for (int i = 0; i < BITS; ++i) dr[g].words[i] = w[g][i];
  }
#pragma unroll
  for (int g = 0; g < N; ++g) {
    *dr[g].s = s[g];
    *dr[g].z = z[g];
  }
}

// a survivor of a quantised class keeps its bytes
template <int N>
__device__ __forceinline__ void copy_groups_of(int bits, const GroupRef (&sr)[N], const GroupRef (&dr)[N]) {
  switch (bits) {
    case 8: copy_groups<8>(sr, dr); break;
    case 4: copy_groups<4>(sr, dr); break;
    case 2: copy_groups<2>(sr, dr); break;
    default: copy_groups<1>(sr, dr);
  }
}

// N quantisation groups: lane, lane + step, ... = channel (K) or (token, channel group) (V) of source block sb ->
// destination block db.
template <bool IS_K, int N>
__device__ __forceinline__ void migrate_groups(const MigClass &sc, const MigClass &dc, int64_t bh, int64_t sb, int64_t db,
                                               int lane, int step, int D) {
  if (sc.bits != 16 && sc.bits == dc.bits) {
    GroupRef sr[N], dr[N];
#pragma unroll
    for (int g = 0; g < N; ++g) {
      sr[g] = group_ref<IS_K>(sc, bh, sb, lane + g * step, D);
      dr[g] = group_ref<IS_K>(dc, bh, db, lane + g * step, D);
    }
    copy_groups_of(sc.bits, sr, dr);
    return;
  }
  const bool sn = sc.layout == HQEKV_LAYOUT_NORMAL1;
#pragma unroll 1
  for (int g = 0; g < N; ++g) {
    const GroupRef s = group_ref<IS_K>(sc, bh, sb, lane + g * step, D), d = group_ref<IS_K>(dc, bh, db, lane + g * step, D);
    uint32_t xp[16];
    switch (sc.bits) {
      case 16: load_f16(s, xp); break;
      case 8: dequant_group<8, false>(s, xp); break;
      case 4: dequant_group<4, false>(s, xp); break;
      case 2: dequant_group<2, false>(s, xp); break;
      default:
        if (sn) dequant_group<1, true>(s, xp);
        else dequant_group<1, false>(s, xp);
    }
    quantize_to(dc, d, xp);
  }
}

__device__ __forceinline__ int dst_class_of(const MigSide &a, int u) {
  int ci = 0;
#pragma unroll
  for (int k = 1; k < HQEKV_MAX_SEGS; ++k) ci += (k < a.n_dst && u >= a.dst_begin[k]) ? 1 : 0;
  return ci;
}

constexpr int MIG_THREADS = 256;
constexpr int MIG_KB = 16;         // K side: destination blocks per workgroup
constexpr int MIG_KC = 32;         // ... and channels
constexpr int MIG_VB = 4;          // V side: destination blocks per workgroup
constexpr int MIG_XC = 16;         // columns of a ring row a thread moves at a time
static_assert(MIG_KC == 2 * (MIG_THREADS / MIG_KB), "a lane of the K side holds two channels of a block");

// The side's class tables in LDS: a lane's classes follow from its plan entry, and tables in the argument block would be
// a second trip to memory behind that of the entry.
struct MigTables {
  MigClass src[HQEKV_MAX_SEGS], dst[HQEKV_MAX_SEGS];
};
__device__ __forceinline__ void fetch_tables(const MigSide &a, MigTables &t) {
  static_assert(offsetof(MigSide, src) == 0 && offsetof(MigSide, dst) == sizeof(MigClass) * HQEKV_MAX_SEGS && sizeof(MigTables) % 4 == 0 &&
                    sizeof(MigTables) / 4 <= MIG_THREADS, "one word per thread");
  if (threadIdx.x < sizeof(MigTables) / 4) reinterpret_cast<uint32_t *>(&t)[threadIdx.x] = reinterpret_cast<const uint32_t *>(&a)[threadIdx.x];
}

// K side.  A group is 32 tokens of ONE channel row -- b words of the row -- and a block's groups lie a whole row
// apart, so a workgroup takes 16 consecutive destination blocks and lets neighbouring lanes take neighbouring
// blocks of a row: 16 b-word pieces side by side (64 bytes at 1 bit ... 512 at 8), and as long as the blocks come
// from consecutive places of one source class (survivors of a class stay in order) the reads line up the same
// way.  (A lane per channel, as on the V side, touched a separate cache line per lane: the K side took four to
// six times as long as the V side for the same bytes.)  A workgroup covers 32 channels, so that a side of a thousand
// blocks is some thousands of short workgroups.  Blocks of new tokens (token-major: the channels of a token are what is
// contiguous) go side by side as well, a lane holding two channels of one.
__device__ __forceinline__ void migrate_keys(const MigArgs &a, int wg, const MigTables &tab) {
  const MigSide &s = a.side[0];
  const int total = s.dst_begin[HQEKV_MAX_SEGS], D = a.D, groups = (total + MIG_KB - 1) / MIG_KB;
  const int u0 = wg % groups * MIG_KB, d0 = wg / groups / a.BH * MIG_KC;
  const int64_t bh = wg / groups % a.BH;
  // thread -> block of the 16: `slot` for the class to class part, `tslot` for blocks of new tokens
  const int slot = threadIdx.x % MIG_KB, tslot = threadIdx.x / 8 % MIG_KB;
  const int u = u0 + slot, tu = u0 + tslot;
  const int uc = min(u, total - 1), tuc = min(tu, total - 1);
  const int32_t code = s.plan_src[uc], pos = s.plan_pos[uc], tcode = s.plan_src[tuc], tpos = s.plan_pos[tuc];
  __syncthreads();   // the tables
  auto token_major = [&](int32_t c) {
    const MigClass &sc = tab.src[(uint32_t)c >> 24];
    return sc.bits == 16 && sc.layout == HQEKV_LAYOUT_TOKEN_MAJOR;
  };
  const bool ok = u < total && plan_entry_ok(tab.src, s.n_src, code, pos, total);
  if (u < total && !ok) plan_refused(a);
  const int ci = dst_class_of(s, uc);
  if (bh == 0 && d0 == 0 && ok && tab.dst[ci].idx) {   // positions of the blocks' tokens
    int64_t *idx = tab.dst[ci].idx + (int64_t)(u - tab.dst[ci].begin) * 32;
    for (int e = threadIdx.x / MIG_KB; e < 32; e += MIG_THREADS / MIG_KB) idx[e] = (int64_t)pos * 32 + e;
  }
  const bool tm = ok && token_major(code);
  if (ok && !tm)
    migrate_groups<true, 2>(tab.src[(uint32_t)code >> 24], tab.dst[ci], bh, code & 0xffffff, u - tab.dst[ci].begin, d0 + threadIdx.x / MIG_KB,
                            MIG_THREADS / MIG_KB, D);
  if (!__syncthreads_or(tm)) return;
  // blocks of new tokens: 16 blocks x 16 channel pairs, eight neighbouring lanes on neighbouring pairs (32 bytes of a
  // token row), the next eight on the next block
  const int pair = threadIdx.x % 8 + threadIdx.x / (8 * MIG_KB) * 8;
  static_assert(MIG_THREADS == MIG_KB * MIG_KC / 2, "one channel pair of one block per thread");
  if (tu >= total || !plan_entry_ok(tab.src, s.n_src, tcode, tpos, total) || !token_major(tcode)) return;
  const int tci = dst_class_of(s, tu);
  const MigClass &sc = tab.src[(uint32_t)tcode >> 24], &dc = tab.dst[tci];
  // 32 tokens of channels d and d + 1: two groups from 32 four-byte loads
  const uint32_t *p = reinterpret_cast<const uint32_t *>((const half_t *)sc.data + (bh * sc.slab_tokens + (tcode & 0xffffff) * 32LL) * D + d0 + 2 * pair);
  uint32_t w[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) w[i] = p[i * (D >> 1)];
#pragma unroll 1
  for (int e = 0; e < 2; ++e) {
    const GroupRef dr = group_ref<true>(dc, bh, tu - dc.begin, d0 + 2 * pair + e, D);
    const uint32_t halves = e ? 0x07060302u : 0x05040100u;   // which channel of every word
    uint32_t x[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) x[j] = __builtin_amdgcn_perm(w[2 * j + 1], w[2 * j], halves);
    quantize_to(dc, dr, x);
  }
}

// V side: half a workgroup per two destination blocks; a block's 32 tokens x D/32 groups are one contiguous stretch of every
// plane.  The two blocks are in flight together where both only move within one class.
__device__ __forceinline__ void migrate_values(const MigArgs &a, int wg, const MigTables &tab) {
  const MigSide &s = a.side[1];
  const int total = s.dst_begin[HQEKV_MAX_SEGS], D = a.D, groups = (total + MIG_VB - 1) / MIG_VB;
  const int64_t bh = wg / groups;
  constexpr int LANES = 2 * MIG_THREADS / MIG_VB;
  const int u0 = wg % groups * MIG_VB + threadIdx.x / LANES * 2, l0 = threadIdx.x % LANES;
  int32_t code[2], pos[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int uc = min(u0 + k, total - 1);
    code[k] = s.plan_src[uc];
    pos[k] = s.plan_pos[uc];
  }
  __syncthreads();   // the tables
  bool ok[2];
  int ci[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {   // uniform: the whole half serves these entries
    ok[k] = u0 + k < total && plan_entry_ok(tab.src, s.n_src, code[k], pos[k], total);
    if (u0 + k < total && !ok[k] && l0 == 0) plan_refused(a);
    ci[k] = dst_class_of(s, min(u0 + k, total - 1));
    int64_t *idx = tab.dst[ci[k]].idx;
    if (ok[k] && bh == 0 && l0 < 32 && idx) idx[(int64_t)(u0 + k - tab.dst[ci[k]].begin) * 32 + l0] = (int64_t)pos[k] * 32 + l0;
  }
  const int bits = tab.dst[ci[0]].bits;
  if (ok[0] && ok[1] && ci[0] == ci[1] && bits != 16 && tab.src[(uint32_t)code[0] >> 24].bits == bits && tab.src[(uint32_t)code[1] >> 24].bits == bits) {
    for (int lane = l0; lane < D; lane += LANES) {
      GroupRef sr[2], dr[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        sr[k] = group_ref<false>(tab.src[(uint32_t)code[k] >> 24], bh, code[k] & 0xffffff, lane, D);
        dr[k] = group_ref<false>(tab.dst[ci[k]], bh, u0 + k - tab.dst[ci[k]].begin, lane, D);
      }
      copy_groups_of(bits, sr, dr);
    }
    return;
  }
#pragma unroll 1
  for (int k = 0; k < 2; ++k) {
    const int32_t c = k ? code[1] : code[0];
    const MigClass &dc = tab.dst[k ? ci[1] : ci[0]];
    if (!(k ? ok[1] : ok[0])) continue;
    for (int lane = l0; lane < D; lane += LANES)
      migrate_groups<false, 1>(tab.src[(uint32_t)c >> 24], dc, bh, c & 0xffffff, u0 + k - dc.begin, lane, 0, D);
  }
}

struct __attribute__((packed, aligned(2))) ring_quad_t { uint64_t v; };   // four fp16 columns at an element's alignment

// What rides along: workgroup by workgroup the rows of the importance ring without the evicted columns, the token ranges
// without them, and the residual rows that stay behind.
__device__ __forceinline__ void migrate_extras(const MigArgs &a, int wg) {
  const hqekv_migrate_extra &x = a.x;
  if (wg < x.ring_rows) {
    // In place, ascending: a column moves to the left or stays, so a pass overwrites nothing a later pass reads, and
    // within a pass every thread holds its columns before the first is stored.
    half_t *row = (half_t *)x.ring + (int64_t)wg * x.ring_stride;
    const int n = x.n_alive * 32;
    for (int c0 = x.first_moved * 32; c0 < n; c0 += MIG_THREADS * MIG_XC) {
      const int c = c0 + threadIdx.x * MIG_XC;
      ring_quad_t v[MIG_XC / 4];
      if (c < n) {
        const ring_quad_t *from = reinterpret_cast<const ring_quad_t *>(row + (int64_t)x.alive[c >> 5] * 32 + (c & 31));
#pragma unroll
        for (int i = 0; i < MIG_XC / 4; ++i) v[i] = from[i];
      }
      __syncthreads();
      if (c < n) {
        ring_quad_t *to = reinterpret_cast<ring_quad_t *>(row + c);
#pragma unroll
        for (int i = 0; i < MIG_XC / 4; ++i) to[i] = v[i];
      }
      __syncthreads();
    }
    return;
  }
  wg -= x.ring_rows;
  const int range_wgs = x.range_out ? (x.n_alive * 32 + MIG_THREADS - 1) / MIG_THREADS : 0;
  if (wg < range_wgs) {
    const int c = wg * MIG_THREADS + threadIdx.x;
    if (c < x.n_alive * 32) ((half_t *)x.range_out)[c] = ((const half_t *)x.range_in)[(int64_t)x.alive[c >> 5] * 32 + (c & 31)];
    return;
  }
  wg -= range_wgs;
  // 16-byte pieces of the residual rows of both sides
  const int64_t per_slab = (int64_t)x.res_rows * a.D / 8, i = (int64_t)wg * MIG_THREADS + threadIdx.x;
  if (i >= 2 * a.BH * per_slab) return;
  const int side = i >= a.BH * per_slab ? 1 : 0;
  const int64_t j = i - side * a.BH * per_slab, bh = j / per_slab, k = j % per_slab;
  const uint4 *src = reinterpret_cast<const uint4 *>((const half_t *)x.res_src[side] + bh * x.res_src_slab[side] * a.D) + k;
  reinterpret_cast<uint4 *>((half_t *)x.res_dst[side] + bh * x.res_dst_slab[side] * a.D)[k] = *src;
}

// Both sides of a layer in one launch, the K workgroups (the longer ones) first.  Bound by latency -- plan entry, group,
// store, each a trip to memory -- at 35 MB in and 35 out at 32k tokens: 22 + 12 us as two launches, with the class tables in
// the argument block and one group in flight per lane; 28 us as one launch of three waves per SIMD, 25 of four, 22.7 with
// two V blocks in flight, 19.3 with neighbouring K workgroups on one XCD (32 bytes of a channel's scales each: lines met in
// memory instead of in one L2; a copy of those bytes takes 14).  4 waves per SIMD are what the 1-bit normal statistics leave.
__global__ __launch_bounds__(MIG_THREADS, 4) void cache_migrate_kernel(MigArgs a) {
  __shared__ MigTables tab;
  int wg = blockIdx.x;
  if (wg < a.side[0].wgs) {
    fetch_tables(a.side[0], tab);
    migrate_keys(a, (int)by_xcd((uint32_t)wg, (uint32_t)a.side[0].wgs), tab);
    return;
  }
  wg -= a.side[0].wgs;
  if (wg < a.side[1].wgs) {
    fetch_tables(a.side[1], tab);
    migrate_values(a, wg, tab);
    return;
  }
  migrate_extras(a, wg - a.side[1].wgs);
}

// Words from page-locked memory: a launch of a few workgroups arrives sooner than a copy through the DMA engines, whose
// completion another queue has to be told of.
__global__ __launch_bounds__(256) void fetch_words_kernel(const uint32_t *__restrict__ src, uint32_t *__restrict__ dst, int n) {
  const int i = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (i + 4 <= n) *reinterpret_cast<uint4 *>(dst + i) = *reinterpret_cast<const uint4 *>(src + i);
  else
    for (int k = i; k < n; ++k) dst[k] = src[k];
}

static int check_class(const hqekv_cache_class &c, bool is_src, int k, int64_t D) {
  const char *side = is_src ? "source" : "destination";
  if (c.n_tokens < 0 || c.n_tokens % 32 != 0)
    return fail(HQEKV_E_ARG, "cache_migrate: %s %d holds %lld tokens (whole blocks of 32 only)", side, k, (long long)c.n_tokens);
  if (c.n_tokens == 0) return HQEKV_OK;
  if (!(c.bits == 16 || c.bits == 8 || c.bits == 4 || c.bits == 2 || c.bits == 1))
    return fail(HQEKV_E_ARG, "cache_migrate: %s %d bits=%d", side, k, c.bits);
  if (!c.data || (c.bits != 16 && (!c.scale || !c.zero)))
    return fail(HQEKV_E_ARG, "cache_migrate: %s %d lacks data / scale / zero", side, k);
  if ((uintptr_t)c.data & (c.bits == 16 ? 15 : 3)) return fail(HQEKV_E_ALIGN, "cache_migrate: %s %d data misaligned", side, k);
  if (c.n_tokens * D >= (1LL << 40)) return fail(HQEKV_E_UNSUPPORTED, "cache_migrate: %s %d too large", side, k);
  return HQEKV_OK;
}

// One side's tables, checked.
static int fill_side(bool is_k, const hqekv_cache_class *src, int n_src, const hqekv_cache_class *dst, int n_dst, const int32_t *plan,
                     int64_t BH, int64_t D, MigSide *a) {
  if (n_src < 0 || n_src > HQEKV_MAX_SEGS || n_dst < 0 || n_dst > HQEKV_MAX_SEGS || (n_src && !src) || (n_dst && !dst))
    return fail(HQEKV_E_ARG, "cache_migrate: bad class tables");
  int64_t total = 0;
  for (int k = 0; k < n_src; ++k) {
    const int rc = check_class(src[k], true, k, D);
    if (rc) return rc;
    // fp16 sources are read 32 values at a time: channel-major rows and token-major rows start 16-byte aligned
    const int64_t slab = src[k].slab_tokens > 0 ? src[k].slab_tokens : src[k].n_tokens;
    if (slab < src[k].n_tokens || (slab != src[k].n_tokens && !(src[k].bits == 16 && (!is_k || src[k].layout == HQEKV_LAYOUT_TOKEN_MAJOR))))
      return fail(HQEKV_E_ARG, "cache_migrate: source %d: slab_tokens applies to token-major fp16 sources and must be >= n_tokens", k);
    a->src[k] = MigClass{src[k].data, (half_t *)src[k].scale, (half_t *)src[k].zero, nullptr, src[k].n_tokens, slab, src[k].bits, src[k].layout, 0, 0};
  }
  for (int k = 0; k < n_dst; ++k) {
    const int rc = check_class(dst[k], false, k, D);
    if (rc) return rc;
    if (dst[k].bits == 16 && dst[k].layout == HQEKV_LAYOUT_TOKEN_MAJOR && is_k)
      return fail(HQEKV_E_UNSUPPORTED, "cache_migrate: the fp16 K class is stored channel-major");
    if (dst[k].slab_tokens != 0 && dst[k].slab_tokens != dst[k].n_tokens)
      return fail(HQEKV_E_ARG, "cache_migrate: destination %d must be stored densely", k);
    a->dst[k] = MigClass{dst[k].data, (half_t *)dst[k].scale, (half_t *)dst[k].zero, dst[k].idx, dst[k].n_tokens, dst[k].n_tokens, dst[k].bits, dst[k].layout, (int32_t)total, 0};
    a->dst_begin[k] = (int32_t)total;
    total += dst[k].n_tokens / 32;
  }
  for (int k = n_dst; k <= HQEKV_MAX_SEGS; ++k) a->dst_begin[k] = (int32_t)total;
  if (total == 0) return HQEKV_OK;
  if (total >= (1 << 24)) return fail(HQEKV_E_UNSUPPORTED, "cache_migrate: %lld blocks (limit 2^24)", (long long)total);
  if (!plan) return fail(HQEKV_E_ARG, "cache_migrate: null plan");
  a->n_dst = n_dst;
  a->n_src = n_src;
  a->plan_src = plan;
  a->plan_pos = plan + total;
  const int64_t wgs = is_k ? (total + MIG_KB - 1) / MIG_KB * BH * (D / MIG_KC) : (total + MIG_VB - 1) / MIG_VB * BH;
  if (wgs > 0x3fffffff) return fail(HQEKV_E_UNSUPPORTED, "cache_migrate: too many blocks and heads for one launch");
  a->wgs = (int32_t)wgs;
  return HQEKV_OK;
}

static int launch_migrate(MigArgs &a, int64_t BH, int64_t D, hipStream_t stream) {
  a.BH = (int32_t)BH;
  a.D = (int32_t)D;
  const hqekv_migrate_extra &x = a.x;
  const int64_t extra = x.ring_rows + (x.range_out ? ((int64_t)x.n_alive * 32 + MIG_THREADS - 1) / MIG_THREADS : 0) +
                        (2 * BH * x.res_rows * D / 8 + MIG_THREADS - 1) / MIG_THREADS;
  const int64_t wgs = a.side[0].wgs + a.side[1].wgs + extra;
  if (wgs == 0) return HQEKV_OK;
  if (wgs > 0x7fffffff) return fail(HQEKV_E_UNSUPPORTED, "cache_migrate: too many blocks and heads for one launch");
  hipLaunchKernelGGL(cache_migrate_kernel, dim3((unsigned)wgs), dim3(MIG_THREADS), 0, stream, a);
  return check_launch("cache_migrate_kernel");
}

}  // namespace hq

using namespace hq;

extern "C" int hqekv_cache_migrate(int is_k, const hqekv_cache_class *src, int n_src, const hqekv_cache_class *dst,
                                   int n_dst, const int32_t *plan, int64_t BH, int64_t D, int32_t *status, void *stream) {
  if (BH <= 0 || BH > 65535 || D <= 0 || D % 32 != 0 || D > 1024)
    return fail(HQEKV_E_ARG, "cache_migrate: need 0 < B*H <= 65535 and head_dim a multiple of 32 up to 1024");
  MigArgs a{};
  a.status = status;
  const int rc = fill_side(is_k != 0, src, n_src, dst, n_dst, plan, BH, D, &a.side[is_k ? 0 : 1]);
  return rc ? rc : launch_migrate(a, BH, D, (hipStream_t)stream);
}

extern "C" int hqekv_cache_migrate_both(const hqekv_cache_class *k_src, int n_k_src, const hqekv_cache_class *k_dst, int n_k_dst,
                                        const int32_t *k_plan, const hqekv_cache_class *v_src, int n_v_src,
                                        const hqekv_cache_class *v_dst, int n_v_dst, const int32_t *v_plan, int64_t BH, int64_t D,
                                        const hqekv_migrate_extra *extra, void *stream) {
  if (BH <= 0 || BH > 65535 || D <= 0 || D % 32 != 0 || D > 1024)
    return fail(HQEKV_E_ARG, "cache_migrate: need 0 < B*H <= 65535 and head_dim a multiple of 32 up to 1024");
  MigArgs a{};
  int rc = fill_side(true, k_src, n_k_src, k_dst, n_k_dst, k_plan, BH, D, &a.side[0]);
  if (!rc) rc = fill_side(false, v_src, n_v_src, v_dst, n_v_dst, v_plan, BH, D, &a.side[1]);
  if (rc) return rc;
  if (extra) {
    const hqekv_migrate_extra &x = *extra;
    const bool columns = x.ring_rows > 0 || x.range_out;
    if (x.ring_rows < 0 || x.res_rows < 0 || x.res_rows > 0x7fffff || x.n_alive < 0 || x.n_alive >= (1 << 24) || x.first_moved < 0 ||
        (columns && !x.alive) || (x.ring_rows > 0 && !x.ring) || (x.range_out && !x.range_in))
      return fail(HQEKV_E_ARG, "cache_migrate: bad eviction or residual arguments");
    for (int k = 0; k < 2 && x.res_rows; ++k)
      if (!x.res_src[k] || !x.res_dst[k] || (((uintptr_t)x.res_src[k] | (uintptr_t)x.res_dst[k]) & 15) || x.res_src_slab[k] < 0 || x.res_dst_slab[k] < x.res_rows)
        return fail(HQEKV_E_ARG, "cache_migrate: the residual rows must be 16-byte aligned and fit their destination");
    a.x = x;
  }
  return launch_migrate(a, BH, D, (hipStream_t)stream);
}

extern "C" int hqekv_fetch_words(const void *host_src, void *dst, int64_t n, void *stream) {
  if (n < 0 || n > 0x7fffff00LL || (n && (!host_src || !dst))) return fail(HQEKV_E_ARG, "fetch_words: null pointer or bad count");
  if (((uintptr_t)host_src | (uintptr_t)dst) & 15) return fail(HQEKV_E_ALIGN, "fetch_words: 16-byte aligned buffers only");
  if (n == 0) return HQEKV_OK;
  hipLaunchKernelGGL(fetch_words_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, (hipStream_t)stream, (const uint32_t *)host_src,
                     (uint32_t *)dst, (int)n);
  return check_launch("fetch_words_kernel");
}
