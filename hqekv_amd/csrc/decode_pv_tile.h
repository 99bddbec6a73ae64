// p.V of a decode step on matrix instructions (see decode_tiles.h): blocks of a class by a workgroup of four waves.
#pragma once

#include "decode_tiles.h"
#include "step_epilogue.h"

#pragma clang fp contract(off)

namespace hq {

// A workgroup takes `per_unit` consecutive blocks of one class: 256 tokens of codes (128 of the 8-bit and fp16
// classes, whose rows are long), 64 (32) per wave.  Lane l owns channels 8 (l % 16) ... + 7 of eight consecutive tokens 8 (l / 16) ... of a step of
// 32, so a step is eight products, one per channel.  Scale and zero rows of the block and its probabilities are staged in
// LDS by the whole workgroup, which gathers the heads' logits at the block's positions, turns them into probabilities,
// writes those back for the caller and parks them.  Several blocks: two buffers, so one barrier per block.
constexpr int PT_WAVES = 4;

template <int BITS>
struct PtGeom {
  static constexpr int STEPS = BITS >= 8 ? 1 : 2;             // per wave and block
  static constexpr int BLOCK = PT_WAVES * 32 * STEPS;
  static constexpr int ROWB = 128 * BITS / 8;                  // bytes per token row
  static constexpr int WPL = BITS == 16 ? 4 : BITS == 8 ? 2 : 1;
};
constexpr int PT_BLOCK = 256;
constexpr int PT_PSTRIDE = PT_BLOCK + 8;   // halves between two heads' probabilities

template <int HP, bool LOOP>
struct PtLds {
  static constexpr int BUFS = LOOP ? 2 : 1;
  uint2 sz[BUFS][PT_BLOCK / 2][4];         // token pair x channel group: (s, s'), (z, z')
  half_t p[BUFS][HP][PT_PSTRIDE];
};

// (max, 1 / sum exp) of a row from its tiles' pairs, by sixteen lanes; up to 64 of them are read at once (past the last one:
// the last one again, left out of the sum)
__device__ __forceinline__ void row16_read(const float2 *sp, int n_stat, int lane, float2 (&sv)[4]) {
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (k == 0 || n_stat > 16 * k) {
      uint32_t w[2];
      load_words<2, Words4<2>>(sp, 8u * (uint32_t)min(lane + 16 * k, n_stat - 1), w);
      sv[k] = make_float2(__builtin_bit_cast(float, w[0]), __builtin_bit_cast(float, w[1]));
    }
}
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, dpp_f<0xB1>(v));
  v = fmaxf(v, dpp_f<0x4E>(v));
  v = fmaxf(v, dpp_f<0x141>(v));
  return fmaxf(v, dpp_f<0x140>(v));
}
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp_f<0xB1>(v);
  v += dpp_f<0x4E>(v);
  v += dpp_f<0x141>(v);
  return v + dpp_f<0x140>(v);
}
__device__ __forceinline__ float2 row16_merge(const float2 *sp, int n_stat, int lane, const float2 (&sv)[4]) {
  float m = sv[0].x;
#pragma unroll
  for (int k = 1; k < 4; ++k)
    if (n_stat > 16 * k) m = fmaxf(m, sv[k].x);
  for (int e = lane + 64; e < n_stat; e += 16) m = fmaxf(m, sp[e].x);
  m = row16_max(m);
  float l = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (k == 0 || n_stat > 16 * k) l += lane + 16 * k < n_stat ? sv[k].y * __expf(sv[k].x - m) : 0.f;
  for (int e = lane + 64; e < n_stat; e += 16) {
    const float2 w = sp[e];
    l += w.y * __expf(w.x - m);
  }
  return make_float2(m, 1.0f / row16_sum(l));
}
// TWICE: the product is rounded to fp32 before it is rounded to fp16, always.  Left to the compiler some places get a mixed
// multiply-add that rounds once: one in some ten thousand probabilities is another fp16 number then, and the ring row would
// not be the sum of the probabilities that the caller sees.
template <bool TWICE>
__device__ __forceinline__ half_t pt_probability(half_t x, float m, float inv_l) {
  float p = __expf((float)x - m) * inv_l;
  if (TWICE) asm("" : "+v"(p));
  return (half_t)p;
}

constexpr int PT_LAST_ROWS = 16;    // partial rows whose loads are in flight together
constexpr int PT_RING_ROWS = 256;   // (b, head) rows of a step whose ring row rides in the p.V launch

// What a thread holds of a block's logits on their way to LDS.  Positions in runs of 32 and an even token count: a pair
// of neighbouring tokens for every other head (thread t: pair t % 128, heads t / 128, t / 128 + 2, ...), one 4-byte access
// each.  Else: token t for every head.
template <int HP>
struct PtValues {
  uint32_t pos;
  uint32_t x[HP];
};

// Where a block's logits come from: the heads' rows in memory, or rows that other workgroups of the same launch have written
// past the L2 (QtRowThrough).
struct PtRows {
  const half_t *rows;
  int64_t Tall;
  __device__ __forceinline__ uint32_t pair(int h, uint32_t off) const {
    uint32_t one[1];
    load_words<1, Words2<1>>(rows + (int64_t)h * Tall, off, one);
    return one[0];
  }
  __device__ __forceinline__ uint32_t single(int h, uint32_t off) const { return gload<uint16_t>(rows + (int64_t)h * Tall, off); }
};
struct PtRowsThrough {
  rsrc_t rows;
  uint32_t first, stride;   // bytes to the first head's row, and between two
  __device__ __forceinline__ uint32_t pair(int h, uint32_t off) const {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rows, (int)(first + (uint32_t)h * stride + off), 0, HQ_THROUGH);
  }
  __device__ __forceinline__ uint32_t single(int h, uint32_t off) const {
    return (uint32_t)(unsigned short)__builtin_amdgcn_raw_buffer_load_b16(rows, (int)(first + (uint32_t)h * stride + off), 0, HQ_THROUGH);
  }
};

// What a thread asks for first, the position of the first of its tokens in a block of the class (pt_class_job's): a form that
// does not depend on the class at compile time.
__device__ __forceinline__ uint32_t pt_first_position(const TileSeg &sg, int block_index, int tid) {
  const uint32_t block = sg.bits >= 8 ? PtGeom<8>::BLOCK : PT_BLOCK, n_tok = (uint32_t)sg.n_tokens;
  const bool paired = qt_runs(sg) && n_tok % 2 == 0;
  return Positions(sg).fetch(min((uint32_t)block_index * block + (paired ? 2u * (tid & (block / 2 - 1)) : (uint32_t)tid), n_tok - 1));
}

// READY: the statistics are merged (ml), and `position` is pt_first_position's.
template <int BITS, int HP, bool EXACT, bool NORMAL, bool LOOP, bool FUSED, bool LAST, bool READY, bool PAIRED, typename Rows, typename StatsLoad, typename StatsMerge>
__device__ __forceinline__ void pt_class_job(const TileSeg &sg, int blk0, int blk1, int bh, int wave, int lane, const Rows &rows, half_t *prows, int64_t Tall,
                                             int nrep_arg, PtLds<HP, LOOP> &lds, const float *ml, f4_t (&acc)[8], uint32_t position0,
                                             StatsLoad &&load_stats, StatsMerge &&merge_stats) {
  using G = PtGeom<BITS>;
  constexpr bool QUANT = BITS != 16;
  constexpr int STEPS = G::STEPS, BLOCK = G::BLOCK, ROWB = G::ROWB, WPL = G::WPL;
  const int nrep = EXACT ? HP : nrep_arg;
  const int n = lane & 15, r = lane >> 4, tid = wave * 64 + lane;
  const uint32_t n_tok = (uint32_t)sg.n_tokens;
  const char *codes = (const char *)sg.data + (int64_t)bh * sg.slab_tokens * ROWB;
  const half_t *sc = QUANT ? sg.scale + (int64_t)bh * sg.slab_tokens * 4 : nullptr;
  const half_t *zr = QUANT ? sg.zero + (int64_t)bh * sg.slab_tokens * 4 : nullptr;
  const Positions position(sg);

  uint32_t cur[STEPS][8][WPL];
  auto load_codes = [&](int blk, uint32_t (&w)[STEPS][8][WPL]) {
    const uint32_t ch = (uint32_t)n * BITS, last = (n_tok - 1) * ROWB + ch;   // tokens past the end repeat the last row, and count with probability zero
    const uint32_t off0 = ((uint32_t)blk * BLOCK + (uint32_t)wave * 32u * STEPS + 8u * r) * ROWB + ch;
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t off = min(off0 + (uint32_t)(32 * s + i) * ROWB, last);
        if constexpr (BITS == 2) {
          w[s][i][0] = gload<uint16_t>(codes, off);
        } else if constexpr (BITS == 1) {
          w[s][i][0] = gload<uint8_t>(codes, off);
        } else {
          load_words<WPL, Words4<WPL>>(codes, off, w[s][i]);
        }
      }
  };
  PtValues<HP> f;
  // thread t in the paired form: pair pt, heads ph, ph + 2, ...
  constexpr int PAIRS = BLOCK / 2, HSTEP = PT_WAVES * 64 / PAIRS, PHEADS = HP / HSTEP > 0 ? HP / HSTEP : 1;
  static_assert(HP % HSTEP == 0, "heads are dealt evenly");
  const int pt = tid % PAIRS, ph = tid / PAIRS;
  auto fetch_position = [&](int blk) {
    f.pos = position.fetch(min((uint32_t)blk * BLOCK + (PAIRED ? 2u * pt : (uint32_t)tid), n_tok - 1));
  };
  auto fetch_values = [&](int blk) {
    const uint32_t t = min((uint32_t)blk * BLOCK + (PAIRED ? 2u * pt : (uint32_t)tid), n_tok - 1);
    f.pos = 2u * position.of(t, f.pos);   // byte offset in a row
    if constexpr (PAIRED) {
      // (past the end: the class's last pair once more.  min() above gives its second token: one step back)
      f.pos -= t == n_tok - 1 ? 2u : 0u;
#pragma unroll
      for (int k = 0; k < PHEADS; ++k) {
        const int h = ph + k * HSTEP;
        f.x[k] = rows.pair(EXACT ? h : min(h, nrep - 1), f.pos);
      }
    } else {
#pragma unroll
      for (int h = 0; h < HP; ++h)
        if (h < nrep) f.x[h] = rows.single(h, f.pos);
    }
  };
  uint32_t sa[2], sb[2], za[2], zb[2];
  auto fetch_scales = [&](int blk) {
    if (QUANT && tid < BLOCK / 2) {
      const uint32_t a = min((uint32_t)blk * BLOCK + 2u * tid, n_tok - 1), b = min(a + 1, n_tok - 1);
      load_words<2, Words4<2>>(sc, a * 8u, sa);
      load_words<2, Words4<2>>(sc, b * 8u, sb);
      load_words<2, Words4<2>>(zr, a * 8u, za);
      load_words<2, Words4<2>>(zr, b * 8u, zb);
    }
  };
  // fused: the row holds scaled logits: p = rnd16(exp(x - M) / L), written back for the caller.  Every position belongs to
  // exactly one token of exactly one V class, so nobody else touches it.
  auto probability = [&](half_t x, int h) { return FUSED ? pt_probability<LAST>(x, ml[2 * h], ml[2 * h + 1]) : x; };
  auto commit = [&](int blk, int buf) {
    if constexpr (PAIRED) {
      const bool valid = (uint32_t)blk * BLOCK + 2u * pt < n_tok;
#pragma unroll
      for (int k = 0; k < PHEADS; ++k) {
        const int h = ph + k * HSTEP;
        if (EXACT || h < nrep) {
          const half2_t x = as_h2(f.x[k]);
          const uint32_t p = as_u32(pack_h2(probability(x[0], h), probability(x[1], h)));
          if (FUSED && valid) {
            Words2<1> w;
            w.v[0] = p;
            gstore(prows + (int64_t)h * Tall, f.pos, w);
          }
          *reinterpret_cast<uint32_t *>(&lds.p[buf][h][2 * pt]) = valid ? p : 0u;
        }
      }
    } else if (tid < BLOCK) {
      const bool valid = (uint32_t)blk * BLOCK + tid < n_tok;
#pragma unroll
      for (int h = 0; h < HP; ++h)
        if (h < nrep) {
          const half_t p = probability(__builtin_bit_cast(half_t, (uint16_t)f.x[h]), h);
          if (FUSED && valid) gstore(prows + (int64_t)h * Tall, f.pos, p);
          lds.p[buf][h][tid] = valid ? p : (half_t)0;
        }
    }
    if (QUANT && tid < BLOCK / 2) {
      uint32_t v[8];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        v[2 * g] = (g & 1) ? as_u32(half_pair<1>(sa[g >> 1], sb[g >> 1])) : as_u32(half_pair<0>(sa[g >> 1], sb[g >> 1]));
        v[2 * g + 1] = (g & 1) ? as_u32(half_pair<1>(za[g >> 1], zb[g >> 1])) : as_u32(half_pair<0>(za[g >> 1], zb[g >> 1]));
      }
      // Tokens past the end hold the last row's codes and probability zero; with scale and zero point zero too they are
      // zeros, where an infinity in the last row would be 0 x inf.  Only in a block that ends short: masks in every block cost
      // a step at 32k tokens 0.2 us (19.6 -> 19.8), these 0.1, and nothing at 8 x 64k (masks everywhere: 152.4 -> 152.9).
      if ((uint32_t)(blk + 1) * BLOCK > n_tok) {
        const uint32_t left = n_tok - min((uint32_t)blk * BLOCK + 2u * tid, n_tok), mask = (left > 0 ? 0xffffu : 0u) | (left > 1 ? 0xffff0000u : 0u);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] &= mask;
      }
      uint4 *dst = reinterpret_cast<uint4 *>(lds.sz[buf][tid]);
      dst[0] = make_uint4(v[0], v[1], v[2], v[3]);
      dst[1] = make_uint4(v[4], v[5], v[6], v[7]);
    }
  };

  // The longest chain of dependent loads is position -> logit: it goes first, with the statistics beside it (code words
  // asked for ahead of the logits would queue in front of them).
  if constexpr (READY) f.pos = position0;
  else fetch_position(blk0);
  load_stats();
  fetch_values(blk0);
  HQ_LOADS_ABOVE();
  fetch_scales(blk0);
  load_codes(blk0, cur);
  HQ_LOADS_ABOVE();
  merge_stats();
  commit(blk0, 0);
  if (LOOP && blk0 + 1 < blk1) fetch_position(blk0 + 1);
  __syncthreads();
#pragma unroll 1
  for (int blk = blk0; blk < (LOOP ? blk1 : blk0 + 1); ++blk) {
    const int buf = LOOP ? (blk - blk0) & 1 : 0;
    const bool more = LOOP && blk + 1 < blk1;
    uint32_t nxt[STEPS][8][WPL];
    if (more) {
      fetch_values(blk + 1);
      load_codes(blk + 1, nxt);
      fetch_scales(blk + 1);
    }
    HQ_LOADS_ABOVE();
    if (!QUANT && (uint32_t)(blk + 1) * BLOCK > n_tok) {   // (rows past the end: zeros, as commit() makes of codes)
#pragma unroll
      for (int s = 0; s < STEPS; ++s)
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int k = 0; k < WPL; ++k)
            cur[s][i][k] = (uint32_t)blk * BLOCK + (uint32_t)((wave * STEPS + s) * 32 + 8 * r + i) < n_tok ? cur[s][i][k] : 0u;
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int t = (wave * STEPS + s) * 32 + 8 * r;   // this lane's first token of the step, inside the block
      const u32x4 a = *reinterpret_cast<const u32x4 *>(&lds.p[buf][min(n, nrep - 1)][t]);
      half2_t s2[4], z2[4];
      if constexpr (QUANT) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint2 e = lds.sz[buf][t / 2 + i][n >> 2];
          s2[i] = as_h2(e.x);
          z2[i] = as_h2(e.y);
          if (NORMAL) s2[i] = normal1_spread(s2[i]);
        }
        constexpr int B = BITS == 16 ? 8 : BITS;   // (named for the discarded instantiation)
        static_for<B>([&](auto K_) {   // byte K of a lane's channels
          constexpr int K = decltype(K_)::value;
          uint32_t u[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) u[i] = byte_pair<K % 4>(cur[s][2 * i][K / 4 % WPL], cur[s][2 * i + 1][K / 4 % WPL]);
          static_for<8 / B>([&](auto F_) {
            constexpr int F = decltype(F_)::value, C = K * (8 / B) + F;
            u32x4 b;
#pragma unroll
            for (int i = 0; i < 4; ++i) b[i] = as_u32(dequant_field<B, F, NORMAL>(u[i], s2[i], z2[i]));
            acc[C] = mfma16(a, b, acc[C]);
          });
        });
      } else {
        static_for<8>([&](auto C_) {
          constexpr int C = decltype(C_)::value;
          u32x4 b;
#pragma unroll
          for (int i = 0; i < 4; ++i) b[i] = as_u32(half_pair<C & 1>(cur[s][2 * i][C / 2 % WPL], cur[s][2 * i + 1][C / 2 % WPL]));
          acc[C] = mfma16(a, b, acc[C]);
        });
      }
    }
    if (more) {
      commit(blk + 1, buf ^ 1);
      if (blk + 2 < blk1) fetch_position(blk + 2);
#pragma unroll
      for (int s = 0; s < STEPS; ++s)
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int k = 0; k < WPL; ++k) cur[s][i][k] = nxt[s][i][k];
      __syncthreads();
    }
  }
}

// The same for a unit of whatever class.
template <int HP, bool EXACT, bool LOOP, bool FUSED, bool LAST, bool READY, typename Rows, typename StatsLoad, typename StatsMerge>
__device__ __forceinline__ void pt_unit(const TileSeg &sg, int unit, int per, int bh, int wave, int lane, const Rows &rows, half_t *prows, int64_t Tall, int nrep,
                                        PtLds<HP, LOOP> &lds, const float *ml, f4_t (&acc)[8], uint32_t position0, StatsLoad &&load_stats, StatsMerge &&merge_stats) {
  const int b0 = unit * per;
  const bool paired = qt_runs(sg) && sg.n_tokens % 2 == 0;
#define HQ_JOB_P(B_, NORMAL_, PAIRED_)                                                                                                                   \
  pt_class_job<B_, HP, EXACT, NORMAL_, LOOP, FUSED, LAST, READY, PAIRED_>(                                                                               \
      sg, b0, min(b0 + per, (int)((sg.n_tokens + PtGeom<B_>::BLOCK - 1) / PtGeom<B_>::BLOCK)), bh, wave, lane, rows, prows, Tall, nrep, lds, ml, acc, \
      position0, load_stats, merge_stats)
#define HQ_JOB(B_, NORMAL_)                  \
  do {                                       \
    if (paired) HQ_JOB_P(B_, NORMAL_, true); \
    else HQ_JOB_P(B_, NORMAL_, false);       \
  } while (0)
  switch (sg.bits) {
    case 1:
      if ((sg.layout & 3) == HQEKV_LAYOUT_NORMAL1) HQ_JOB(1, true);
      else HQ_JOB(1, false);
      break;
    case 2: HQ_JOB(2, false); break;
    case 4: HQ_JOB(4, false); break;
    case 8: HQ_JOB(8, false); break;
    default: HQ_JOB(16, false);
  }
#undef HQ_JOB
#undef HQ_JOB_P
}

// What a unit leaves: the heads' sums over its tokens, of the four waves in order; `store` takes two channels, at pair
// 64 head + channel / 2.
template <int HP, bool EXACT, typename Store>
__device__ __forceinline__ void pt_store_partial(const f4_t (&acc)[8], float (&red)[PT_WAVES][HP][128], int wave, int lane, int nrep, Store &&store) {
  // lane l holds heads 4 (l / 16) ... + 3 of channels 8 (l % 16) ... + 7
  const int n = lane & 15, r = lane >> 4;
  if (4 * r < HP) {
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      float4 *to = reinterpret_cast<float4 *>(&red[wave][4 * r + h][8 * n]);
      to[0] = make_float4(acc[0][h], acc[1][h], acc[2][h], acc[3][h]);
      to[1] = make_float4(acc[4][h], acc[5][h], acc[6][h], acc[7][h]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = wave * 64 + lane; k < (EXACT ? HP : nrep) * 64; k += PT_WAVES * 64) {
    const int h = k >> 6, c = 2 * (k & 63);
    float2 v[PT_WAVES];
#pragma unroll
    for (int w = 0; w < PT_WAVES; ++w) v[w] = *reinterpret_cast<const float2 *>(&red[w][h][c]);
    const float2 sum = make_float2(((v[0].x + v[1].x) + v[2].x) + v[3].x, ((v[0].y + v[1].y) + v[2].y) + v[3].y);
    store(k, sum);
  }
}

// The sum of what `units` units have left there, by one workgroup: `partial` and `out` from the (b, kv head)'s first head on.
// 16 bytes of a row per lane, the even and the odd rows apart (HP = 4: by one half of the workgroup each).
template <int HP, bool EXACT>
__device__ __forceinline__ void pt_sum_partials(const float *partial, uint32_t n_bhq, int units, int nrep, float *half, half_t *out) {
  constexpr int LANES = HP * 32, GROUPS = PT_WAVES * 64 / LANES;
  static_assert(GROUPS >= 1, "a row in one go");
  const int at = threadIdx.x % LANES, g = threadIdx.x / LANES;
  const bool mine = EXACT || at < nrep * 32;
  const uint32_t row_b = n_bhq * 512u;   // (the rows of a short launch span a few MB)
  const rsrc_t rows_of = make_rsrc(partial, (uint32_t)(units - 1) * row_b + (uint32_t)nrep * 512u);
  f4_t v = (f4_t){0.f, 0.f, 0.f, 0.f}, odd = v;
  if (mine) {
    for (int c0 = 0; c0 < units; c0 += GROUPS * PT_LAST_ROWS) {
      f4_t t[PT_LAST_ROWS];
      static_for<PT_LAST_ROWS>([&](auto I_) {   // (past the last row: zeros, without a trip to memory)
        constexpr int I = decltype(I_)::value;
        t[I] = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(rows_of, 16 * at + (c0 + GROUPS * I + g) * (int)row_b, 0, HQ_THROUGH));
      });
      static_for<PT_LAST_ROWS>([&](auto I_) {
        constexpr int I = decltype(I_)::value;
        (GROUPS == 1 && I % 2 ? odd : v) += t[I];
      });
    }
  }
  static_assert(GROUPS <= 2 && PT_LAST_ROWS % 2 == 0, "two sums");
  if constexpr (GROUPS == 1) v += odd;
  if constexpr (GROUPS > 1) {
    if (g == 1 && mine) *reinterpret_cast<f4_t *>(half + 4 * at) = v;
    __syncthreads();
    if (g == 0 && mine) v += *reinterpret_cast<const f4_t *>(half + 4 * at);
  }
  if (g == 0 && mine) {
    const uint2 w = make_uint2(as_u32(pack_h2((half_t)v[0], (half_t)v[1])), as_u32(pack_h2((half_t)v[2], (half_t)v[3])));
    *reinterpret_cast<uint2 *>(out + 4 * at) = w;
  }
}

struct PtEpilogue {
  half_t ring[RING_LDS_HEADS * RING_SPAN_SHORT];
  float2 ml[PT_RING_ROWS];   // (max, 1 / sum exp) of every (b, head) row
};
// The ring row's probabilities out of the logits; THROUGH as for PtRowsThrough.
template <bool THROUGH_>
struct PtRingProb {
  static constexpr bool THROUGH = THROUGH_;
  const float2 *ml;
  __device__ __forceinline__ uint64_t operator()(int row, uint64_t quad) const {
    const float2 s = ml[row];
    uint64_t v = 0;
#pragma unroll
    for (int i = 0; i < RING_V; ++i)
      v |= (uint64_t)__builtin_bit_cast(uint16_t, pt_probability<true>(__builtin_bit_cast(half_t, (uint16_t)(quad >> (16 * i))), s.x, s.y)) << (16 * i);
    return v;
  }
};

}  // namespace hq
