// q.K^T of a decode step on matrix instructions (see decode_tiles.h): one tile of a class by a workgroup of four waves.
#pragma once

#include "decode_tiles.h"

#pragma clang fp contract(off)

namespace hq {

// A workgroup of four waves takes one tile of one class of one (b, kv head): 256 tokens of codes (128 of the fp16 class)
// and all of head_dim.  Wave w owns channels 32 w ... + 31; lane l holds, of eight of them, the code words of 16 (8)
// consecutive tokens -- one load of one, two or four words per channel, all requested at once -- so the four heads or bands
// of its column end up with four (HP) consecutive tokens each, whatever the class.  The four partial sums meet in LDS,
// after which wave w finishes one head of every lane's four.
//
// What bounds it: the serial life of a wave in a short launch, vector instructions in a long one.  Hence equal tokens (not
// bytes) per wave: a wave spends about 270 instructions on dequantising 256 x 32 codes and 200 around them.  With tiles
// of equal bytes (256 tokens at 2 bit ... 32 at fp16) a 32k-token cache took 7800 waves instead of 3500, two thirds of
// whose instructions were overhead, and asked for every line of the scale planes eight times (TA 63 % busy): 11.8 us.
// Scale rows are fetched wide, 8 groups per lane and channel, by each wave for its own channels.
constexpr int QT_WAVES = 4;

template <int BITS>
struct QtGeom {
  static constexpr int TOK = BITS == 16 ? 8 : 16;        // tokens per lane column
  static constexpr int TILE = 16 * TOK;
  static constexpr int COLB = TOK * BITS / 8;            // bytes of a column in one channel row: 2 ... 16
  static constexpr int NW = COLB < 4 ? 1 : COLB / 4;     // words that hold it
};
constexpr int QT_NG = 8;     // 32-token groups per tile
constexpr int QT_NGP = 10;   // LDS row of a channel pair, in 8-byte entries: padded, the four lane groups of a read meet different banks

// A wave's corner of LDS: the scales and zeros of its channels while it multiplies -- (channel pair, group): (s, s'), (z, z')
// -- and its partial scores afterwards: head of the lane's four, four tokens at a time, lane.
template <int HP>
struct QtLds {
  char bytes[QT_WAVES][4 * HP * 64 * 4];
  static_assert(4 * HP * 64 * 4 >= 16 * QT_NGP * 8, "one corner serves both");
  __device__ __forceinline__ uint2 *sz(int wave) { return reinterpret_cast<uint2 *>(bytes[wave]); }
  __device__ __forceinline__ float *part(int wave, int head) { return reinterpret_cast<float *>(bytes[wave]) + head * HP * 64; }
};

// One score element by element.  Tokens of different bands share an accumulator, with zeros in the others' rows of A: a key
// that is not finite (or overflows in its group's scale) makes 0 x inf = NaN of up to three other tokens' sums.  A tile
// with a NaN among its sums -- never, in a cache of numbers -- takes those scores again here, each token to itself.  The
// test is one addition per score (a step at 32k tokens 19.72 -> 19.80 us, at 3 x 16k with five heads per KV head 25.34 ->
// 25.50, at 8 x 64k 152.1 -> 151.9); a select per lane after products without bands would cost four times the accumulators.
template <int BITS, bool NORMAL, bool ROWS>
__device__ __forceinline__ float qk_alone(const TileSeg &sg, int bh, uint32_t token, const half_t *q) {
  const uint32_t n_tok = (uint32_t)sg.n_tokens;
  float sum = 0.f;
#pragma unroll 1
  for (int c = 0; c < 128; ++c) {
    half_t x;
    const int64_t row = (int64_t)bh * 128 + c;
    if constexpr (ROWS) {
      x = gload<half_t>((const half_t *)sg.data + (int64_t)bh * sg.slab_tokens * 128, token * 256u + 2u * c);
    } else if constexpr (BITS == 16) {
      x = gload<half_t>((const half_t *)sg.data + row * n_tok, token * 2u);
    } else {
      const uint8_t byte = gload<uint8_t>((const char *)sg.data + row * (n_tok * BITS / 8), token * BITS / 8);
      const half_t code = (half_t)(unsigned short)((byte >> (token * BITS & 7)) & ((1 << BITS) - 1));
      const int64_t g = row * (n_tok / 32) + token / 32;
      const half2_t c2 = {code, code}, s2 = {sg.scale[g], sg.scale[g]}, z2 = {sg.zero[g], sg.zero[g]};
      x = (NORMAL ? dequant_pair_normal1(c2, normal1_spread(s2), z2) : dequant_pair(c2, s2, z2))[0];
    }
    sum += (float)x * (float)gload<half_t>(q, 2u * c);
  }
  return sum;
}

// Where a tile's scores go: a head's row in memory -- or, where other workgroups of the same launch read them, through the L2
// (which the XCDs do not share) to memory.
struct QtRow {
  half_t *row;
  template <int N>
  __device__ __forceinline__ void store(uint32_t pos, const half_t (&x)[N]) const {
    struct __attribute__((packed, aligned(2))) Run { half_t v[N]; };
    Run r;
#pragma unroll
    for (int t = 0; t < N; ++t) r.v[t] = x[t];
    gstore(row, pos * 2u, r);
  }
};
struct QtRowThrough {
  rsrc_t rows;
  uint32_t row;   // bytes to the head's row
  template <int N>
  __device__ __forceinline__ void store(uint32_t pos, const half_t (&x)[N]) const {
    const int at = (int)(row + pos * 2u);
    if constexpr (N == 1) {
      __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, x[0]), rows, at, 0, HQ_THROUGH);
    } else {
      uint32_t w[N / 2];
#pragma unroll
      for (int t = 0; t < N / 2; ++t) w[t] = as_u32(pack_h2(x[2 * t], x[2 * t + 1]));
      if constexpr (N == 2) __builtin_amdgcn_raw_buffer_store_b32(w[0], rows, at, 0, HQ_THROUGH);
      else if constexpr (N == 4) __builtin_amdgcn_raw_buffer_store_b64((u32x2){w[0], w[1]}, rows, at, 0, HQ_THROUGH);
      else {
#pragma unroll
        for (int k = 0; k < N / 8; ++k)
          __builtin_amdgcn_raw_buffer_store_b128((u32x4){w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]}, rows, at + 16 * k, 0, HQ_THROUGH);
      }
    }
  }
};

// The end of a tile: the partial sums of this wave's head are added up in order, rounded, scaled, stored, and turned into
// the lane's (max, sum exp).  `pos(t)`: position of the lane's token t, the first `n_valid` of which exist; `run`: they
// are consecutive; `alone(t)`: its score once more.
template <int HP, bool FUSED, int TPV, typename Row, typename Pos, typename Alone>
__device__ __forceinline__ void qt_finish_tile(QtLds<HP> &lds, const f4_t (&acc)[TPV], int wave, int lane, Pos &&pos, int n_valid, bool run,
                                               const Row &row, float inv_sqrt_d, float &m_lane, float &l_lane, Alone &&alone) {
  constexpr int P = TPV < 4 ? TPV : 4;   // tokens side by side
#pragma unroll
  for (int h = 0; h < 4; ++h)
#pragma unroll
    for (int t = 0; t < TPV; ++t) lds.part(wave, h)[(t / P) * 64 * P + lane * P + t % P] = acc[t][h];
  __syncthreads();
  half_t x[TPV];
  float m = SM_FLOOR, sum[TPV], all = 0.f;
#pragma unroll
  for (int t = 0; t < TPV; ++t) {
    const int at = (t / P) * 64 * P + lane * P + t % P;
    sum[t] = ((lds.part(0, wave)[at] + lds.part(1, wave)[at]) + lds.part(2, wave)[at]) + lds.part(3, wave)[at];
    all += sum[t];
  }
  if (HP < 16 && __builtin_expect(__builtin_amdgcn_ballot_w64(all != all && n_valid > 0) != 0, 0)) {
#pragma unroll 1
    for (int t = 0; t < n_valid; ++t) {
      bool bad = false;
#pragma unroll
      for (int k = 0; k < TPV; ++k) bad = bad || (k == t && sum[k] != sum[k]);
      const float again = bad ? alone(t) : 0.f;
#pragma unroll
      for (int k = 0; k < TPV; ++k) sum[k] = k == t && bad ? again : sum[k];
    }
  }
#pragma unroll
  for (int t = 0; t < TPV; ++t) {
    x[t] = (half_t)sum[t];
    if (FUSED) {   // the fp16 steps of the reference epilogue: round the score, scale, round again
      x[t] = (half_t)((float)x[t] * inv_sqrt_d);
      m = fmaxf(m, t < n_valid ? (float)x[t] : SM_FLOOR);
    }
  }
  if (TPV > 1 && run && n_valid >= TPV) {
    row.store(pos(0), x);
  } else {
#pragma unroll
    for (int t = 0; t < TPV; ++t)
      if (t < n_valid) row.store(pos(t), {x[t]});
  }
  if (FUSED) {
    float l = 0.f;
#pragma unroll
    for (int t = 0; t < TPV; ++t) l += t < n_valid ? __expf((float)x[t] - m) : 0.f;
    m_lane = m;
    l_lane = l;
  }
}

template <int BITS, int HP, bool FUSED, bool NORMAL, typename Row, typename QueryRow>
__device__ __forceinline__ void qt_class_tile(const TileSeg &sg, int tile, int bh, int n_bh, int wave, int lane, u32x4 q, QtLds<HP> &lds,
                                              const Row &row, bool has_head, float inv_sqrt_d, float &m, float &l, QueryRow &&qrow) {
  using G = QtGeom<BITS>;
  constexpr bool QUANT = BITS != 16;
  constexpr int BANDS = 16 / HP, TPV = G::TOK / BANDS > 0 ? G::TOK / BANDS : 1;   // tokens a lane ends up with = accumulators
  static_assert(TPV * BANDS == G::TOK, "whole tokens per band");
  constexpr int PF = BITS == 16 ? 2 : 32 / BITS;
  const int n = lane & 15, r = lane >> 4;
  const uint32_t n_tok = (uint32_t)sg.n_tokens, row_b = n_tok * BITS / 8;   // (a multiple of the column width)
  const uint32_t col0 = (uint32_t)tile * G::TILE + G::TOK * n;              // first token of the lane's column
  const int band = (4 * r) / HP;
  const bool runs = qt_runs(sg) && n_tok % 32 == 0;
  const Positions position(sg);

  // ---- scales (lanes 0 - 31) and zeros of channel l % 32 of this wave's: the tile's eight groups.  What lies past the row's
  // end is never used; at the plane's end the window is moved back so that it stays inside.
  const uint32_t Gn = n_tok / 32, g0 = (uint32_t)tile * QT_NG;
  const int64_t at = ((int64_t)bh * 128 + 32 * wave + (lane & 31)) * Gn + g0, from = min(at, (int64_t)n_bh * 128 * Gn - QT_NG);
  uint32_t sw[4];
  if constexpr (QUANT) load_words<4, Words2<4>>((lane < 32 ? sg.scale : sg.zero) + from, 0u, sw);
  // ---- code words (a column past the row's end repeats the last one, unused)
  const char *codes = (const char *)sg.data + ((int64_t)bh * 128 + 32 * wave) * row_b;
  uint32_t cur[8][G::NW];
  {
    const uint32_t off = 8u * r * row_b + min(col0, n_tok - G::TOK) * BITS / 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if constexpr (BITS == 1) {
        cur[i][0] = gload<uint16_t>(codes, off + i * row_b);
      } else {
        load_words<G::NW, Words2<G::NW>>(codes, off + i * row_b, cur[i]);
      }
    }
  }
  const uint32_t tok0 = col0 + band * TPV;   // this lane's first token
  const int n_valid = has_head && tok0 < n_tok ? TPV : 0;
  // (a lane's tokens never cross a run: TPV divides 32 and tok0; without runs the positions are read when they are needed)
  const uint32_t tok0c = min(tok0, n_tok - 1), index0 = position.fetch(tok0c);
  HQ_LOADS_ABOVE();
  half2_t s2[4], z2[4];
  if constexpr (QUANT) {
    for (uint32_t back = (uint32_t)(at - from); back; --back) {   // a moved window (the plane's last rows): down to where it belongs
#pragma unroll
      for (int w = 0; w < 4; ++w) sw[w] = sw[w] >> 16 | (w < 3 ? sw[(w + 1) % 4] << 16 : 0u);
    }
    uint16_t *e = reinterpret_cast<uint16_t *>(lds.sz(wave)) + ((lane & 31) >> 1) * (QT_NGP * 4) + (lane & 1) + (lane < 32 ? 0 : 2);
#pragma unroll
    for (int g = 0; g < QT_NG; ++g) e[4 * g] = (uint16_t)(g & 1 ? sw[g / 2] >> 16 : sw[g / 2]);
    wave_lds_fence();
    const uint32_t gi = min((uint32_t)n / 2, Gn - 1 - g0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint2 v = lds.sz(wave)[(4 * r + i) * QT_NGP + gi];
      s2[i] = as_h2(v.x);
      z2[i] = as_h2(v.y);
      if (NORMAL) s2[i] = normal1_spread(s2[i]);
    }
    wave_lds_fence();   // (the partial scores come to lie where these were)
  }
  f4_t acc[TPV];
#pragma unroll
  for (int t = 0; t < TPV; ++t) acc[t] = (f4_t){0.f, 0.f, 0.f, 0.f};
  u32x4 a;   // the query in one band of A only (made where it is used: four copies would cost sixteen registers)
  auto into_band = [&](int j) {
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = BANDS == 1 || n / HP == j ? q[i] : 0u;
  };
  static_for<(BITS == 16 ? 4 : G::COLB)>([&](auto K_) {   // a byte of eight bits' worth of tokens; a word of two at fp16
    constexpr int K = decltype(K_)::value;
    __builtin_amdgcn_sched_barrier(0);   // (the operands of one byte's tokens at a time)
    if constexpr (QUANT) {
      constexpr int B = BITS == 16 ? 8 : BITS;   // (named for the discarded instantiation)
      uint32_t u[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) u[i] = byte_pair<K % 4>(cur[2 * i][K / 4 % G::NW], cur[2 * i + 1][K / 4 % G::NW]);
      static_for<8 / B>([&](auto F_) {
        constexpr int F = decltype(F_)::value, TOK = K * (8 / B) + F;
        if (TOK % TPV == 0) into_band(TOK / TPV);
        u32x4 b;
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = as_u32(dequant_field<B, F, NORMAL>(u[i], s2[i], z2[i]));
        acc[TOK % TPV] = mfma16(a, b, acc[TOK % TPV]);
      });
    } else {
      static_for<2>([&](auto H_) {
        constexpr int H = decltype(H_)::value, TOK = 2 * K + H;
        if (TOK % TPV == 0) into_band(TOK / TPV);
        u32x4 b;
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = as_u32(half_pair<H>(cur[2 * i][K % G::NW], cur[2 * i + 1][K % G::NW]));
        acc[TOK % TPV] = mfma16(a, b, acc[TOK % TPV]);
      });
    }
  });
  qt_finish_tile<HP, FUSED, TPV>(lds, acc, wave, lane, [&](int t) { return runs ? position.of(tok0c, index0) + t : position(tok0 + t); }, n_valid,
                                 runs, row, inv_sqrt_d, m, l, [&](int t) { return qk_alone<BITS, NORMAL, false>(sg, bh, tok0 + t, qrow()); });
}

// fp16 K rows stored token by token (the residual, a step's own key): four blocks of 16 tokens; lane l reads 16 bytes of
// token l % 16 of every block -- already a B operand.
constexpr int QT_TM_TILE = 64;

template <int HP, bool FUSED, typename Row, typename QueryRow>
__device__ __forceinline__ void qt_rows_tile(const TileSeg &sg, int tile, int bh, int wave, int lane, u32x4 q, QtLds<HP> &lds, const Row &row,
                                             bool has_head, float inv_sqrt_d, float &m, float &l, QueryRow &&qrow) {
  constexpr int BANDS = 16 / HP, TPV = 4 / BANDS;
  const int n = lane & 15, r = lane >> 4;
  const uint32_t n_tok = (uint32_t)sg.n_tokens;
  const char *src = (const char *)sg.data + (int64_t)bh * sg.slab_tokens * 256 + 64 * wave;
  const int band = (4 * r) / HP;
  const uint32_t t0 = (uint32_t)tile * QT_TM_TILE;
  auto token = [&](int t) { return t0 + 16u * (band * TPV + t) + n; };   // block band * TPV + t
  const Positions position(sg);
  f4_t acc[TPV];
#pragma unroll
  for (int t = 0; t < TPV; ++t) acc[t] = (f4_t){0.f, 0.f, 0.f, 0.f};
  u32x4 x[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) x[k] = gload<u32x4>(src, min(t0 + 16u * k + n, n_tok - 1) * 256u + 16u * r);
  int n_valid = 0;
#pragma unroll
  for (int t = 0; t < TPV; ++t) n_valid += has_head && token(t) < n_tok ? 1 : 0;   // (blocks ascend: the valid ones come first)
  static_for<4>([&](auto K_) {
    constexpr int K = decltype(K_)::value;
    u32x4 a;
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = BANDS == 1 || n / HP == K / TPV ? q[i] : 0u;
    acc[K % TPV] = mfma16(a, x[K], acc[K % TPV]);
  });
  qt_finish_tile<HP, FUSED, TPV>(lds, acc, wave, lane, [&](int t) { return position(token(t)); }, n_valid, false, row, inv_sqrt_d, m, l,
                                 [&](int t) { return qk_alone<16, false, true>(sg, bh, token(t), qrow()); });
}

// A tile of whatever class, and with it (max, sum exp) of each head's scores, in every lane of the row of 16 that holds the head.
template <int HP, bool FUSED, typename Row, typename QueryRow>
__device__ __forceinline__ void qt_unit(const TileSeg &sg, int tile, int bh, int n_bh, int wave, int lane, u32x4 q, QtLds<HP> &lds, const Row &row,
                                        bool has_head, float inv_sqrt_d, float &mm, float &l, QueryRow &&qrow) {
  float m = SM_FLOOR;
  l = 0.f;
#define HQ_TILE(B_, NORMAL_) qt_class_tile<B_, HP, FUSED, NORMAL_>(sg, tile, bh, n_bh, wave, lane, q, lds, row, has_head, inv_sqrt_d, m, l, qrow)
  switch (sg.bits) {
    case 1:
      if ((sg.layout & 3) == HQEKV_LAYOUT_NORMAL1) HQ_TILE(1, true);
      else HQ_TILE(1, false);
      break;
    case 2: HQ_TILE(2, false); break;
    case 4: HQ_TILE(4, false); break;
    case 8: HQ_TILE(8, false); break;
    default:
      if ((sg.layout & 3) == HQEKV_LAYOUT_TOKEN_MAJOR) qt_rows_tile<HP, FUSED>(sg, tile, bh, wave, lane, q, lds, row, has_head, inv_sqrt_d, m, l, qrow);
      else HQ_TILE(16, false);
  }
#undef HQ_TILE
  if (!FUSED) return;
  // lanes of a row of 16 hold the same head; so do the rows r and r' with the same 4 r % HP
  mm = m;
  mm = fmaxf(mm, dpp_f<0xB1>(mm));
  mm = fmaxf(mm, dpp_f<0x4E>(mm));
  mm = fmaxf(mm, dpp_f<0x141>(mm));
  mm = fmaxf(mm, dpp_f<0x140>(mm));
  if (HP <= 4) mm = fmaxf(mm, xor_f(mm, 16));
  if (HP <= 8) mm = fmaxf(mm, xor_f(mm, 32));
  l = m == mm ? l : l * __expf(m - mm);   // (a lane that saw no token: l = 0, m the floor)
  l += dpp_f<0xB1>(l);
  l += dpp_f<0x4E>(l);
  l += dpp_f<0x141>(l);
  l += dpp_f<0x140>(l);
  if (HP <= 4) l += xor_f(l, 16);
  if (HP <= 8) l += xor_f(l, 32);
}

}  // namespace hq
