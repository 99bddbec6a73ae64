// q.K^T of a decode step on matrix instructions (see decode_tiles.h), and how the decode launches are cut up.
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

// The end of a tile: the partial sums of this wave's head are added up in order, rounded, scaled, stored, and turned into
// the lane's (max, sum exp).  `pos(t)`: position of the lane's token t, the first `n_valid` of which exist; `run`: they
// are consecutive; `alone(t)`: its score once more.
template <int HP, bool FUSED, int TPV, typename Pos, typename Alone>
__device__ __forceinline__ void qt_finish_tile(QtLds<HP> &lds, const f4_t (&acc)[TPV], int wave, int lane, Pos &&pos, int n_valid, bool run,
                                               half_t *row, float inv_sqrt_d, float &m_lane, float &l_lane, Alone &&alone) {
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
    struct __attribute__((packed, aligned(2))) Run { half_t v[TPV]; };
    Run r;
#pragma unroll
    for (int t = 0; t < TPV; ++t) r.v[t] = x[t];
    gstore(row, pos(0) * 2u, r);
  } else {
#pragma unroll
    for (int t = 0; t < TPV; ++t)
      if (t < n_valid) gstore(row, pos(t) * 2u, x[t]);
  }
  if (FUSED) {
    float l = 0.f;
#pragma unroll
    for (int t = 0; t < TPV; ++t) l += t < n_valid ? __expf((float)x[t] - m) : 0.f;
    m_lane = m;
    l_lane = l;
  }
}

template <int BITS, int HP, bool FUSED, bool NORMAL, typename QueryRow>
__device__ __forceinline__ void qt_class_tile(const TileSeg &sg, int tile, int bh, int n_bh, int wave, int lane, u32x4 q, QtLds<HP> &lds,
                                              half_t *row, bool has_head, float inv_sqrt_d, float &m, float &l, QueryRow &&qrow) {
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

template <int HP, bool FUSED, typename QueryRow>
__device__ __forceinline__ void qt_rows_tile(const TileSeg &sg, int tile, int bh, int wave, int lane, u32x4 q, QtLds<HP> &lds, half_t *row,
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

// COUNT: the p.V launch of the same call counts arrivals, from zero (a form of its own: a test for it costs every launch a
// scalar load in its prologue, 0.3 us of a step at 32k tokens).
template <int HP, bool FUSED, bool COUNT>
__global__ __launch_bounds__(QT_WAVES * 64, HP == 16 ? 2 : HP == 4 || FUSED ? 5 : 4) void qk_tiles_kernel(
    u32x4 begins, const half_t *__restrict__ q, half_t *__restrict__ scores, float2 *__restrict__ stats, uint32_t heads, uint32_t div_hkv, int64_t Tall,
    int32_t n_bh, int32_t n_stat, float inv_sqrt_d, uint32_t *__restrict__ arrive, TileTable tb) {
  __shared__ __align__(16) QtLds<HP> lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int bh = blockIdx.x, u = (int)blockIdx.y;
  const TileSeg sg = tb.seg[tiles_segment(begins, u)];
  const int Hq = heads & 0xffffu, Hkv = heads >> 16, nrep = tiles_nrep(begins);
  const int b = tiles_batch_row(Hkv, div_hkv, bh), head0 = (bh - b * Hkv) * nrep;
  const int n = lane & 15, r = lane >> 4;
  // row l % 16 of A: head (l % 16) % HP of this launch (rows without a head repeat one, their results are dropped)
  u32x4 qv;
  {
    uint32_t w[4];
    load_words<4, Words2<4>>(q + ((int64_t)b * Hq + head0) * 128, (uint32_t)min(n % HP, nrep - 1) * 256u + 64u * wave + 16u * r, w);
    qv = (u32x4){w[0], w[1], w[2], w[3]};
  }
  if (COUNT && u == 0 && threadIdx.x == 0) arrive[bh] = 0u;
  const int tile = u - sg.unit_begin;
  const int head = (4 * r) % HP + wave;   // the head this lane finishes
  const bool has_head = head < nrep;
  half_t *row = scores + ((int64_t)b * Hq + head0 + min(head, nrep - 1)) * Tall;
  auto qrow = [&]() { return q + ((int64_t)b * Hq + head0 + min((4 * (lane >> 4)) % HP + wave, nrep - 1)) * 128; };
  float m = SM_FLOOR, l = 0.f;
#define HQ_TILE(B_, NORMAL_) qt_class_tile<B_, HP, FUSED, NORMAL_>(sg, tile, bh, n_bh, wave, lane, qv, lds, row, has_head, inv_sqrt_d, m, l, qrow)
  switch (sg.bits) {
    case 1:
      if ((sg.layout & 3) == HQEKV_LAYOUT_NORMAL1) HQ_TILE(1, true);
      else HQ_TILE(1, false);
      break;
    case 2: HQ_TILE(2, false); break;
    case 4: HQ_TILE(4, false); break;
    case 8: HQ_TILE(8, false); break;
    default:
      if ((sg.layout & 3) == HQEKV_LAYOUT_TOKEN_MAJOR) qt_rows_tile<HP, FUSED>(sg, tile, bh, wave, lane, qv, lds, row, has_head, inv_sqrt_d, m, l, qrow);
      else HQ_TILE(16, false);
  }
#undef HQ_TILE
  if (!FUSED) return;
  // lanes of a row of 16 hold the same head; so do the rows r and r' with the same 4 r % HP
  float mm = m;
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
  if (n == 0 && 4 * r < HP && has_head) stats[((int64_t)b * Hq + head0 + head) * n_stat + u] = make_float2(mm, l);
}

// ---- Long launches: four tiles per workgroup, one per wave, which walks all of head_dim in four steps of 32 channels with
// the next step's words on their way.  Its sums stay in the accumulators -- nothing is exchanged between waves but the
// scales, which the workgroup fetches together: 64 bytes of a scale row at a time where a tile of its own has 16, so that a
// cache line is asked for by two workgroups instead of eight, and what a wave spends around its products is spent once per
// tile instead of four times.  Bound by memory: at 8 x 64k tokens (224 MB of codes, 56 MB of scales, 34 MB of scores
// written) 79.7 -> 74.3 us, vector instructions 25.3 -> 20.8 million, cache requests 6.5 -> 3.6 million; without its
// arithmetic it takes 63.  A wave lives four times as long, which a launch of few resident rounds feels: 4096 one-tile
// workgroups -- 3 per slot -- are faster as they are (40.9 against 44.6 us for the call), 8192 break even (95.1, 94.8), 16384
// gain 4 to 5 %.
constexpr int QL_TILES = QT_WAVES;               // tiles per workgroup
constexpr int64_t QT_LONG = 8192;                // one-tile workgroups of a launch above which it pays (see below)
constexpr int QL_NG = QL_TILES * QT_NG;          // 32-token groups
constexpr int QL_NGP = QL_NG + 2;                // LDS row of a channel pair: the four lane groups of a read meet different banks

template <int BITS, int HP, bool FUSED, int TPV, typename Pos, typename Alone>
__device__ __forceinline__ void ql_finish(f4_t (&acc)[TPV], int r, Pos &&pos, int n_valid, bool run, half_t *rows, int64_t Tall, int nrep,
                                          float inv_sqrt_d, float (&m)[4], float (&l)[4], Alone &&alone) {
  if constexpr (HP < 16) {   // a NaN among the sums: see qk_alone
    f4_t all = acc[0];
#pragma unroll
    for (int t = 1; t < TPV; ++t) all += acc[t];
    const float any = (all[0] + all[1]) + (all[2] + all[3]);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(any != any && n_valid > 0) != 0, 0)) {
#pragma unroll 1
      for (int e = 0; e < 4 * n_valid; ++e) {
        bool bad = false;
#pragma unroll
        for (int k = 0; k < 4 * TPV; ++k) bad = bad || (k == e && acc[k / 4][k % 4] != acc[k / 4][k % 4]);
        const float again = bad ? alone(min((4 * r) % HP + e % 4, nrep - 1), e / 4) : 0.f;
#pragma unroll
        for (int k = 0; k < 4 * TPV; ++k) acc[k / 4][k % 4] = k == e && bad ? again : acc[k / 4][k % 4];
      }
    }
  }
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const int head = (4 * r) % HP + h;
    const int nv = head < nrep ? n_valid : 0;
    half_t *row = rows + (int64_t)min(head, nrep - 1) * Tall;
    half_t x[TPV];
    float mm = SM_FLOOR;
#pragma unroll
    for (int t = 0; t < TPV; ++t) {
      x[t] = (half_t)acc[t][h];
      if (FUSED) {   // the fp16 steps of the reference epilogue: round the score, scale, round again
        x[t] = (half_t)((float)x[t] * inv_sqrt_d);
        mm = fmaxf(mm, t < nv ? (float)x[t] : SM_FLOOR);
      }
    }
    if (TPV > 1 && run && nv >= TPV) {
      struct __attribute__((packed, aligned(2))) Run { half_t v[TPV]; };
      Run w;
#pragma unroll
      for (int t = 0; t < TPV; ++t) w.v[t] = x[t];
      gstore(row, pos(0) * 2u, w);
    } else {
#pragma unroll
      for (int t = 0; t < TPV; ++t)
        if (t < nv) gstore(row, pos(t) * 2u, x[t]);
    }
    if (FUSED) {
      float ll = 0.f;
#pragma unroll
      for (int t = 0; t < TPV; ++t) ll += t < nv ? __expf((float)x[t] - mm) : 0.f;
      m[h] = mm;
      l[h] = ll;
    }
  }
}

template <int BITS, int HP, bool FUSED, bool NORMAL>
__device__ __forceinline__ void ql_class(const TileSeg &sg, int unit, int bh, int n_bh, int wave, int lane, const half_t *qrow, uint2 *sz, half_t *rows,
                                         int64_t Tall, int nrep, float inv_sqrt_d, float (&m)[4], float (&l)[4], const half_t *q0) {
  using G = QtGeom<BITS>;
  constexpr bool QUANT = BITS != 16;
  constexpr int BANDS = 16 / HP, TPV = G::TOK / BANDS > 0 ? G::TOK / BANDS : 1;
  const int n = lane & 15, r = lane >> 4;
  const uint32_t n_tok = (uint32_t)sg.n_tokens, row_b = n_tok * BITS / 8;
  const uint32_t tile = (uint32_t)unit * QL_TILES + wave, col0 = tile * G::TILE + G::TOK * n;
  const bool live = tile * G::TILE < n_tok;   // (uniform)
  const int band = (4 * r) / HP;
  const bool runs = qt_runs(sg) && n_tok % 32 == 0;
  const Positions position(sg);
  // ---- scales and zeros of channels 2 p and 2 p + 1, eight groups: thread 4 p + piece
  const uint32_t Gn = n_tok / 32, g0 = (uint32_t)unit * QL_NG;
  uint32_t sw[4][4];
  int back[2];
  if constexpr (QUANT) {
    const int64_t end = (int64_t)n_bh * 128 * Gn - QT_NG;
#pragma unroll
    for (int c = 0; c < 2; ++c) {   // (past a row's end: never used; at the plane's end the window is moved back to stay inside)
      const int64_t at = ((int64_t)bh * 128 + 2 * (threadIdx.x >> 2) + c) * Gn + g0 + QT_NG * (threadIdx.x & 3), from = min(at, end);
      back[c] = (int)min(at - from, (int64_t)QT_NG);
      load_words<4, Words2<4>>(sg.scale + from, 0u, sw[c]);
      load_words<4, Words2<4>>(sg.zero + from, 0u, sw[2 + c]);
    }
  }
  // ---- code words of step c (a column past the row's end repeats the last one, unused)
  const char *codes = (const char *)sg.data + (int64_t)bh * 128 * row_b;
  const uint32_t off = 8u * r * row_b + min(col0, n_tok - G::TOK) * BITS / 8;
  auto load_codes = [&](int c, uint32_t (&w)[8][G::NW]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const char *base = codes + (int64_t)(32 * c + i) * row_b;
      if constexpr (BITS == 1) w[i][0] = gload<uint16_t>(base, off);
      else load_words<G::NW, Words2<G::NW>>(base, off, w[i]);
    }
  };
  constexpr int NB = BITS <= 2 ? 4 : 2;   // steps whose words a wave holds: about 32 registers
  uint32_t cur[NB][8][G::NW], q[2][4];
  auto load_q = [&](int c, uint32_t (&w)[4]) { load_words<4, Words2<4>>(qrow, 64u * c + 16u * r, w); };
  load_q(0, q[0]);
  static_for<NB>([&](auto C_) { load_codes(decltype(C_)::value, cur[decltype(C_)::value]); });
  const uint32_t tok0 = col0 + band * TPV;   // this lane's first token
  const int n_valid = tok0 < n_tok ? TPV : 0;
  const uint32_t tok0c = min(tok0, n_tok - 1), index0 = position.fetch(tok0c);
  HQ_LOADS_ABOVE();
  if constexpr (QUANT) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
      for (int k = back[c]; k; --k) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          sw[c][w] = sw[c][w] >> 16 | (w < 3 ? sw[c][(w + 1) % 4] << 16 : 0u);
          sw[2 + c][w] = sw[2 + c][w] >> 16 | (w < 3 ? sw[2 + c][(w + 1) % 4] << 16 : 0u);
        }
      }
    uint2 *e = sz + (threadIdx.x >> 2) * QL_NGP + QT_NG * (threadIdx.x & 3);
#pragma unroll
    for (int g = 0; g < QT_NG; ++g)
      e[g] = (g & 1) ? make_uint2(as_u32(half_pair<1>(sw[0][g / 2], sw[1][g / 2])), as_u32(half_pair<1>(sw[2][g / 2], sw[3][g / 2])))
                     : make_uint2(as_u32(half_pair<0>(sw[0][g / 2], sw[1][g / 2])), as_u32(half_pair<0>(sw[2][g / 2], sw[3][g / 2])));
    __syncthreads();
  }
  if (!live) return;
  const uint32_t gi = QUANT ? min((uint32_t)(QT_NG * wave + n / 2), Gn - 1 - g0) : 0;
  f4_t acc[TPV];
#pragma unroll
  for (int t = 0; t < TPV; ++t) acc[t] = (f4_t){0.f, 0.f, 0.f, 0.f};
  static_for<4>([&](auto C_) {
    constexpr int C = decltype(C_)::value;
    uint32_t (&w)[8][G::NW] = cur[C % NB];
    if constexpr (C < 3) load_q(C + 1, q[(C + 1) & 1]);
    HQ_LOADS_ABOVE();
    half2_t s2[4], z2[4];
    if constexpr (QUANT) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint2 v = sz[(16 * C + 4 * r + i) * QL_NGP + gi];
        s2[i] = as_h2(v.x);
        z2[i] = as_h2(v.y);
        if (NORMAL) s2[i] = normal1_spread(s2[i]);
      }
    }
    u32x4 a;
    auto into_band = [&](int j) {
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = BANDS == 1 || n / HP == j ? q[C & 1][i] : 0u;
    };
    static_for<(BITS == 16 ? 4 : G::COLB)>([&](auto K_) {
      constexpr int K = decltype(K_)::value;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (QUANT) {
        constexpr int B = BITS == 16 ? 8 : BITS;
        uint32_t u[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i] = byte_pair<K % 4>(w[2 * i][K / 4 % G::NW], w[2 * i + 1][K / 4 % G::NW]);
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
          for (int i = 0; i < 4; ++i) b[i] = as_u32(half_pair<H>(w[2 * i][K % G::NW], w[2 * i + 1][K % G::NW]));
          acc[TOK % TPV] = mfma16(a, b, acc[TOK % TPV]);
        });
      }
    });
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (C + NB < 4) load_codes(C + NB, cur[C % NB]);
  });
  ql_finish<BITS, HP, FUSED, TPV>(acc, r, [&](int t) { return runs ? position.of(tok0c, index0) + t : position(tok0 + t); }, n_valid, runs, rows, Tall,
                                  nrep, inv_sqrt_d, m, l, [&](int head, int t) { return qk_alone<BITS, NORMAL, false>(sg, bh, tok0 + t, q0 + head * 128); });
}

// fp16 K rows stored token by token: a wave takes the 64 tokens of one tile, 32 channels at a time
template <int HP, bool FUSED>
__device__ __forceinline__ void ql_rows(const TileSeg &sg, int unit, int bh, int wave, int lane, const half_t *qrow, half_t *rows, int64_t Tall, int nrep,
                                        float inv_sqrt_d, float (&m)[4], float (&l)[4], const half_t *q0) {
  constexpr int BANDS = 16 / HP, TPV = 4 / BANDS;
  const int n = lane & 15, r = lane >> 4;
  const uint32_t n_tok = (uint32_t)sg.n_tokens, t0 = ((uint32_t)unit * QL_TILES + wave) * QT_TM_TILE;
  if (t0 >= n_tok) return;
  const char *src = (const char *)sg.data + (int64_t)bh * sg.slab_tokens * 256;
  const int band = (4 * r) / HP;
  auto token = [&](int t) { return t0 + 16u * (band * TPV + t) + n; };
  const Positions position(sg);
  f4_t acc[TPV];
#pragma unroll
  for (int t = 0; t < TPV; ++t) acc[t] = (f4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int c = 0; c < 4; ++c) {
    uint32_t q[4];
    u32x4 x[4];
    load_words<4, Words2<4>>(qrow, 64u * c + 16u * r, q);
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] = gload<u32x4>(src, min(t0 + 16u * k + n, n_tok - 1) * 256u + 64u * c + 16u * r);
    static_for<4>([&](auto K_) {
      constexpr int K = decltype(K_)::value;
      u32x4 a;
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = BANDS == 1 || n / HP == K / TPV ? q[i] : 0u;
      acc[K % TPV] = mfma16(a, x[K], acc[K % TPV]);
    });
  }
  int n_valid = 0;
#pragma unroll
  for (int t = 0; t < TPV; ++t) n_valid += token(t) < n_tok ? 1 : 0;
  ql_finish<16, HP, FUSED, TPV>(acc, r, [&](int t) { return position(token(t)); }, n_valid, false, rows, Tall, nrep, inv_sqrt_d, m, l,
                           [&](int head, int t) { return qk_alone<16, false, true>(sg, bh, token(t), q0 + head * 128); });
}

template <int HP, bool FUSED>
__global__ __launch_bounds__(QT_WAVES * 64, HP == 4 ? 4 : 2) void qk_long_kernel(
    u32x4 begins, const half_t *__restrict__ q, half_t *__restrict__ scores, float2 *__restrict__ stats, uint32_t heads, uint32_t div_hkv, int64_t Tall,
    int32_t n_bh, int32_t n_stat, float inv_sqrt_d, TileTable tb) {
  __shared__ __align__(16) uint2 sz[64 * QL_NGP];
  __shared__ float2 st[QT_WAVES][HP];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int bh = blockIdx.x, u = (int)blockIdx.y;
  const TileSeg sg = tb.seg[tiles_segment(begins, u)];
  const int Hq = heads & 0xffffu, Hkv = heads >> 16, nrep = tiles_nrep(begins);
  const int b = tiles_batch_row(Hkv, div_hkv, bh), head0 = (bh - b * Hkv) * nrep;
  const int n = lane & 15, r = lane >> 4, unit = u - sg.unit_begin;
  const half_t *q0 = q + ((int64_t)b * Hq + head0) * 128, *qrow = q0 + min(n % HP, nrep - 1) * 128;
  half_t *rows = scores + ((int64_t)b * Hq + head0) * Tall;
  float m[4], l[4];
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    m[h] = SM_FLOOR;
    l[h] = 0.f;
  }
#define HQ_TILE(B_, NORMAL_) ql_class<B_, HP, FUSED, NORMAL_>(sg, unit, bh, n_bh, wave, lane, qrow, sz, rows, Tall, nrep, inv_sqrt_d, m, l, q0)
  switch (sg.bits) {
    case 1:
      if ((sg.layout & 3) == HQEKV_LAYOUT_NORMAL1) HQ_TILE(1, true);
      else HQ_TILE(1, false);
      break;
    case 2: HQ_TILE(2, false); break;
    case 4: HQ_TILE(4, false); break;
    case 8: HQ_TILE(8, false); break;
    default:
      if ((sg.layout & 3) == HQEKV_LAYOUT_TOKEN_MAJOR) ql_rows<HP, FUSED>(sg, unit, bh, wave, lane, qrow, rows, Tall, nrep, inv_sqrt_d, m, l, q0);
      else HQ_TILE(16, false);
  }
#undef HQ_TILE
  if (!FUSED) return;
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    float mm = m[h], ll = l[h];
    mm = fmaxf(mm, dpp_f<0xB1>(mm));
    mm = fmaxf(mm, dpp_f<0x4E>(mm));
    mm = fmaxf(mm, dpp_f<0x141>(mm));
    mm = fmaxf(mm, dpp_f<0x140>(mm));
    if (HP <= 4) mm = fmaxf(mm, xor_f(mm, 16));
    if (HP <= 8) mm = fmaxf(mm, xor_f(mm, 32));
    ll = m[h] == mm ? ll : ll * __expf(m[h] - mm);   // (a lane that saw no token: l = 0, m the floor)
    ll += dpp_f<0xB1>(ll);
    ll += dpp_f<0x4E>(ll);
    ll += dpp_f<0x141>(ll);
    ll += dpp_f<0x140>(ll);
    if (HP <= 4) ll += xor_f(ll, 16);
    if (HP <= 8) ll += xor_f(ll, 32);
    if (n == 0 && 4 * r < HP) st[wave][4 * r + h] = make_float2(mm, ll);
  }
  __syncthreads();
  const int head = threadIdx.x;
  if (head < nrep) {
    float2 v[QT_WAVES];
    float mm = SM_FLOOR, ll = 0.f;
#pragma unroll
    for (int w = 0; w < QT_WAVES; ++w) {
      v[w] = st[w][head];
      mm = fmaxf(mm, v[w].x);
    }
#pragma unroll
    for (int w = 0; w < QT_WAVES; ++w) ll += v[w].x == mm ? v[w].y : v[w].y * __expf(v[w].x - mm);
    stats[((int64_t)b * Hq + head0 + head) * n_stat + u] = make_float2(mm, ll);
  }
}

// =============================================================================== host side
static int64_t qt_tile(const hqekv_seg &s) {   // tokens
  if (s.bits == 16) return (s.layout & 3) == HQEKV_LAYOUT_TOKEN_MAJOR ? QT_TM_TILE : QtGeom<16>::TILE;
  return QtGeom<2>::TILE;
}

bool tiles_fit(const hqekv_seg *segs, int nseg, bool is_k, int64_t D, int64_t B, int64_t Hq, int64_t Hkv) {
  if (nseg < 0 || nseg > HQEKV_MAX_SEGS || (nseg > 0 && !segs)) return false;
  if (D != 128 || Hkv <= 0 || Hq / Hkv > 16 || B * Hkv * Hkv >= (1LL << 32)) return false;
  for (int k = 0; k < nseg; ++k) {
    const hqekv_seg &s = segs[k];
    if (!(s.bits == 16 || s.bits == 8 || s.bits == 4 || s.bits == 2 || s.bits == 1)) return false;   // (reported by the caller's checks)
    if (s.n_tokens > 0 && is_k && s.bits == 16 && (s.layout & 3) != HQEKV_LAYOUT_TOKEN_MAJOR && s.n_tokens % QtGeom<16>::TOK) return false;   // a lane's column of tokens
  }
  return true;
}

TilesPlan tiles_plan(const hqekv_seg *segs, int nseg, bool is_k, int64_t BHkv, int64_t nrep) {
  TilesPlan p{};
  p.is_k = is_k;
  p.per_unit = 1;
  auto count = [&]() {
    int64_t units = 0;
    for (int k = 0; k < nseg; ++k)
      if (segs[k].n_tokens > 0) {
        const int64_t per = tiles_unit_tokens(p, segs[k]);
        units += (segs[k].n_tokens + per - 1) / per;
      }
    return units;
  };
  p.units = count();
  if (is_k) {
    if (p.units * BHkv > QT_LONG) p.per_unit = QL_TILES;
    p.units = count();
  } else {
    // One block per workgroup while all of them are resident at once; else as many as make one resident round of the
    // looping kernel: a second, nearly empty round would cost a workgroup's whole life.
    const int64_t all = p.units * BHkv, loop = pt_loop_units(nrep, all);
    if (all > pt_resident(nrep)) p.per_unit = (int)((all + loop - 1) / loop);
    p.units = count();
  }
  return p;
}
int64_t tiles_unit_tokens(const TilesPlan &p, const hqekv_seg &s) { return (p.is_k ? qt_tile(s) : pv_block_tokens(s.bits)) * p.per_unit; }

int launch_qk_tiles(const SegTable &tb, const void *q, void *scores, int64_t B, int64_t Hq, int64_t Hkv, int64_t Tall, const FuseArgs &fz,
                    hipStream_t st) {
  const TilesHost t = tiles_host(tb, Hq, Hkv);
  const int64_t nrep = Hq / Hkv;
  const dim3 grid((unsigned)(B * Hkv), (unsigned)tb.total_units);
#define LAUNCH(MORE_, ...)                                                                                                                      \
  hipLaunchKernelGGL((__VA_ARGS__), grid, dim3(QT_WAVES * 64), 0, st, t.begins, (const half_t *)q, (half_t *)scores, fz.stats, t.heads, t.div_hkv, \
                     Tall, (int32_t)(B * Hkv), fz.n_stat, fz.inv_sqrt_d MORE_, t.table)
#define COUNTED , fz.arrive
#define LAUNCH_H(HP_)                                                                      \
  if (tb.per_unit > 1 && fz.stats) LAUNCH(, qk_long_kernel<HP_, true>);                    \
  else if (tb.per_unit > 1) LAUNCH(, qk_long_kernel<HP_, false>);                          \
  else if (fz.stats && fz.arrive) LAUNCH(COUNTED, qk_tiles_kernel<HP_, true, (HP_ <= 8)>); \
  else if (fz.stats) LAUNCH(COUNTED, qk_tiles_kernel<HP_, true, false>);                   \
  else LAUNCH(COUNTED, qk_tiles_kernel<HP_, false, false>)
  if (nrep <= 4) { LAUNCH_H(4); } else if (nrep <= 8) { LAUNCH_H(8); } else { LAUNCH_H(16); }
#undef LAUNCH_H
#undef COUNTED
#undef LAUNCH
  return check_launch("qk_tiles_kernel");
}

}  // namespace hq
