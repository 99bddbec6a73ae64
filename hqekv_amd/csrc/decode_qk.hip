// q.K^T of a decode step on matrix instructions (see decode_tiles.h), and how the decode launches are cut up.
#include "decode_qk_tile.h"

#pragma clang fp contract(off)

namespace hq {

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
  const QtRow row{scores + ((int64_t)b * Hq + head0 + min(head, nrep - 1)) * Tall};
  auto qrow = [&]() { return q + ((int64_t)b * Hq + head0 + min((4 * (lane >> 4)) % HP + wave, nrep - 1)) * 128; };
  float mm, l;
  qt_unit<HP, FUSED>(sg, tile, bh, n_bh, wave, lane, qv, lds, row, has_head, inv_sqrt_d, mm, l, qrow);
  if (FUSED && n == 0 && 4 * r < HP && has_head) stats[((int64_t)b * Hq + head0 + head) * n_stat + u] = make_float2(mm, l);
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
