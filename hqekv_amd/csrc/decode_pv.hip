// p.V of a decode step on matrix instructions (see decode_tiles.h).
#include "decode_pv_tile.h"

#pragma clang fp contract(off)

namespace hq {

// `logits` is `p` unless LAST: then the logits lie in the workspace.
template <int HP, bool EXACT, bool LOOP, bool FUSED, bool LAST>
__device__ __forceinline__ void pv_tiles_body(const TileTable &tb, u32x4 begins, const half_t *logits, half_t *p, const float2 *stats, uint32_t heads,
                                              uint32_t div_hkv, int64_t Tall, float *partial, uint32_t n_bhq, int n_stat, int per, int total_units,
                                              uint32_t *arrive, half_t *out) {
  __shared__ __align__(16) PtLds<HP, LOOP> lds;
  __shared__ __align__(16) float red[PT_WAVES][HP][128];
  __shared__ float ml[2 * HP];   // (max, 1 / sum exp) of each head's row
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int bh = blockIdx.x, u = blockIdx.y;
  const TileSeg sg = tb.seg[tiles_segment(begins, u)];
  const int Hq = heads & 0xffffu, Hkv = heads >> 16, nrep = EXACT ? HP : tiles_nrep(begins);
  const int b = tiles_batch_row(Hkv, div_hkv, bh), head0 = (bh - b * Hkv) * nrep;
  const half_t *rows = logits + ((int64_t)b * Hq + head0) * Tall;
  half_t *prows = p + ((int64_t)b * Hq + head0) * Tall;
  f4_t acc[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) acc[c] = (f4_t){0.f, 0.f, 0.f, 0.f};
  // wave w merges the per-tile pairs of heads w, w + 4, ...; up to 256 tiles of the first are read once, ahead of the rest
  // (past the last tile: the last one again, left out of the sum).  LAST: sixteen lanes a head, as the ring row's workgroups
  // do it for every row of the step, hence with the same bits.
  float2 sv[4];
  auto read_stats = [&](const float2 *sp) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k == 0 || n_stat > 64 * k) {
        uint32_t w[2];
        load_words<2, Words4<2>>(sp, 8u * (uint32_t)min(lane + 64 * k, n_stat - 1), w);
        sv[k] = make_float2(__builtin_bit_cast(float, w[0]), __builtin_bit_cast(float, w[1]));
      }
  };
  const int first = LAST ? (int)threadIdx.x >> 4 : wave;
  const float2 *srow = stats + ((int64_t)b * Hq + head0 + min(first, nrep - 1)) * n_stat;
  auto load_stats = [&]() {
    if constexpr (LAST) row16_read(srow, n_stat, lane & 15, sv);
    else if (FUSED) read_stats(srow);
  };
  auto merge_stats = [&]() {
    if (!FUSED) return;
    if constexpr (LAST) {
      if (wave * 4 < nrep) {
        const float2 v = row16_merge(srow, n_stat, lane & 15, sv);
        if ((lane & 15) == 0 && first < nrep) {
          ml[2 * first] = v.x;
          ml[2 * first + 1] = v.y;
        }
      }
      __syncthreads();
      return;
    }
    for (int h = wave; h < nrep; h += PT_WAVES) {
      const float2 *sp = srow + (int64_t)(h - wave) * n_stat;
      if (h != wave) read_stats(sp);
      float m = sv[0].x;
#pragma unroll
      for (int k = 1; k < 4; ++k)
        if (n_stat > 64 * k) m = fmaxf(m, sv[k].x);
      for (int e = lane + 256; e < n_stat; e += 64) m = fmaxf(m, sp[e].x);
      m = wave_max(m);
      float l = 0.f;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k == 0 || n_stat > 64 * k) l += lane + 64 * k < n_stat ? sv[k].y * __expf(sv[k].x - m) : 0.f;
      for (int e = lane + 256; e < n_stat; e += 64) {
        const float2 w = sp[e];
        l += w.y * __expf(w.x - m);
      }
      l = wave_sum(l);
      if (lane == 0) {
        ml[2 * h] = m;
        ml[2 * h + 1] = 1.0f / l;
      }
    }
    __syncthreads();
  };
  pt_unit<HP, EXACT, LOOP, FUSED, LAST, false>(sg, u - sg.unit_begin, per, bh, wave, lane, PtRows{rows, Tall}, prows, Tall, nrep, lds, ml, acc, 0u, load_stats,
                                               merge_stats);
  float *dst = partial + ((int64_t)u * n_bhq + (int64_t)b * Hq + head0) * 128;
  pt_store_partial<HP, EXACT>(acc, red, wave, lane, nrep, [&](int at, float2 sum) {
    if constexpr (LAST) {
      __hip_atomic_store(reinterpret_cast<uint64_t *>(dst) + at, __builtin_bit_cast(uint64_t, sum), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      *(reinterpret_cast<float2 *>(dst) + at) = sum;
    }
  });
  if constexpr (LAST) {
    // The rows are in memory when their stores are acknowledged; whoever counts the last of this (b, kv head)'s workgroups
    // adds them up, in order.  (Agent-scope accesses go past the L2, which the XCDs do not share; see FuseArgs.)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    __shared__ int last;
    if (threadIdx.x == 0) last = __hip_atomic_fetch_add(&arrive[bh], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == (uint32_t)total_units;
    __syncthreads();
    if (!last) return;
    pt_sum_partials<HP, EXACT>(partial + ((int64_t)b * Hq + head0) * 128, n_bhq, total_units, nrep, &red[0][0][0], out + ((int64_t)b * Hq + head0) * 128);
  }
}

template <int HP, bool EXACT, bool LOOP, bool FUSED>
__global__ __launch_bounds__(PT_WAVES * 64, HP <= 8 ? (LOOP ? (HP == 8 ? 3 : 4) : 6) : 2) void pv_tiles_kernel(
    u32x4 begins, half_t *__restrict__ p, const float2 *__restrict__ stats, float *__restrict__ partial, uint32_t heads, uint32_t div_hkv, int64_t Tall,
    uint32_t n_bhq, int32_t n_stat, int32_t per_unit, TileTable tb) {
  pv_tiles_body<HP, EXACT, LOOP, FUSED, false>(tb, begins, p, p, stats, heads, div_hkv, Tall, partial, n_bhq, n_stat, per_unit, 0, nullptr, nullptr);
}

template <int HP, bool EXACT>
__global__ __launch_bounds__(PT_WAVES * 64, 4) void pv_last_kernel(
    u32x4 begins, const half_t *__restrict__ logits, half_t *__restrict__ p, const float2 *__restrict__ stats, uint32_t heads, uint32_t div_hkv,
    int64_t Tall, float *__restrict__ partial, uint32_t n_bhq, int32_t n_stat, int32_t total_units, uint32_t *__restrict__ arrive,
    half_t *__restrict__ out, TileTable tb, StepEpilogue ep) {
  if ((int)blockIdx.y < total_units) {
    pv_tiles_body<HP, EXACT, false, true, true>(tb, begins, logits, p, stats, heads, div_hkv, Tall, partial, n_bhq, n_stat, 1, total_units, arrive, out);
    return;
  }
  __shared__ __align__(16) PtEpilogue sh;
  if (ep.ring_line) {
    const int lane = threadIdx.x & 15, rows = ep.B * ep.Hq;
    for (int row = threadIdx.x >> 4; row < rows; row += 2 * PT_WAVES * 4) {   // two rows at a time
      float2 sv[2][4];
#pragma unroll
      for (int k = 0; k < 2; ++k) row16_read(stats + (int64_t)min(row + k * PT_WAVES * 4, rows - 1) * n_stat, n_stat, lane, sv[k]);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int at = min(row + k * PT_WAVES * 4, rows - 1);
        const float2 v = row16_merge(stats + (int64_t)at * n_stat, n_stat, lane, sv[k]);
        if (lane == 0) sh.ml[at] = v;
      }
    }
    __syncthreads();
  }
  step_epilogue_block<false>(ep, (int64_t)(blockIdx.y - total_units) * gridDim.x + blockIdx.x, (int64_t)(gridDim.y - total_units) * gridDim.x,
                             sh.ring, PtRingProb<false>{sh.ml});
}

// =============================================================================== host side
int64_t pv_block_tokens(int bits) { return bits >= 8 ? PtGeom<8>::BLOCK : PT_BLOCK; }

int launch_pv_tiles(const SegTable &tb, void *p, float *partial, int64_t B, int64_t Hq, int64_t Hkv, int64_t Tall, const FuseArgs &fz,
                    hipStream_t st) {
  const TilesHost t = tiles_host(tb, Hq, Hkv);
  const int64_t nrep = Hq / Hkv;
  const dim3 grid((unsigned)(B * Hkv), (unsigned)tb.total_units), block(PT_WAVES * 64);
#define LAUNCH(HP_, EXACT_, LOOP_, FUSED_) \
  hipLaunchKernelGGL((pv_tiles_kernel<HP_, EXACT_, LOOP_, FUSED_>), grid, block, 0, st, t.begins, (half_t *)p, fz.stats, partial, t.heads, \
                     t.div_hkv, Tall, (uint32_t)(B * Hq), fz.n_stat, tb.per_unit, t.table)
  const bool loop = tb.per_unit > 1;
#define LAUNCH_H(HP_)                                                                 \
  if (!fz.stats) LAUNCH(HP_, false, true, false);                                     \
  else if (HP_ <= 8 && nrep == HP_ && loop) LAUNCH(HP_, (HP_ <= 8), true, true);     \
  else if (HP_ <= 8 && nrep == HP_) LAUNCH(HP_, (HP_ <= 8), false, true);            \
  else if (loop) LAUNCH(HP_, false, true, true);                                      \
  else LAUNCH(HP_, false, false, true)
  if (nrep <= 4) { LAUNCH_H(4); } else if (nrep <= 8) { LAUNCH_H(8); } else { LAUNCH_H(16); }
#undef LAUNCH_H
#undef LAUNCH
  return check_launch("pv_tiles_kernel");
}

// One p.V launch that also adds its partial rows up and carries the step's epilogue, in place of two launches.  What it adds
// to every workgroup's end (stores acknowledged by memory, a counter, 2 KB per partial row into one CU) equals a launch's
// start at about 20 rows; the host saves 2.5 us at any size.  A step of the fp16 / 8 / 4 / 2-bit mix, B = 1, device time in
// us, three launches / two: 1k tokens 11.1 / 10.3, 2k 11.0 / 10.4, 4k (18 rows) 12.1 / 11.6, 5k 12.2 / 12.1, 6k (25 rows)
// 12.6 / 13.0, 8k 13.3 / 14.5; 4 x 2k 13.6 / 12.7, 4 x 4k 15.9 / 15.5, 16 x 2k 21.4 / 20.5, 8 x 4k 20.8 / 20.9; five heads per
// KV head, 4 x 2k 14.7 / 13.0.
bool decode_in_two(const hqekv_seg *v_segs, int n_v, int64_t D, int64_t B, int64_t Hq, int64_t Hkv) {
  if (n_v <= 0 || !tiles_fit(v_segs, n_v, false, D, B, Hq, Hkv) || Hq / Hkv > 8) return false;
  const TilesPlan p = tiles_plan(v_segs, n_v, false, B * Hkv, Hq / Hkv);
  return p.per_unit == 1 && p.units <= STEP_UNITS;
}
bool pv_last_takes(const StepEpilogue &ep, int64_t Tall) {
  return !ep.ring_line || (ep.B <= 8 && ep.Hq <= RING_LDS_HEADS && (int64_t)ep.B * ep.Hq <= PT_RING_ROWS && Tall >= RING_V);   // what the ring's LDS tile covers
}

int64_t pv_epilogue_blocks(const StepEpilogue &ep, int64_t Tall) {
  return ep.ring_line ? (Tall + RING_SPAN_SHORT - 1) / RING_SPAN_SHORT : ep.app_rows > 0 || ep.leave_bits ? 1 : 0;
}

int launch_pv_last(const SegTable &tb, const void *logits, void *probs, float *partial, int64_t B, int64_t Hq, int64_t Hkv, int64_t Tall,
                   const FuseArgs &fz, const StepEpilogue &ep, hipStream_t st) {
  const TilesHost t = tiles_host(tb, Hq, Hkv);
  const int64_t nrep = Hq / Hkv;
  const int64_t more = pv_epilogue_blocks(ep, Tall);
  const dim3 grid((unsigned)(B * Hkv), (unsigned)(tb.total_units + (more + B * Hkv - 1) / (B * Hkv)));
#define LAUNCH(HP_, EXACT_)                                                                                                                     \
  hipLaunchKernelGGL((pv_last_kernel<HP_, EXACT_>), grid, dim3(PT_WAVES * 64), 0, st, t.begins, (const half_t *)logits, (half_t *)probs, fz.stats, \
                     t.heads, t.div_hkv, Tall, partial, (uint32_t)(B * Hq), fz.n_stat, tb.total_units, fz.arrive, fz.out, t.table, ep)
  if (nrep == 4) LAUNCH(4, true);
  else if (nrep < 4) LAUNCH(4, false);
  else if (nrep == 8) LAUNCH(8, true);
  else LAUNCH(8, false);
#undef LAUNCH
  return check_launch("pv_last_kernel");
}

}  // namespace hq
