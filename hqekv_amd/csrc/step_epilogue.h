// What a decode step does beside its attention, carried by extra workgroups of the step's last launch: the row of the
// importance ring, the copies into the residual, the row that leaves it.
#pragma once

#include "attn_common.h"
#include "quant_math.h"

#pragma clang fp contract(off)

namespace hq {

// ---- the importance ring's row, in the order torch's GPU reduction adds fp16 rows in (fp32 accumulators):
// a thread of that reduction walks its rows with FOUR interleaved accumulators (its k-th row goes to accumulator
// k mod 4, each starting from zero) and adds them up as ((a0 + a1) + a2) + a3; the rows of one output are dealt
// round-robin to `by` threads whose results are added in a halving tree.  by is 1 for the sum over the batch, and for
// the sum over the 32 heads it is 2 when the row length is a multiple of 4 of at least 256 on an 8-byte aligned
// input, else 1 (measured against torch.sum on the device; the caller passes the value for its shape).
template <int NBY, typename Load>
__device__ __forceinline__ float torch_row_sum(int n_rows, Load &&load) {
  float v[NBY];
#pragma unroll
  for (int y = 0; y < NBY; ++y) {
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
    int r = y;
    for (; r + 3 * NBY < n_rows; r += 4 * NBY) {
      a0 += load(r);
      a1 += load(r + NBY);
      a2 += load(r + 2 * NBY);
      a3 += load(r + 3 * NBY);
    }
    if (r < n_rows) a0 += load(r);
    if (r + NBY < n_rows) a1 += load(r + NBY);
    if (r + 2 * NBY < n_rows) a2 += load(r + 2 * NBY);
    v[y] = ((a0 + a1) + a2) + a3;
  }
  if constexpr (NBY == 2) return v[0] + v[1];
  return v[0];
}

// torch_row_sum<1> for a row count known at compile time, fully unrolled (row k goes to accumulator k mod 4)
template <int N, typename Load>
__device__ __forceinline__ float torch_row_sum_n(Load &&load) {
  float a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < N; ++r) a[r & 3] += load(r);
  return ((a[0] + a[1]) + a[2]) + a[3];
}

constexpr int RING_V = 4;                 // adjacent columns of the ring row a lane loads at a time (8 bytes)
// Columns a workgroup of 1024 threads covers per pass: 256 with the heads dealt to 16 waves, eight loads per lane -- or 64
// with a head row per 16 lanes, all heads of a batch row in flight at once and four times as many workgroups: the form for
// rows that fit one such pass or two (3.3k columns in a step's last launch: 5.4 -> 4.2 us).
constexpr int RING_SPAN = 64 * RING_V, RING_SPAN_SHORT = 16 * RING_V;
constexpr int RING_BLOCKS = 512;          // workgroups of a launch of its own, at most
constexpr int RING_LDS_HEADS = 64;        // most heads whose batch sums a pass parks in LDS

// The probabilities as a pointer into global memory: the pointer arrives inside a by-value struct, where the
// compiler cannot tell its address space and would fall back to generic (flat) loads.
typedef const __attribute__((address_space(1))) half_t *ring_src_t;
struct __attribute__((packed, aligned(2))) ring_quad_t { uint64_t v; };   // RING_V probabilities at an element's alignment
static_assert(sizeof(half_t) * RING_V == sizeof(uint64_t), "a quad is one 64-bit word");
typedef const __attribute__((address_space(1))) ring_quad_t *ring_quad_src_t;

// what the ring row needs from the epilogue's description, by value (nothing here lives in memory)
struct RingShape {
  ring_src_t w;      // (B, Hq, Tall)
  int64_t Tall;
  int B, Hq, by;
};

// heads g, g + waves, ... of a lane's RING_V columns into the LDS tile, for a batch of NB rows known at compile
// time: the loads of HU heads are issued before the first sum is formed (the additions keep torch_row_sum's order)
// `shift` > 0 marks the row's last, ragged quad: its loads start `shift` columns early, so that they end with the
// row, and the wanted columns are moved down afterwards.
template <int NB, int SPAN, bool ALONE, typename Prob>
__device__ __forceinline__ void ring_heads_to_lds(const RingShape r, ring_src_t col, int shift, int g, int waves,
                                                  half_t *tile_lane, Prob &&prob) {
  // heads in flight per thread: in long passes the 32 heads are dealt to 16 groups of lanes, two each (eight loads at most, or
  // the registers of the pass grow), in short ones to 64 (16) groups.  (A head past the last one is loaded again: with eight
  // heads in flight for one batch row 20 rows of 4099 probabilities took 9.7 us, now 8.5, of 32768 32.1 / 23.8.)
  constexpr int HU = SPAN == RING_SPAN ? (NB > 4 ? 1 : 2) : ALONE ? 1 : 2;
  const int64_t hs = r.Tall, bs = (int64_t)r.Hq * r.Tall;
  for (int h0 = g; h0 < r.Hq; h0 += waves * HU) {
    uint64_t raw[HU][NB];   // a quad is loaded, shifted and stored as one 64-bit word
#pragma unroll
    for (int u = 0; u < HU; ++u) {
      const int h = min(h0 + u * waves, r.Hq - 1);
#pragma unroll
      for (int b = 0; b < NB; ++b) {   // 8 bytes at the alignment of an element: the target reads unaligned
        if constexpr (std::remove_reference_t<Prob>::THROUGH) {   // (written past the L2 in this launch; below 2 GB)
          const uint32_t at = (uint32_t)(((int64_t)b * r.Hq + h) * hs * 2) + (uint32_t)((uintptr_t)col - (uintptr_t)r.w);
          raw[u][b] = __builtin_bit_cast(uint64_t, __builtin_amdgcn_raw_buffer_load_b64(make_rsrc((const void *)(uintptr_t)r.w, 0x7fffffffu), (int)at, 0, 16)) >> (16 * shift);
        } else {
          raw[u][b] = reinterpret_cast<ring_quad_src_t>(col + (int64_t)b * bs + (int64_t)h * hs)->v >> (16 * shift);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < HU; ++u) {
      const int h = h0 + u * waves;
#pragma unroll
      for (int b = 0; b < NB; ++b) raw[u][b] = prob(b * r.Hq + min(h, r.Hq - 1), raw[u][b]);
      uint64_t v = raw[u][0];
      if constexpr (NB > 1) {
        v = 0;
#pragma unroll
        for (int i = 0; i < RING_V; ++i) {
          const half_t s = (half_t)torch_row_sum_n<NB>(
              [&](int b) { return (float)__builtin_bit_cast(half_t, (uint16_t)(raw[u][b] >> (16 * i))); });
          v |= (uint64_t)__builtin_bit_cast(uint16_t, s) << (16 * i);
        }
      }
      if (h < r.Hq) *reinterpret_cast<uint64_t *>(tile_lane + h * SPAN) = v;   // 8-byte aligned: lane * RING_V halves
    }
  }
}

// Column t for any batch size and head count, one load at a time: for the shapes the tiled path does not take.
// Kept out of line so that its registers do not add to the tiled path's.
static __device__ __noinline__ float ring_column_alone(const RingShape r, int64_t t) {
  ring_src_t col = r.w + t;
  const int64_t hs = r.Tall, bs = (int64_t)r.Hq * r.Tall;
  auto head = [&](int h) -> float {
    if (r.B == 1) return (float)col[(int64_t)h * hs];
    return (float)(half_t)torch_row_sum<1>(r.B, [&](int b) { return (float)col[(int64_t)b * bs + (int64_t)h * hs]; });
  };
  return r.by == 2 ? torch_row_sum<2>(r.Hq, head) : torch_row_sum<1>(r.Hq, head);
}

// Columns [c0, c1) of the ring row, SPAN per pass (c0 a multiple of SPAN).  The loads are spread over the whole workgroup
// -- lane l of every group of SPAN / 4 threads looks at columns 4 l .. 4 l + 3 of the pass, group g at heads g, g + groups,
// ... -- so every load is independent of the others and 8 bytes wide; the head values (fp16 by construction) meet
// in LDS, where the first SPAN threads add them up in torch's order, one column each.  Every thread of the
// workgroup must call this with the same arguments; blockDim.x is a multiple of 64 and at least SPAN.
template <int SPAN, bool ALONE, typename Prob>
__device__ __forceinline__ void ring_row_columns(const StepEpilogue &e, int64_t c0, int64_t c1, half_t *tile, Prob &&prob) {
  const RingShape r{(ring_src_t)(uintptr_t)e.weights, e.Tall, e.B, e.Hq, e.ring_by};
  half_t *const line = e.ring_line;
  constexpr int QUADS = SPAN / RING_V;
  const int lane = threadIdx.x % QUADS, g = threadIdx.x / QUADS, groups = blockDim.x / QUADS;
  const bool lds = r.Hq <= RING_LDS_HEADS && r.B <= 8;
  for (int64_t t0 = c0; t0 < c1; t0 += SPAN) {
    const int64_t t = t0 + threadIdx.x;   // the column this thread sums in the end (threads below SPAN)
    if (lds) {
      const int64_t c = t0 + lane * RING_V;
      // the row's last quad may stick out by `shift` columns (the passes of all workgroups but the last end on a
      // multiple of SPAN): it is loaded from `shift` columns earlier, which needs a row of RING_V columns at least
      const int shift = (int)max((int64_t)0, c + RING_V - c1);
      const bool mine = shift < RING_V && c - shift >= 0;
      ring_src_t col = r.w + (mine ? c - shift : 0);
      half_t *tile_lane = tile + lane * RING_V;
      switch (mine ? r.B : 0) {
        case 1: ring_heads_to_lds<1, SPAN, ALONE>(r, col, shift, g, groups, tile_lane, prob); break;
        case 2: ring_heads_to_lds<2, SPAN, ALONE>(r, col, shift, g, groups, tile_lane, prob); break;
        case 3: ring_heads_to_lds<3, SPAN, ALONE>(r, col, shift, g, groups, tile_lane, prob); break;
        case 4: ring_heads_to_lds<4, SPAN, ALONE>(r, col, shift, g, groups, tile_lane, prob); break;
        case 5: ring_heads_to_lds<5, SPAN, ALONE>(r, col, shift, g, groups, tile_lane, prob); break;
        case 6: ring_heads_to_lds<6, SPAN, ALONE>(r, col, shift, g, groups, tile_lane, prob); break;
        case 7: ring_heads_to_lds<7, SPAN, ALONE>(r, col, shift, g, groups, tile_lane, prob); break;
        case 8: ring_heads_to_lds<8, SPAN, ALONE>(r, col, shift, g, groups, tile_lane, prob); break;
        default: break;
      }
      __syncthreads();
    }
    if (threadIdx.x < SPAN && t < c1) {
      float sum = 0.f;
      if (!ALONE || (lds && c1 >= RING_V)) {
        auto head = [&](int h) -> float { return (float)tile[h * SPAN + threadIdx.x]; };
        sum = r.by == 2 ? torch_row_sum<2>(r.Hq, head) : torch_row_sum<1>(r.Hq, head);
      } else if constexpr (ALONE) {   // outside what the LDS tile covers: the thread walks its column alone
        sum = ring_column_alone(r, t);
      }
      // (several rows at once: the columns are (row, token) pairs)
      if (e.ring_tokens) {   // (the store holds fewer than 2^31 elements)
        const uint32_t n = (uint32_t)e.ring_tokens, row = (uint32_t)t / n;
        line[row * (uint32_t)e.ring_stride + ((uint32_t)t - row * n)] = (half_t)sum;
      } else {
        line[t] = (half_t)sum;
      }
    }
    if (lds) __syncthreads();
  }
}

struct RingAsIs {
  static constexpr bool THROUGH = false;
  __device__ __forceinline__ uint64_t operator()(int, uint64_t quad) const { return quad; }
};

// block `blk` of `nblk` of the epilogue: a share of the ring row's columns, and of the appended rows
template <bool ALONE = true, typename Prob = RingAsIs>
__device__ __forceinline__ void step_epilogue_block(const StepEpilogue &e, int64_t blk, int64_t nblk, half_t *sh, Prob &&prob = Prob{}) {
  if (e.ring_line) {
    if (!ALONE || e.Tall <= 2 * RING_SPAN_SHORT * nblk) {
      const int64_t per = ((e.Tall + nblk - 1) / nblk + RING_SPAN_SHORT - 1) / RING_SPAN_SHORT * RING_SPAN_SHORT;
      ring_row_columns<RING_SPAN_SHORT, ALONE>(e, min(e.Tall, blk * per), min(e.Tall, (blk + 1) * per), sh, prob);
    } else {
      const int64_t per = ((e.Tall + nblk - 1) / nblk + RING_SPAN - 1) / RING_SPAN * RING_SPAN;
      ring_row_columns<RING_SPAN, ALONE>(e, min(e.Tall, blk * per), min(e.Tall, (blk + 1) * per), sh, prob);
    }
  }
  if (e.ring_fill_rows) {   // a new store: zeros wherever these rows do not reach
    const uint32_t stride = (uint32_t)e.ring_stride, n = (uint32_t)e.ring_fill_rows * stride;
    const uint32_t rows = (uint32_t)(e.Tall / e.ring_tokens), tokens = (uint32_t)e.ring_tokens;
    for (uint32_t i = (uint32_t)blk * blockDim.x + threadIdx.x; i < n; i += (uint32_t)nblk * blockDim.x)
      if (i / stride >= rows || i % stride >= tokens) e.ring_line[i] = (half_t)0;
  }
  if (e.app_rows > 0) {   // 16-byte pieces of the appended rows, dealt over the blocks
    const int64_t row16 = e.app_row_elems / 8;   // pieces per row (head_dim is a multiple of 32)
    const int64_t per_side = (int64_t)e.app_bh * e.app_rows * row16;
    for (int64_t i = blk * blockDim.x + threadIdx.x; i < 2 * per_side; i += nblk * blockDim.x) {
      const int side = i >= per_side ? 1 : 0;
      const int64_t j = i - side * per_side;
      const int64_t bh = j / (e.app_rows * row16), rem = j % (e.app_rows * row16);
      const uint4 *src = reinterpret_cast<const uint4 *>(e.app_src[side] + bh * e.app_src_slab[side]) + rem;
      uint4 *dst = reinterpret_cast<uint4 *>(e.app_dst[side] + bh * e.app_dst_slab[side]) + rem;
      *dst = *src;
    }
  }
  if (e.leave_bits) {   // four lanes per group of 32 (a KIVI layer's step: a launch of 2.6 us of its own before)
    const int64_t n = (int64_t)e.app_bh * e.leave_groups * 4;
    for (int64_t i = blk * blockDim.x + threadIdx.x; i < n; i += nblk * blockDim.x) {
      const int64_t bh = (i >> 2) / e.leave_groups, g = (i >> 2) % e.leave_groups, at = bh * e.leave_rows * e.leave_groups + g;
      const half_t *src = e.leave_src + bh * e.leave_slab + 32 * g;
      const uint32_t sub = (uint32_t)i & 3u;
      switch (e.leave_bits) {
        case 8: quant_group_of_4<8>(src, sub, e.leave_code + at * 8, e.leave_scale + at, e.leave_zero + at); break;
        case 4: quant_group_of_4<4>(src, sub, e.leave_code + at * 4, e.leave_scale + at, e.leave_zero + at); break;
        case 2: quant_group_of_4<2>(src, sub, e.leave_code + at * 2, e.leave_scale + at, e.leave_zero + at); break;
        default: quant_group_of_4<1>(src, sub, e.leave_code + at, e.leave_scale + at, e.leave_zero + at);
      }
    }
  }
}

}  // namespace hq
