// Decode launches (decode_qk.hip: q.K^T, decode_pv.hip: p.V) on 16x16x32 matrix instructions, head_dim 128, up to 16 query
// heads per KV head.
//
// One instruction multiplies 16 rows of heads with 16 columns.  Lane l of the wave supplies eight consecutive elements
// of the reduction axis, 8 (l / 16) ..., of row l % 16 of A and of column l % 16 of B, and receives rows 4 (l / 16) ... + 3
// of column l % 16 of D.  So a lane dequantises eight codes along the reduction axis -- eight channels of a K token, eight
// tokens of a V channel -- straight into a B operand, packed in pairs exactly as the dequantiser works, and the sums over
// head_dim or tokens stay on the matrix pipe up to the four-fold split over a workgroup's waves.
//
// With fewer than 16 heads the spare rows of A are put to use in q.K^T: A is laid out HP heads (4, 8 or 16) to a "band"
// of rows, and the operand for token i of a packed word has only band i / (tokens per band) filled.  Products of different
// bands then share one accumulator, every lane ends up with the scores of its own tokens, and four heads need a quarter
// of the accumulators (and leave all 64 lanes busy in the softmax statistics instead of 16).  A key that is not a number
// or not finite reaches the other bands' tokens through the zeros: such scores are taken again (qk_alone, decode_qk.hip).
#pragma once

#include "attn_common.h"

#pragma clang fp contract(off)

namespace hq {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f4_t mfma16(u32x4 a, u32x4 b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
}

#if defined(__HIP_DEVICE_COMPILE__)
#define HQ_GLOBAL __attribute__((address_space(1)))   // pointers out of the segment table carry no address space of their own
#else
#define HQ_GLOBAL
#endif

// loads of N words at the alignment of an element (the target reads unaligned)
template <int N>
struct __attribute__((packed, aligned(2))) Words2 { uint32_t v[N]; };
template <int N>
struct __attribute__((packed, aligned(4))) Words4 { uint32_t v[N]; };

template <int N, typename W>
__device__ __forceinline__ void load_words(const void *base, uint32_t off, uint32_t (&out)[N]) {
  typedef const HQ_GLOBAL W *src_t;
  const W w = *(src_t)(uintptr_t)((const char *)base + off);
#pragma unroll
  for (int i = 0; i < N; ++i) out[i] = w.v[i];
}
template <typename T>
__device__ __forceinline__ T gload(const void *base, uint32_t off) {
  return *(const HQ_GLOBAL T *)(uintptr_t)((const char *)base + off);
}
template <typename T>
__device__ __forceinline__ void gstore(void *base, uint32_t off, T v) {
  *(HQ_GLOBAL T *)(uintptr_t)((char *)base + off) = v;
}

// keep LDS traffic of one wave in program order (the hardware does; this holds the compiler to it)
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// =============================================================================== what both launches take apart
// What a workgroup needs before it can ask for anything -- the segments' first units, the pointers it starts from, the head
// counts -- stands first among the arguments, as 14 words that the command processor puts into scalar registers before the
// wave starts (build.py: -amdgpu-kernarg-preload-count).  Its first load is then the segment's entry, one cache line; with the
// begins in memory that was the second round, a fifth of a microsecond per launch: a step at 32k tokens 19.37 -> 18.89 us, 3 x
// 16k with five heads per KV head 24.2 -> 23.5, 8 x 64k 150.3 -> 148.6, a KIVI layer's 24 steps at 4k 450 -> 440.
struct __attribute__((aligned(64))) TileSeg {
  const void *data;
  const half_t *scale;
  const half_t *zero;
  const int64_t *idx;
  int64_t slab_tokens;   // as SegDev's
  int32_t pos_base, n_tokens;
  int32_t bits, layout;
  int32_t unit_begin;
};
static_assert(sizeof(TileSeg) == 64, "one line");
struct TileTable {
  TileSeg seg[HQEKV_MAX_SEGS];
};
// Seven begins of 16 bits (0xffff: unused; the first segment's is 0) and, in the first half word, the heads per KV head;
// Hq | Hkv << 16 beside them.
__device__ __forceinline__ int tiles_nrep(u32x4 begins) { return (int)(begins[0] & 0xffffu); }
__device__ __forceinline__ int tiles_segment(u32x4 begins, int u) {   // scalar arithmetic only: everything waits for it
  int s = 0;
#pragma unroll
  for (int k = 1; k < HQEKV_MAX_SEGS; ++k) s -= ((int)(k & 1 ? begins[k / 2] >> 16 : begins[k / 2] & 0xffffu) - u - 1) >> 31;
  return s;
}
// div_hkv = ceil(2^32 / Hkv): bh / Hkv is the high word of the product as long as bh Hkv < 2^32
__device__ __forceinline__ int tiles_batch_row(int Hkv, uint32_t div_hkv, int bh) { return Hkv == 1 ? bh : (int)__umulhi((uint32_t)bh, div_hkv); }

// Position of token t, below 2^31 (it indexes a row of Tall scores): the low word of its index is enough, read at the first
// token of its run of 32 where positions come in runs (HQEKV_LAYOUT_RUNS).  In two parts without a branch between them, so
// that the load is not waited for where it is issued: a segment without an index reads a word it ignores.
struct Positions {
  const void *src;      // the index, or anything readable
  uint32_t keep, scale, run, base;
  __device__ __forceinline__ explicit Positions(const TileSeg &sg) {
    const bool has = sg.idx != nullptr;
    src = has ? (const void *)sg.idx : sg.data;
    keep = __builtin_amdgcn_readfirstlane(has ? ~0u : 0u);   // (or the compiler makes two code paths of it)
    scale = keep & 8u;
    run = ((sg.layout & HQEKV_LAYOUT_RUNS) ? 31u : 0u) | ~keep;   // bits of t that are added to what was read
    base = (uint32_t)sg.pos_base & ~keep;
  }
  __device__ __forceinline__ uint32_t fetch(uint32_t t) const { return gload<uint32_t>(src, scale * (t & ~run)); }
  __device__ __forceinline__ uint32_t of(uint32_t t, uint32_t fetched) const { return (fetched & keep) + (t & run) + base; }
  __device__ __forceinline__ uint32_t operator()(uint32_t t) const { return of(t, fetch(t)); }
};
__device__ __forceinline__ bool qt_runs(const TileSeg &sg) { return (sg.layout & HQEKV_LAYOUT_RUNS) || !sg.idx; }

// =============================================================================== host side
// p.V workgroups the chip holds at once, of the single-block form, and the workgroups a looping launch is made of: one
// resident round.  Single block: six per CU up to eight heads per KV head (80 registers), three above (45 KB of LDS).
// Looping: four per CU up to four heads (128 registers), three up to eight -- the 33 KB of LDS would let four in, but at
// their 128 registers 43 are spilled, inside the loop; at three per CU it takes 150 and spills none.  A step of the fp16 / 8 /
// 4 / 2-bit mix, four / three per CU, us: 5 heads x 8 KV heads at 48k tokens 32.0 / 30.9, at 64k 38.2 / 35.8, at 8 x 32k 107.8 /
// 100.1; 8 heads, 8 x 32k 116.3 / 109.5; 7 heads x 4, 4 x 64k 59.8 / 55.7; two per CU 31.1, 37.4, 112.6, 120.8, 58.3.  (Up to
// four heads three per CU is a tie, and single blocks for fewer than six per CU lose up to 2 %.)  Above eight heads two
// per CU (58 KB of LDS) -- two rounds of those for launches of more than 4096 blocks, whose last round weighs less than the
// runs of a workgroup that meets the end of its class.  p.V at 16 heads, 512 / 1024 workgroups: 1800 blocks (B=1, 64k tokens)
// 27.4 / 33.2 us, 3700 (4 x 32k) 42.0 / 46.9, 5500 (8 x 24k) 64.8 / 65.1, 7400 (8 x 32k) 84.3 / 81.8, 14700 (8 x 64k) 155.8 /
// 152.2.
constexpr int64_t pt_resident(int64_t nrep) { return (nrep <= 8 ? 6 : 3) * 256; }
constexpr int64_t pt_loop_units(int64_t nrep, int64_t blocks) { return (nrep <= 4 ? 4 : nrep <= 8 ? 3 : blocks > 4096 ? 4 : 2) * 256; }

// How a launch is cut up.
struct TilesPlan {
  bool is_k;
  int per_unit;       // p.V: blocks per workgroup
  int64_t units;      // workgroups per (b, kv head); q.K^T leaves one softmax pair per query head in each
};
// head_dim 128, at most 16 query heads per KV head (the rows of A), channel-major fp16 K classes of whole 8-token columns.
// Every ratio up to there is faster here than in the forms of attn.hip, also where rows are spare.  A step at 1k, 32k and
// 8 x 64k tokens of the fp16 / 8 / 4 / 2-bit mix, us, here against there: 1 head 10.1 / 14.4, 19.4 / 25.1, 153 / 178; 2 heads
// 10.1 / 15.5, 19.9 / 26.8, 159 / 187; 4 heads 10.2 / 17.3, 20.7 / 29.3, 172 / 205; 5 heads 10.7 / 20.9, 22.6 / 38.8, 180 /
// 260; 8 heads 10.6 / 23.3, 24.6 / 51.9, 200 / 322; 9 heads 13.3 / 35.7, 28.3 / 70.4, 225 / 489; 16 heads 14.2 / 45.8, 32.4 /
// 98.2, 275 / 644.  (One head: p.V alone is a tie, q.K^T is what gains.)
bool tiles_fit(const hqekv_seg *segs, int nseg, bool is_k, int64_t D, int64_t B, int64_t Hq, int64_t Hkv);
TilesPlan tiles_plan(const hqekv_seg *segs, int nseg, bool is_k, int64_t BHkv, int64_t nrep);
int64_t tiles_unit_tokens(const TilesPlan &p, const hqekv_seg &s);

// The arguments of both launches.
struct TilesHost {
  u32x4 begins;
  uint32_t heads, div_hkv;
  TileTable table;
};
inline TilesHost tiles_host(const SegTable &tb, int64_t Hq, int64_t Hkv) {
  TilesHost h{};
  for (int k = 0; k < HQEKV_MAX_SEGS; ++k) {
    const uint32_t v = k == 0 ? (uint32_t)(Hq / Hkv) : k < tb.nseg ? (uint32_t)tb.begin[k] : 0xffffu;   // (65535 units at most)
    h.begins[k / 2] |= v << (16 * (k & 1));
    if (k >= tb.nseg) continue;
    const SegDev &s = tb.seg[k];
    h.table.seg[k] = TileSeg{s.data, s.scale, s.zero, s.idx, s.slab_tokens, (int32_t)s.pos_base, (int32_t)s.n_tokens, s.bits, s.layout, s.unit_begin};
  }
  h.heads = (uint32_t)Hq | (uint32_t)Hkv << 16;
  h.div_hkv = (uint32_t)(((1ULL << 32) + Hkv - 1) / Hkv);
  return h;
}

int64_t pv_block_tokens(int bits);   // tokens of a p.V block
int launch_qk_tiles(const SegTable &tb, const void *q, void *scores, int64_t B, int64_t Hq, int64_t Hkv, int64_t Tall, const FuseArgs &fz,
                    hipStream_t st);
int launch_pv_tiles(const SegTable &tb, void *p, float *partial, int64_t B, int64_t Hq, int64_t Hkv, int64_t Tall, const FuseArgs &fz,
                    hipStream_t st);
// Short steps in two launches: p.V, the sum of its partial rows and the step's epilogue in one of them (decode_pv.hip).
bool decode_in_two(const hqekv_seg *v_segs, int n_v, int64_t D, int64_t B, int64_t Hq, int64_t Hkv);
bool pv_last_takes(const StepEpilogue &ep, int64_t Tall);
int64_t pv_epilogue_blocks(const StepEpilogue &ep, int64_t Tall);   // workgroups for the epilogue
// The same steps in one launch (decode_step.hip), with the same bits.
constexpr int STEP_UNITS = 20;        // most p.V units (and partial rows) of a (b, kv head) of a short step
constexpr int STEP_RECORDS = 64;      // most tiles, in one launch
int launch_step(const SegTable &kt, const SegTable &vt, const void *q, void *logits, void *probs, void *records, void *pairs, void *out,
                int64_t B, int64_t Hq, int64_t Hkv, int64_t Tall, float inv_sqrt_d, const StepEpilogue &ep, int patience, hipStream_t st);
int launch_pv_last(const SegTable &tb, const void *logits, void *probs, float *partial, int64_t B, int64_t Hq, int64_t Hkv, int64_t Tall,
                   const FuseArgs &fz, const StepEpilogue &ep, hipStream_t st);

}  // namespace hq
