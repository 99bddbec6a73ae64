// A whole short decode step in one launch (see decode_tiles.h).
#include "decode_pv_tile.h"
#include "decode_qk_tile.h"

#pragma clang fp contract(off)

namespace hq {

// The grid's rows are, for every (b, kv head), the q.K^T tiles, then the p.V units, then the epilogue's workgroups.  A tile
// leaves its logits and, once these are acknowledged by memory, a record per head: (max, sum exp) beside the launch's number,
// which no other launch has.  p.V has fetched its positions and touched its rows by then; it reads the records again and again
// until they bear the number, merges them and fetches its logits.  A unit's sums bear the number themselves, two channels in
// sixteen bytes, and the last units' workgroups add them up.  Nothing has to be cleared beforehand: memory that does not hold
// this number, 64 bits of it, is not ready.  (All of this goes past the L2, which the XCDs do not share.)
//
// Nobody depends on being scheduled beside others: a workgroup that has looked `patience` times works through the missing tiles
// or units itself -- the same instructions on the same operands, so that whoever else does them writes the same bits -- and
// goes on (step_again).
//
// Bound by its chain, 8 us whatever the length: entry of the table 0.6 us, operands of q.K^T, products and sums to 2.7 (8 bit and fp16
// 3.1), logits acknowledged 0.3 - 0.6, records seen 0.7, logits fetched and p.V 1.3, sums seen and added 1.5.  What it saves
// against two launches is the end of one and the start of the other, what p.V does ahead of the logits, and 2.4 us of the host.
// A step in two launches / in one, back to back, us (the fp16 / 8 / 4 / 2-bit mix, 32 heads over 8): 512 tokens 10.2 / 8.0, 1k
// 10.3 / 8.2, 2k 10.5 / 8.6, 4k 10.9 / 8.9, 2 x 2k 11.4 / 8.9, 4 x 2k 11.8 / 9.4, 4 x 4k 13.5 / 11.4, 8 x 2k 13.8 / 11.5, 16 x 1k
// 14.3 / 13.5; 40 heads over 8, 2k 10.7 / 8.9, 4 x 2k 12.0 / 9.8.  Beyond twenty units three launches: the same exchange took
// 12.4 us at 8k tokens against 10.9, 16.7 / 12.8 at 16k -- there the bytes take longer than the launches, and p.V's touches stand in
// q.K^T's way.
template <int HP>
union StepLds {
  QtLds<HP> qk;
  struct {
    PtLds<HP, false> tile;
    float red[PT_WAVES][HP][128];
    float ml[2 * HP];
  } pv;
  PtEpilogue ep;
  __device__ StepLds() {}
};

// How long p.V's workgroups keep away from memory that q.K^T's need, in 64 clocks: 0.7 us before they touch their rows, 1.7 after a
// first look at the records that finds some missing, then little.  A step with these / with one clock each, us: 1k tokens 8.0 /
// 8.6, 4k 8.9 / 9.7, 4 x 2k 9.3 / 10.0, 4 x 4k 11.5 / 13.2, 8 x 2k 11.5 / 12.7, 16 x 1k 13.4 / 13.2.
constexpr int STEP_SLEEP_TOUCH = 24, STEP_SLEEP_FIRST = 60, STEP_SLEEP = 2;

struct StepArgs {
  half_t *logits, *probs;
  u32x4 *records;        // (B * Hq, tiles)
  u32x4 *pairs;          // (units, B * Hq, 64)
  half_t *out;
  int64_t Tall;
  uint32_t lo, hi;       // the launch's number
  uint32_t logits_bytes, n_bhq;
  float inv_sqrt_d;
  int32_t patience;
};

// The records of a row, by sixteen lanes, up to 64 of them; false: not all are there after `patience` looks.
__device__ __forceinline__ bool row16_wait(const StepArgs &a, uint32_t row, int n, int lane, int patience, float2 (&sv)[4]) {
  const rsrc_t from = make_rsrc(a.records, a.n_bhq * (uint32_t)n * 16u);
  for (int look = 0;; ++look) {
    bool ready = true;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k == 0 || n > 16 * k) {
        const u32x4 w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(from, (int)((row * (uint32_t)n + (uint32_t)min(lane + 16 * k, n - 1)) * 16u), 0, HQ_THROUGH));
        ready = ready && w[1] == a.lo && w[3] == a.hi;
        const uint32_t m = w[0], l = w[2];   // (bit_cast of a vector's element reads its first)
        sv[k] = make_float2(__builtin_bit_cast(float, m), __builtin_bit_cast(float, l));
      }
    if (__builtin_amdgcn_ballot_w64(!ready) == 0) return true;
    if (look >= patience) return false;
    if (look == 0) __builtin_amdgcn_s_sleep(STEP_SLEEP_FIRST);
    else __builtin_amdgcn_s_sleep(STEP_SLEEP);
  }
}
// The kernel's arguments as they lie in memory.
struct StepKernarg {
  u32x4 k_begins, v_begins;
  const half_t *q;
  uint32_t heads, div_hkv, units;
  int32_t n_bh;
  StepArgs a;
  TileTable kt, vt;
  StepEpilogue ep;
};
struct StepShape {   // a (b, kv head)
  int nrep, row0;    // its first row of (B * Hq)
};
template <int HP, bool EXACT>
__device__ __forceinline__ StepShape step_shape(u32x4 begins, uint32_t heads, uint32_t div_hkv, int bh) {
  const int Hq = heads & 0xffffu, Hkv = heads >> 16, nrep = EXACT ? HP : tiles_nrep(begins), b = tiles_batch_row(Hkv, div_hkv, bh);
  return StepShape{nrep, b * Hq + (bh - b * Hkv) * nrep};
}

// Tile `i` of (b, kv head) `bh`, announced.
template <int HP, bool EXACT>
__device__ __forceinline__ void step_tile(const StepArgs &a, const half_t *q, const TileSeg &sg, StepShape s, int i, int n_k, int bh, int n_bh, int wave, int lane, QtLds<HP> &lds) {
  const int n = lane & 15, r = lane >> 4;
  const half_t *q0 = q + (int64_t)s.row0 * 128;
  u32x4 qv;   // row l % 16 of A: head (l % 16) % HP (rows without a head repeat one, their results are dropped)
  {
    uint32_t w[4];
    load_words<4, Words2<4>>(q0, (uint32_t)min(n % HP, s.nrep - 1) * 256u + 64u * wave + 16u * r, w);
    qv = (u32x4){w[0], w[1], w[2], w[3]};
  }
  const int head = (4 * r) % HP + wave;   // the head this lane finishes
  const bool has_head = head < s.nrep;
  const int row = s.row0 + min(head, s.nrep - 1);
  const QtRowThrough to{make_rsrc(a.logits, a.logits_bytes), (uint32_t)row * (uint32_t)a.Tall * 2u};
  float mm, l;
  qt_unit<HP, true>(sg, i - sg.unit_begin, bh, n_bh, wave, lane, qv, lds, to, has_head, a.inv_sqrt_d, mm, l,
                    [&]() { return q0 + min((4 * (lane >> 4)) % HP + wave, s.nrep - 1) * 128; });
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the wave's own logits: its heads' records say nothing of others)
  if (n == 0 && 4 * r < HP && has_head)
    __builtin_amdgcn_raw_buffer_store_b128((u32x4){__builtin_bit_cast(uint32_t, mm), a.lo, __builtin_bit_cast(uint32_t, l), a.hi},
                                           make_rsrc(a.records, a.n_bhq * (uint32_t)n_k * 16u), (row * n_k + i) * 16, 0, HQ_THROUGH);
}

// The sums of a unit, two channels at a time beside the launch's number: (unit, row of B * Hq, pair of channels).
__device__ __forceinline__ rsrc_t step_pairs(const StepArgs &a, int n_v) { return make_rsrc(a.pairs, (uint32_t)n_v * a.n_bhq * 1024u); }
__device__ __forceinline__ uint32_t step_pair(const StepArgs &a, StepShape s, int unit, int at) { return ((uint32_t)unit * a.n_bhq + (uint32_t)s.row0) * 1024u + 16u * (uint32_t)at; }

// Unit `unit` of p.V, announced; false, and nothing done, where its logits are not there after `patience` looks.
template <int HP, bool EXACT>
__device__ __forceinline__ bool step_unit(const StepArgs &a, const TileSeg &sg, StepShape s, int unit, int n_k, int n_v, int bh, int wave, int lane, StepLds<HP> &sh,
                                          int (&word)[4]) {
  const int n = lane & 15, tid = wave * 64 + lane;
  // While the logits are not there: where they will be, and the unit's rows of codes, scales and zero points into the L2 (a
  // line of the codes per thread, and one of the others).  Codes held in registers across the wait would be twelve copies of it.
  const int block = unit - sg.unit_begin;
  const uint32_t position0 = pt_first_position(sg, block, tid);
  uint32_t touch[2] = {0u, 0u};
  __builtin_amdgcn_s_sleep(STEP_SLEEP_TOUCH);
  {
    const uint32_t t0 = (uint32_t)block * (sg.bits >= 8 ? PtGeom<8>::BLOCK : PT_BLOCK), row_b = 16u * sg.bits;
    const uint32_t left = min((uint32_t)sg.n_tokens - t0, (uint32_t)(sg.bits >= 8 ? PtGeom<8>::BLOCK : PT_BLOCK)), at = 128u * tid;
    const int64_t token = (int64_t)bh * sg.slab_tokens + t0;
    if (at < left * row_b) touch[0] = gload<uint32_t>((const char *)sg.data + token * row_b, at);
    if (sg.bits < 16 && (uint32_t)(tid & 127) * 128u < left * 8u)
      touch[1] = gload<uint32_t>((const char *)(tid < 128 ? sg.scale : sg.zero) + token * 8, (uint32_t)(tid & 127) * 128u);
  }
  if (wave * 4 < s.nrep) {
    float2 sv[4];
    const int first = tid >> 4;
    const bool there = row16_wait(a, (uint32_t)(s.row0 + min(first, s.nrep - 1)), n_k, n, a.patience, sv);
    if (there) {
      const float2 v = row16_merge(nullptr, n_k, n, sv);
      if (n == 0 && first < s.nrep) {
        sh.pv.ml[2 * first] = v.x;
        sh.pv.ml[2 * first + 1] = v.y;
      }
    }
    if (lane == 0) word[wave] = there;
  }
  __syncthreads();
  const bool ready = word[0] && (HP <= 4 || s.nrep <= 4 || word[1]);
  asm volatile("" ::"v"(touch[0]), "v"(touch[1]));
  if (!ready) return false;
  f4_t acc[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) acc[c] = (f4_t){0.f, 0.f, 0.f, 0.f};
  const PtRowsThrough rows{make_rsrc(a.logits, a.logits_bytes), (uint32_t)s.row0 * (uint32_t)a.Tall * 2u, (uint32_t)a.Tall * 2u};
  pt_unit<HP, EXACT, false, true, true, true>(sg, block, 1, bh, wave, lane, rows, a.probs + (int64_t)s.row0 * a.Tall, a.Tall, s.nrep, sh.pv.tile, sh.pv.ml, acc,
                                              position0, [] {}, [] {});
  pt_store_partial<HP, EXACT>(acc, sh.pv.red, wave, lane, s.nrep, [&](int at, float2 sum) {
    __builtin_amdgcn_raw_buffer_store_b128((u32x4){__builtin_bit_cast(uint32_t, sum.x), a.lo, __builtin_bit_cast(uint32_t, sum.y), a.hi}, step_pairs(a, n_v),
                                           (int)step_pair(a, s, unit, at), 0, HQ_THROUGH);
  });
  return true;
}

// The sums of two heads of what all units have left: a lane has two channels of a head, of the even or of the odd units, as
// pt_sum_partials adds them.  -> -1, or a unit that is not there after `patience` looks.
constexpr int STEP_HEADS = 2, STEP_APART = PT_WAVES / STEP_HEADS;
template <int HP>
__device__ __forceinline__ int step_sum(const StepArgs &a, StepShape s, int j, int n_v, int wave, int lane, StepLds<HP> &sh, int (&word)[4]) {
  const int part = wave % STEP_APART;
  const rsrc_t from = step_pairs(a, n_v);
  const int head = STEP_HEADS * j + wave / STEP_APART, at = 64 * head + lane;   // (a head past the last one: read, not stored)
  constexpr int FLIGHT = STEP_UNITS / STEP_APART;
  u32x4 t[FLIGHT];
  int missing = -1;
  for (int look = 0;; ++look) {
    uint64_t no = 0;
    int first = 0;
#pragma unroll
    for (int i = 0; i < FLIGHT; ++i)
      if (STEP_APART * i + part < n_v)
        t[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(from, (int)step_pair(a, s, STEP_APART * i + part, min(at, 64 * s.nrep - 1)), 0, HQ_THROUGH));
#pragma unroll
    for (int i = FLIGHT - 1; i >= 0; --i)
      if (STEP_APART * i + part < n_v) {
        const uint64_t b = __builtin_amdgcn_ballot_w64(t[i][1] != a.lo || t[i][3] != a.hi);
        no |= b;
        first = b ? i : first;
      }
    if (!no) break;
    if (look >= a.patience) {
      missing = STEP_APART * first + part;
      break;
    }
    __builtin_amdgcn_s_sleep(STEP_SLEEP);
  }
  float2 sum = make_float2(0.f, 0.f);
#pragma unroll
  for (int i = 0; i < FLIGHT; ++i)
    if (STEP_APART * i + part < n_v) {
      const uint32_t x = t[i][0], y = t[i][2];
      sum.x += __builtin_bit_cast(float, x);
      sum.y += __builtin_bit_cast(float, y);
    }
  float2 *odd = reinterpret_cast<float2 *>(&sh.pv.red[0][0][0]);
  __syncthreads();
  if (part) odd[wave / STEP_APART * 64 + lane] = sum;
  if (lane == 0) word[wave] = missing;
  __syncthreads();
  const int next = max(max(word[0], word[1]), max(word[2], word[3]));
  if (!part) {
    const float2 v = odd[wave / STEP_APART * 64 + lane];
    sum = make_float2(sum.x + v.x, sum.y + v.y);
    if (next < 0 && head < s.nrep) *reinterpret_cast<uint32_t *>(a.out + (int64_t)s.row0 * 128 + 2 * at) = as_u32(pack_h2((half_t)sum.x, (half_t)sum.y));
  }
  return next;
}
// The statistics of every row, for the ring row; false after `patience` looks at one of them.
template <int HP>
__device__ __forceinline__ bool step_row_stats(const StepArgs &a, int rows, int n_k, int tid, StepLds<HP> &sh, int (&word)[4]) {
  __syncthreads();
  if (tid == 0) word[0] = 1;
  __syncthreads();
  const int l16 = tid & 15;
  for (int row = tid >> 4; row < rows; row += PT_WAVES * 4) {
    float2 sv[4];
    if (!row16_wait(a, (uint32_t)row, n_k, l16, a.patience, sv)) {
      word[0] = 0;
      break;
    }
    const float2 v = row16_merge(nullptr, n_k, l16, sv);
    if (l16 == 0) sh.ep.ml[row] = v;
  }
  __syncthreads();
  return word[0] != 0;
}

// ---- For a workgroup that others have left waiting, out of line and to the end of its work, so that the kernel keeps nothing in
// registers for it: what is missing is done here.  `unit`: the unit that waits (n_v: none), `j`: the group whose sums wait (below
// zero: none); past the units: the epilogue's block.
// Each round brings a tile, a unit or a group's sums.  Nothing is to be kept in registers from one to the next, so the place is
// hidden from the compiler anew: with what it moves out of the loop the function took 0.5 KB of stack per lane, which a queue
// holds for every wave that the chip could run.
typedef const __attribute__((address_space(4))) StepKernarg *step_kernarg_t;
template <int HP, bool EXACT>
__device__ __attribute__((noinline)) void step_again(step_kernarg_t kp, uint32_t lds, uint32_t words, int unit0, int j, int bh0, int blk, int nblk) {
#define HQ_UNIFORM(x_) x_ = __builtin_amdgcn_readfirstlane(x_)   // (the caller's scalars arrive in vector registers)
  HQ_UNIFORM(lds), HQ_UNIFORM(words), HQ_UNIFORM(unit0), HQ_UNIFORM(j), HQ_UNIFORM(bh0), HQ_UNIFORM(blk), HQ_UNIFORM(nblk);
#undef HQ_UNIFORM
  const uint64_t from = (uint64_t)kp;
  kp = (step_kernarg_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(from >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)from));
  int tiles = -1, unit = unit0;   // tiles to do before anything else (-1: not decided)
  const int limit = ((const StepKernarg *)kp)->n_bh * STEP_RECORDS + 4 * STEP_UNITS;
  for (int round = 0; round <= limit; ++round) {
    int bh = bh0, tid = threadIdx.x;
    uint64_t args = (uint64_t)kp;
    uint32_t at = lds, wat = words;
    asm volatile("" : "+s"(bh), "+v"(tid), "+s"(args), "+s"(at), "+s"(wat));
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const StepKernarg &k = *(const StepKernarg *)(step_kernarg_t)args;
    StepLds<HP> &sh = *(StepLds<HP> *)(__attribute__((address_space(3))) StepLds<HP> *)(uintptr_t)at;
    int(&word)[4] = *(int(*)[4])(__attribute__((address_space(3))) int(*)[4])(uintptr_t)wat;
    const int n_k = k.units & 0xffffu, n_v = k.units >> 16;
    const bool rest = unit0 > n_v;
    if (tiles < 0) tiles = rest ? k.n_bh * n_k : unit < n_v ? n_k : 0;
    if (tiles > 0) {
      const int g = rest ? (tiles - 1) / n_k : bh, i = (tiles - 1) % n_k;
      const TileSeg sg = k.kt.seg[tiles_segment(k.k_begins, i)];
      step_tile<HP, EXACT>(k.a, k.q, sg, step_shape<HP, EXACT>(k.k_begins, k.heads, k.div_hkv, g), i, n_k, g, k.n_bh, wave, lane, sh.qk);
      --tiles;
      __syncthreads();   // (the next tile's scales and sums lie where this one's were)
      continue;
    }
    if (rest) {
      step_row_stats<HP>(k.a, k.ep.B * k.ep.Hq, n_k, tid, sh, word);
      step_epilogue_block<false>(k.ep, blk, nblk, sh.ep.ring, PtRingProb<true>{sh.ep.ml});
      return;
    }
    const StepShape s = step_shape<HP, EXACT>(k.k_begins, k.heads, k.div_hkv, bh);
    const int groups = (s.nrep + STEP_HEADS - 1) / STEP_HEADS;
    if (unit < n_v) {
      const TileSeg sg = k.vt.seg[tiles_segment(k.v_begins, unit)];
      step_unit<HP, EXACT>(k.a, sg, s, unit, n_k, n_v, bh, wave, lane, sh, word);   // (its logits are there: first look)
      __syncthreads();
    }
    if (j < 0 || j >= groups) return;
    unit = step_sum<HP>(k.a, s, j, n_v, wave, lane, sh, word);
    if (unit < 0) {
      unit = n_v;
      j += min(n_v, groups);
    }
    __syncthreads();
  }
}

template <int HP, bool EXACT>
__global__ __launch_bounds__(PT_WAVES * 64, HP == 4 ? 5 : 4) void step_kernel(u32x4 k_begins, u32x4 v_begins, const half_t *__restrict__ q, uint32_t heads,
                                                                             uint32_t div_hkv, uint32_t units, int32_t n_bh, StepArgs a, TileTable kt,
                                                                             TileTable vt, StepEpilogue ep) {
  static_assert(QT_WAVES == PT_WAVES, "one workgroup serves both");
  __shared__ __align__(16) StepLds<HP> sh;
  __shared__ int word[4];
  const int bh = blockIdx.x, u = blockIdx.y, n_k = units & 0xffffu, n_v = units >> 16, unit = u - n_k;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const StepShape s = step_shape<HP, EXACT>(k_begins, heads, div_hkv, bh);
  if (u < n_k) {
    const TileSeg sg = kt.seg[tiles_segment(k_begins, u)];
    step_tile<HP, EXACT>(a, q, sg, s, u, n_k, bh, n_bh, wave, lane, sh.qk);
    return;
  }
  const step_kernarg_t kp = (step_kernarg_t)__builtin_amdgcn_kernarg_segment_ptr();
  const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)&sh, words = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)&word;
  if (unit < n_v) {
    const int groups = (s.nrep + STEP_HEADS - 1) / STEP_HEADS, summing = min(n_v, groups);   // the last units' workgroups add up
    int j = unit - (n_v - summing);
    const TileSeg sg = vt.seg[tiles_segment(v_begins, unit)];
    if (!step_unit<HP, EXACT>(a, sg, s, unit, n_k, n_v, bh, wave, lane, sh, word)) {
      __syncthreads();
      step_again<HP, EXACT>(kp, lds, words, unit, j, bh, 0, 0);
      return;
    }
    if (j < 0) return;
    for (; j < groups; j += summing) {
      if (step_sum<HP>(a, s, j, n_v, wave, lane, sh, word) >= 0) {
        __syncthreads();
        step_again<HP, EXACT>(kp, lds, words, n_v, j, bh, 0, 0);
        return;
      }
      __syncthreads();
    }
    return;
  }
  const int blk = (int)((blockIdx.y - n_k - n_v) * gridDim.x + blockIdx.x), nblk = (int)((gridDim.y - n_k - n_v) * gridDim.x);
  if (ep.ring_line && !step_row_stats<HP>(a, ep.B * ep.Hq, n_k, threadIdx.x, sh, word)) {
    __syncthreads();
    step_again<HP, EXACT>(kp, lds, words, n_v + 1, -1, bh, blk, nblk);
    return;
  }
  step_epilogue_block<false>(ep, blk, nblk, sh.ep.ring, PtRingProb<true>{sh.ep.ml});
}

// =============================================================================== host side
int launch_step(const SegTable &kt, const SegTable &vt, const void *q, void *logits, void *probs, void *records, void *pairs, void *out,
                int64_t B, int64_t Hq, int64_t Hkv, int64_t Tall, float inv_sqrt_d, const StepEpilogue &ep, int patience, hipStream_t st) {
  const TilesHost k = tiles_host(kt, Hq, Hkv), v = tiles_host(vt, Hq, Hkv);
  const int64_t nrep = Hq / Hkv, more = pv_epilogue_blocks(ep, Tall);
  const uint64_t number = launch_number();
  const StepArgs a{(half_t *)logits, (half_t *)probs, (u32x4 *)records, (u32x4 *)pairs, (half_t *)out, Tall,
                   (uint32_t)number, (uint32_t)(number >> 32), (uint32_t)(B * Hq * Tall * 2), (uint32_t)(B * Hq), inv_sqrt_d, patience};
  const dim3 grid((unsigned)(B * Hkv), (unsigned)(kt.total_units + vt.total_units + (more + B * Hkv - 1) / (B * Hkv)));
#define LAUNCH(HP_, EXACT_)                                                                                                                               \
  hipLaunchKernelGGL((step_kernel<HP_, EXACT_>), grid, dim3(PT_WAVES * 64), 0, st, k.begins, v.begins, (const half_t *)q, k.heads, k.div_hkv, \
                     (uint32_t)kt.total_units | (uint32_t)vt.total_units << 16, (int32_t)(B * Hkv), a, k.table, v.table, ep)
  if (nrep == 4) LAUNCH(4, true);
  else if (nrep < 4) LAUNCH(4, false);
  else if (nrep == 8) LAUNCH(8, true);
  else LAUNCH(8, false);
#undef LAUNCH
  return check_launch("step_kernel");
}

}  // namespace hq
