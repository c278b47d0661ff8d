// zx_prefill.hip -- blocks of queries attending to K/V straight from the paged FP8 pool:
// one ring step of QuantizedRingAttention (README.md:344), with the step's result merged
// into a running (output, log-sum-exp) so that the steps of a ring compose into full
// attention.  The ring exchange itself needs more than one GPU and is not here.
//
// A block owns (sequence, G query heads of one kv head, a tile of 32 * 4 / G query rows);
// its 4 waves each take one head and 32 rows (two 16-row MFMA tiles), so every K/V tile
// is read from HBM once per block and serves 128 query rows.  Steps of 64 keys (four
// 16-key tiles, each inside one page):
//   * the block loads the step's K and V runs with contiguous 16-byte lane loads (whole
//     cache lines; a thread takes channels 16 g ..+16 of two adjacent keys), one step
//     ahead of the compute; K goes to LDS decoded to bf16 rows, V goes transposed
//     (V^T[channel][key], bf16, the two keys of a thread as one 32-bit word), both double
//     buffered so one block barrier per step suffices;
//   * each wave computes the transposed problem, so that one query row sits in one lane
//     column of every MFMA tile: S^T = K . Q^T on v_mfma_f32_16x16x32_bf16 (K rows as A,
//     Q rows as B), key range / causal mask only on the steps that cross a boundary,
//     online softmax in the exp2 domain with row maxima over the 4 lane rows by
//     v_permlane32/16_swap, P^T kept in registers as the B operand (fp16 by default,
//     see PM below), O^T += V^T . P^T on the matrix cores, and the row sums of P as a
//     ninth tile against ones (the rescale of O skipped unless a row maximum was raised).
// At the end each row is normalised; with MERGE the step's (O, lse2) is combined with
// the running one in o_acc / lse2 (each (row, head) belongs to one block, so no races);
// with the bf16 flag the merged row is also written as bf16.
#include <algorithm>

#include "zx_attn_common.h"

namespace zx {

constexpr int PF_THREADS = 256;
constexpr int PF_KEYS = 64;                  // keys per step
constexpr int PF_KROW = 272;                 // K row in LDS (128 channels bf16 + 16 pad: conflict-free reads)
constexpr int PF_VROW = 144;                 // V^T row (64 keys bf16 + 16 pad)
constexpr int PF_KBYTES = PF_KEYS * PF_KROW;
constexpr int PF_VBYTES = 128 * PF_VROW;
constexpr int PF_RTAB = 64;  // key ranges whose bounds a block keeps in LDS
constexpr int PF_MERGE = 1, PF_WRITE_BF16 = 2, PF_INIT = 4, PF_LAST = 8, PF_FINAL = 16;
// a row's running maximum m is raised only when a score exceeds it by more than this
// (log2 units), so p = 2^(s - m) <= 2^PF_LAZY and O is rarely rescaled
constexpr float PF_LAZY = 8.0f;

struct PrefillArgs {
  const uint16_t *q;  // [n_q][Hq][128] bf16
  const int32_t *cu_q, *q_pos0;
  const uint8_t *pool;
  const float *scales;  // [2][Hkv]
  const int32_t *bt, *kv_begin, *kv_end;  // [n_ranges][n_seqs] key ranges, walked in order
  float *o_acc;   // [n_q][Hq][128] fp32, normalised
  float *lse2;    // [n_q][Hq]
  uint16_t *out;  // [n_q][Hq][128] bf16 (PF_WRITE_BF16)
  int32_t *err;
  int64_t n_pages;
  int32_t n_q_heads, n_kv_heads, page_size, max_blocks, mode, causal, n_ranges, n_seqs;
  int32_t n_qt;  // query tiles per sequence (the grid is n_qt x n_split x head groups x sequences)
  int64_t max_rows;     // rows of a sequence that are computed: max_q_per_seq up to a multiple of 128 / G
  int32_t n_split;      // blocks that share a query tile's keys; each writes a part of its own:
  int64_t part_stride;  // rows (x heads) between the parts in o_acc / lse2
  int32_t *parts;       // [n_qt x head groups x sequences] of them that a tile has
  uint32_t p_magic;
  int32_t p_shift;
  float sm_log2e;  // sm_scale * log2 e
};

__device__ __forceinline__ uint32_t pf_page_of(const PrefillArgs &a, uint32_t t) {
  return (uint32_t)(((uint64_t)t * a.p_magic) >> (31 + a.p_shift));
}

// MFMA k order of a step's keys: the 64 keys form two k-blocks of 32 (one PV MFMA each);
// inside k-block kb, k = 8 kg + 4 KT + i is key 32 kb + 16 KT + 4 kg + i, which is where
// the S^T tiles leave that key (tile 2 kb + KT, lane row kg, element i).  V^T rows hold
// the keys in this order, in 16-byte chunks (8 keys) swizzled by channel / 16.
__device__ __forceinline__ int pf_vslot_byte(int c, int key) {
  const int kb = key >> 5, KT = (key >> 4) & 1, kg = (key >> 2) & 3, i = key & 3;
  return c * PF_VROW + ((((kb << 2) + kg) ^ (c >> 4)) << 4) + 2 * (4 * KT + i);
}

// How P enters P.V (and the row sums, which use the same P):
//   PF_P_F16   P * 2^7 rounded once to fp16 (11 significant bits, relative error <= 2^-11;
//              the 2^7 keeps P's range (<= 2^PF_LAZY) inside fp16 and pushes its
//              subnormal range 7 octaves down), V^T in LDS as fp16 (e4m3 values are exact
//              in fp16), one fp16 MFMA per tile;
//   PF_P_BF16  P rounded once to bf16 (relative error <= 2^-9), one bf16 MFMA per tile,
//              the usual flash-attention numerics;
//   PF_P_EXACT P as bf16 hi + lo, two bf16 MFMAs per tile: P carried to ~2^-17.
constexpr int PF_P_F16 = 0, PF_P_BF16 = 1, PF_P_EXACT = 2;
constexpr float PF_F16_SHIFT = 7.0f;  // log2 of the factor P carries in PF_P_F16
typedef _Float16 att_f16x8 __attribute__((ext_vector_type(8)));

// O^T (or the row sums) += A . B on 16x16x32 tiles, A and B given as the bits of 8 values
__device__ __forceinline__ att_f32x4 pf_mfma_bf16(att_u32x4 a, att_u32x4 b, att_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(att_bf16x8, a), __builtin_bit_cast(att_bf16x8, b),
                                                 c, 0, 0, 0);
}
__device__ __forceinline__ att_f32x4 pf_mfma_f16(att_u32x4 a, att_u32x4 b, att_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(att_f16x8, a), __builtin_bit_cast(att_f16x8, b), c,
                                                0, 0, 0);
}
__device__ __forceinline__ uint32_t pack_f16(float lo, float hi) {
  typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
  f16x2_t v;
  v[0] = (_Float16)lo;
  v[1] = (_Float16)hi;
  return __builtin_bit_cast(uint32_t, v);
}
// 16 e4m3 codes -> 8 fp16 pairs (exact: every e4m3 value is an fp16 value).
__device__ __forceinline__ void decode16_f16(uint4 c, uint32_t (&b)[8]) {
  const uint32_t w[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    b[2 * i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)w[i], 1.0f, false));
    b[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)w[i], 1.0f, true));
  }
}

// Parts of a tile with `steps` steps: as many as the call has room for (the host knows the
// width of the block table only), of at least 2 steps each.  Unused ones end at once, and a
// tile of one part is written as if the call were not cut.  With a table of 32,768 positions
// (exact table in brackets): 64 rows on 448 keys 127 -> 20 us (22; 23 with parts of 4 steps,
// 30 of 8), 16 x 4 rows on 500 19 (30), 4 x 64 rows of new sequences 54 -> 15 (11: the rest
// is the empty blocks and the second launch).
__device__ __forceinline__ int pf_parts(int64_t steps, int n_split) {
  return (int)max((int64_t)1, min((int64_t)n_split, steps / 2));
}

// PARTS: the blocks share each tile's keys (a.n_split > 1).  An instantiation of its own: the
// extra live values cost the kernel without parts 3-7% (a ring of 8 launches over 4 x 8,192
// rows 3,081 -> 3,297 us, exact weights 2,950 -> 3,054).
template <int G, int PM, bool PARTS>
__global__ void __launch_bounds__(PF_THREADS, 2) paged_prefill_mfma_kernel(PrefillArgs a) {
  constexpr bool EXACT = PM == PF_P_EXACT, F16 = PM == PF_P_F16;
  constexpr int D = 128;
  constexpr int QT = 32 * 4 / G;  // query rows per block
  // one-dimensional grid, query tile slowest: the last query tiles see the most keys under
  // a causal mask, so every (head group, sequence)'s last tile is launched first, then
  // every second-to-last, ... (globally longest first: the shortest blocks make the tail)
  const int n_hg = a.n_q_heads / G;
  const int64_t per_rank = (int64_t)n_hg * a.n_seqs;
  int64_t qt_rev = (int64_t)blockIdx.x / per_rank;
  const int rem = (int)((int64_t)blockIdx.x - qt_rev * per_rank);
  int split = 0;
  if constexpr (PARTS) {  // parts of one tile next to each other
    split = (int)(qt_rev % a.n_split);
    qt_rev /= a.n_split;
  }
  const int hg = rem % n_hg, b = rem / n_hg;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, kg = lane >> 4;
  const int grp = a.n_q_heads / a.n_kv_heads;
  const int hq = hg * G + wave % G;
  const int h = (hg * G) / grp;  // the block's KV head (G divides grp: its G query heads share it)
  // What the set-up reads that depends only on the (sequence, head group) is loaded in one
  // round trip: the sequence's queries, its first key range and the head's scales.  Every
  // dependent round trip of a block's set-up or final merge is a wait of that block, and
  // they count where blocks are short: a ring step of 1,024 keys per launch (one launch per
  // step, as a multi-GPU ring runs) took 7% less time per ring with the set-up below (the
  // pages of the first two steps and Q read together, then the first K/V and the block
  // table check) and the running output read in one go at the end.
  const int32_t cq0 = a.cu_q[b], cq1 = a.cu_q[b + 1], qp0_32 = a.q_pos0[b];
  const int32_t kb0 = a.kv_begin[b], ke0 = a.kv_end[b];
  const float sk = a.scales[h], sv = a.scales[a.n_kv_heads + h];
  // (the empty asm takes every value as an operand, so the compiler issues the loads
  // together here instead of sinking each one to its first use past a branch)
  asm volatile("" ::"s"(cq0), "s"(cq1), "s"(qp0_32), "s"(kb0), "s"(ke0), "s"(sk), "s"(sv));
  const int64_t qp0 = qp0_32;
  const int64_t q_lo = cq0;
  const int n_qb = cq1 - cq0;
  const int64_t row0_64 = ((int64_t)a.n_qt - 1 - qt_rev) * QT;
  if (row0_64 >= n_qb) return;
  const int row0_blk = (int)row0_64;
  const int wrow0 = row0_blk + 32 * (wave / G);  // this wave's first row (in the sequence)
  const int64_t page_bytes = 2LL * a.n_kv_heads * a.page_size * D;
  const int64_t head_off = (int64_t)h * a.page_size * D;
  const int64_t v_off = (int64_t)a.n_kv_heads * a.page_size * D;
  const int32_t *bt = a.bt + (int64_t)b * a.max_blocks;
  int32_t e = 0;
  // rows past max_rows (n_qt tiles; max_q_per_seq too small) are not computed: flag it
  if (qt_rev == 0 && a.max_rows < n_qb) e |= ZX_KERR_POS_RANGE;
  const int kmax = a.max_blocks * a.page_size;  // < 2^31 (checked by the host)
  // keys past the block's last query position never count when causal
  const int last_row = min(row0_blk + QT, n_qb) - 1;
  // Range r of this sequence: keys [kb, ke) (ke clipped to the block table), walked in
  // 64-key steps from s_first (kb rounded down to a 16-key tile) while below ke_blk (ke,
  // or the block's last causal key + 1).  All block-uniform.
  struct Range {
    int kb, ke, s_first, ke_blk;
  };
  // With several ranges, their bounds go to LDS in one round trip here: read where the
  // walk reaches them, each would stall the steps for a dependent load.
  __shared__ int32_t rtab[2][PF_RTAB];
  const int n_tab = a.n_ranges > 1 ? min(a.n_ranges, PF_RTAB) : 0;
  // PARTS: ranges that follow each other without a gap (a ring's shards) are walked as one,
  // which saves the blocks of a short part the walk over all ranges (64 rows on 4,032 keys as
  // a ring of 64: 106 us with it, 56 without; 200 when each range was dealt by itself)
  int n_ranges = a.n_ranges, ke_one = ke0;
  if (n_tab) {  // block-uniform
    bool gap = a.n_ranges > PF_RTAB;
    for (int r = threadIdx.x; r < n_tab; r += PF_THREADS) {
      const int64_t i = (int64_t)r * a.n_seqs + b;
      const int32_t kbr = a.kv_begin[i], ker = a.kv_end[i];
      rtab[0][r] = kbr;
      rtab[1][r] = ker;
      if constexpr (PARTS) gap |= kbr < 0 || ker < kbr || (r > 0 && a.kv_end[i - a.n_seqs] != kbr);
    }
    if constexpr (PARTS) {
      if (!__syncthreads_or(gap)) {
        n_ranges = 1;
        ke_one = __builtin_amdgcn_readfirstlane(rtab[1][n_tab - 1]);
      }
    } else {
      __syncthreads();
    }
  }
  auto steps_of = [](const Range &g) -> int {
    return g.s_first < g.ke_blk ? (g.ke_blk - g.s_first - 1) / PF_KEYS + 1 : 0;
  };
  auto range = [&](int r) -> Range {
    Range g;
    const int64_t i = (int64_t)r * a.n_seqs + b;
    int32_t kbr, ker;
    if (r == 0) {
      kbr = kb0;
      ker = ke_one;
    } else if (r < n_tab) {
      kbr = __builtin_amdgcn_readfirstlane(rtab[0][r]);
      ker = __builtin_amdgcn_readfirstlane(rtab[1][r]);
    } else {
      kbr = a.kv_begin[i];
      ker = a.kv_end[i];
    }
    g.kb = kbr > 0 ? kbr : 0;
    g.ke = ker;
    if (g.ke > kmax) {
      e |= ZX_KERR_POS_RANGE;
      g.ke = kmax;
    }
    g.ke_blk = a.causal ? (int)max((int64_t)-1, min((int64_t)g.ke, qp0 + last_row + 1)) : g.ke;
    g.s_first = (g.kb / 16) * 16;
    return g;
  };
  // PARTS: the steps of all ranges, laid end to end, are dealt to the tile's blocks in equal
  // runs; this block's is [part_lo, part_hi).  (Dealt range by range, ranges with fewer steps
  // than there are parts leave the same parts empty each time.)
  int64_t part_lo = 0, part_hi = 0;
  if constexpr (PARTS) {
    int64_t total = 0;
    for (int r = 0; r < n_ranges; ++r) total += steps_of(range(r));
    const int parts = pf_parts(total, a.n_split);
    if (split >= parts) {  // block-uniform exit
      if (e && a.err && threadIdx.x == 0) atomicOr(a.err, e);
      return;
    }
    if (split == 0 && threadIdx.x == 0) a.parts[qt_rev * per_rank + rem] = parts;
    if (parts == 1) {  // the whole tile: its rows go to out, nothing is combined
      a.mode = PF_WRITE_BF16;
      part_hi = total;
    } else {  // normalised rows and log2 sums of the part's own
      a.mode = PF_MERGE | PF_INIT;
      a.o_acc += split * a.part_stride * 128;
      a.lse2 += split * a.part_stride;
      part_lo = total * split / parts;
      part_hi = total * (split + 1) / parts;
    }
  }
  // range g, whose first step is step `before` of the tile, cut to this block's run
  auto cut = [&](Range &g, int64_t &before) {
    const int64_t n = steps_of(g), lo = max((int64_t)0, part_lo - before), hi = min(n, part_hi - before);
    before += n;
    if (lo >= hi) {
      g.ke = g.ke_blk = g.s_first;
      return;
    }
    if (hi < n) g.ke = g.ke_blk = g.s_first + PF_KEYS * (int)hi;
    g.s_first += PF_KEYS * (int)lo;
    g.kb = max(g.kb, g.s_first);
  };
  // the first range with a step at or after r (n_ranges if none); r grows from call to call
  int64_t before = 0;
  auto next_range = [&](int r, Range &g) -> int {
    for (; r < n_ranges; ++r) {
      g = range(r);
      if constexpr (PARTS) cut(g, before);
      if (g.s_first < g.ke_blk) return r;
    }
    return n_ranges;
  };
  Range cur;
  int rc = next_range(0, cur);
  // rows that reach no key still have something to write on a first step (the empty
  // running output), on a step that writes bf16 for every row, and on a FINAL ring's last
  // step (rows beyond the keys, finished now)
  const bool rows_without_keys_write =
      (a.mode & PF_INIT) ||
      ((a.mode & PF_WRITE_BF16) && (!(a.mode & PF_FINAL) || (a.mode & PF_LAST)));
  // a FINAL step leaves rows below kv_begin alone: a block of such rows only would read
  // the running output for nothing
  const bool rows_all_done = (a.mode & PF_FINAL) && !(a.mode & PF_INIT) && qp0 + last_row < (int64_t)kb0;
  if ((rc == n_ranges && !rows_without_keys_write) || rows_all_done) {
    // no key of any range reaches the block's rows: merging would leave o_acc and lse2 as
    // they are, and a FINAL step's rows below kv_begin were finished before (block-uniform
    // exit)
    if (e && a.err && threadIdx.x == 0) atomicOr(a.err, e);
    return;
  }

  __shared__ __attribute__((aligned(16))) uint8_t kst[2][PF_KBYTES];
  __shared__ __attribute__((aligned(16))) uint8_t vtl[2][PF_VBYTES];

  // every page the block may load inside the pool? (then the steps skip the per-tile
  // block-table checks; otherwise tiles on bad pages count as masked).  Found below, once
  // the first step's loads are in flight.
  bool all_ok = false;

  // Q rows as the B operand of S^T = K . Q^T: lane (n, kg) of row tile rt holds row
  // wrow0 + 16 rt + n, channels 32 kg + 8 c ..+8 for MFMA c (the K operand's channel order);
  // loaded below, after the first step's page lookup
  att_bf16x8 qa[2][4];
  const float qs = sk * a.sm_log2e;  // K's dequant scale folds into the scores
  const float vscale = sv;

  // O^T tiles: o[rt][jt] holds channels 16 jt + 4 kg ..+4 of row 16 rt + n; m per row.
  // The softmax denominator l is a ninth tile on the matrix cores: V^T rows of ones, so
  // every element of ol[rt] is the row's sum of the same P that O uses.
  att_f32x4 o[2][8], ol[2];
  float m[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
    for (int jt = 0; jt < 8; ++jt) o[rt][jt] = att_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    ol[rt] = att_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    m[rt] = -INFINITY;
  }
  const uint32_t one2 = F16 ? 0x3C003C00u : 0x3F803F80u;  // two ones (fp16 / bf16)
  const att_u32x4 ones = {one2, one2, one2, one2};
  // the factor 2^PF_F16_SHIFT that P carries in PF_P_F16 (it cancels in O / l)
  const float p_shift = F16 ? PF_F16_SHIFT : 0.0f;

  // block-cooperative load of one step: thread t moves 16 bytes of K and of V of keys
  // 2 (t / 8) and 2 (t / 8) + 1 (so wave w loads 16-key tile w), channels 16 (t % 8) ..+16;
  // tiles past the range or on a bad page load through zero-length resources
  const int kp2 = threadIdx.x >> 3, g8 = threadIdx.x & 7;
  const int kk0 = 2 * kp2;
  auto tile_ok = [&](int tp, int ke) -> bool {  // uniform
    if (tp >= ke) return false;
    if (all_ok) return true;
    const int64_t page = bt[pf_page_of(a, (uint32_t)tp)];
    return page >= 0 && page < a.n_pages;
  };
  // a step's page, looked up one step before its K/V loads are issued, so that the
  // block-table read is never waited for on its own (3% on the ring workload).  The row's
  // byte size fits the resource: page_size >= 16 and max_blocks * page_size < 2^31.
  const __amdgpu_buffer_rsrc_t rbt = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int32_t *>(bt), (short)0, a.max_blocks * (int)sizeof(int32_t), 0x00020000);
  struct StepPage {
    int tc, live;
    uint32_t bi;
    int32_t page;
  };
  auto lookup_step = [&](int s0, int ke) -> StepPage {
    StepPage p;
    const int tp = s0 + 16 * wave;  // this wave's 16-key tile (scalar: the buffer resources stay in SGPRs)
    p.live = max(0, min(16, ke - tp));
    p.tc = tp < ke ? tp : (ke > 0 ? ke - 1 : 0);
    p.bi = pf_page_of(a, (uint32_t)p.tc);
    // a range-checked load (entries past the block table read as 0; a tile with no key
    // never uses its page), issued without a branch so the wait for it can be counted
    p.page = __builtin_amdgcn_raw_buffer_load_b32(rbt, (int)(p.bi * 4u), 0, 0);
    return p;
  };
  auto issue_step = [&](const StepPage &p, att_u32x4 (&kc)[2], att_u32x4 (&vc)[2]) {
    const int64_t page = __builtin_amdgcn_readfirstlane(p.page);
    const bool ok = p.live > 0 && page >= 0 && page < a.n_pages;
    e |= (p.live > 0 && !ok) ? ZX_KERR_PAGE_RANGE : 0;
    const int nrec = ok ? p.live * D : 0;
    const uint8_t *src =
        a.pool + (ok ? page * page_bytes + head_off + (int64_t)(p.tc - (int)p.bi * a.page_size) * D : 0);
    const __amdgpu_buffer_rsrc_t rk =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(src), (short)0, nrec, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(src + (ok ? v_off : 0)), (short)0, nrec, 0x00020000);
    const int off = (kk0 & 15) * D + 16 * g8;
    // default cache policy: other query tiles read the same pages soon after (4 x 8,192 causal:
    // 2.36 -> 2.30 ms, exact mode 3.14 -> 2.99 ms against nontemporal loads)
    kc[0] = __builtin_amdgcn_raw_buffer_load_b128(rk, off, 0, 0);
    kc[1] = __builtin_amdgcn_raw_buffer_load_b128(rk, off + D, 0, 0);
    vc[0] = __builtin_amdgcn_raw_buffer_load_b128(rv, off, 0, 0);
    vc[1] = __builtin_amdgcn_raw_buffer_load_b128(rv, off + D, 0, 0);
  };
  // K/V of one step stored into an LDS buffer, in 8 pieces so that the store can be spread
  // over the matrix products of the step before: 0, 1 the two K rows (decoded once per
  // block, read as bf16 by the 4 waves); 2 the V decode into v0, v1; 3 .. 6 two V^T channel
  // pairs each (channel c = 16 g8 + 2 p (+1) gets keys kk0, kk0 + 1, adjacent k slots, as
  // one word); 7 nothing
  auto store_piece = [&](int buf, int j, const att_u32x4 (&kc)[2], const att_u32x4 (&vc)[2], uint32_t (&v0)[8],
                         uint32_t (&v1)[8]) {
    if (j < 2) {
      uint32_t kb8[8];
      decode16_bf16(make_uint4(kc[j].x, kc[j].y, kc[j].z, kc[j].w), kb8);
      uint4 *kd = reinterpret_cast<uint4 *>(&kst[buf][(kk0 + j) * PF_KROW + 32 * g8]);
      kd[0] = make_uint4(kb8[0], kb8[1], kb8[2], kb8[3]);
      kd[1] = make_uint4(kb8[4], kb8[5], kb8[6], kb8[7]);
    } else if (j == 2) {
      if constexpr (F16) {
        decode16_f16(make_uint4(vc[0].x, vc[0].y, vc[0].z, vc[0].w), v0);
        decode16_f16(make_uint4(vc[1].x, vc[1].y, vc[1].z, vc[1].w), v1);
      } else {
        decode16_bf16(make_uint4(vc[0].x, vc[0].y, vc[0].z, vc[0].w), v0);
        decode16_bf16(make_uint4(vc[1].x, vc[1].y, vc[1].z, vc[1].w), v1);
      }
    } else if (j < 7) {
      const int slot0 = pf_vslot_byte(16 * g8, kk0);  // channel 16 g8; the others add c * PF_VROW
#pragma unroll
      for (int pp = 0; pp < 2; ++pp) {
        const int p = 2 * (j - 3) + pp;
        uint8_t *row = &vtl[buf][slot0 + 2 * p * PF_VROW];
        *reinterpret_cast<uint32_t *>(row) = __builtin_amdgcn_perm(v1[p], v0[p], 0x05040100u);
        *reinterpret_cast<uint32_t *>(row + PF_VROW) = __builtin_amdgcn_perm(v1[p], v0[p], 0x07060302u);
      }
    }
  };
  auto store_step = [&](int buf, const att_u32x4 (&kc)[2], const att_u32x4 (&vc)[2]) {
    uint32_t v0[8], v1[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) store_piece(buf, j, kc, vc, v0, v1);
  };

  // one step: S^T, softmax, then the P.V products with the next step's K/V stored between
  // them
  auto compute_step = [&](int buf, int s0, int kb, int ke, const att_u32x4 (&kc)[2], const att_u32x4 (&vc)[2]) {
    bool tok[4];
#pragma unroll
    for (int KT = 0; KT < 4; ++KT) tok[KT] = tile_ok(s0 + 16 * KT, ke);
    // S^T tiles: sc[rt][KT] lane (n, kg) holds keys 16 KT + 4 kg + i of row 16 rt + n
    att_f32x4 sc[2][4];
    // A operand: key 16 KT + n, channels 32 kg + 8 c ..+8, read one tile ahead
    att_bf16x8 kar[2][4];
    auto ld_ka = [&](int KT, att_bf16x8 (&dst)[4]) {
      const uint8_t *kr = &kst[buf][(16 * KT + n) * PF_KROW + kg * 64];
#pragma unroll
      for (int c = 0; c < 4; ++c)
        dst[c] = __builtin_bit_cast(att_bf16x8, *reinterpret_cast<const att_u32x4 *>(kr + 16 * c));
    };
    ld_ka(0, kar[0]);
    // wave priority: low while this wave issues its products, high for its softmax and the
    // rest of the step, so that on a SIMD the other block's wave (in another phase) keeps
    // the matrix core fed while this one's VALU work goes first (3% on the ring workload;
    // the exact mode, with twice the P.V products, loses 1% with it and keeps one level)
    if constexpr (!EXACT) __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int KT = 0; KT < 4; ++KT) {
      if (KT + 1 < 4) ld_ka(KT + 1, kar[(KT + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      const att_bf16x8 (&ka)[4] = kar[KT & 1];
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        att_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < 4; ++c) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[c], qa[rt][c], acc, 0, 0, 0);
        sc[rt][KT] = acc;
      }
    }
    if constexpr (!EXACT) __builtin_amdgcn_s_setprio(1);
    // wave-uniform: every (row, key) of the step counts, no mask needed (and qs >= 0, so
    // the row maximum of s * qs is qs times the maximum of s)
    const bool full = tok[0] && tok[1] && tok[2] && tok[3] && s0 >= kb && s0 + PF_KEYS <= ke &&
                      wrow0 + 32 <= n_qb && qs >= 0.0f &&
                      (!a.causal || (int64_t)s0 + PF_KEYS - 1 <= qp0 + wrow0);
    float alpha[2];
    bool grow_any = false;
    att_u32x4 ph[2][2], pl[2][2];  // [rt][k-block] P^T (hi) / lo as 16-bit pairs: word 2 KT + i / 2
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const int r = wrow0 + 16 * rt + n;
      // last key position the row may see (keys are < 2^31)
      const int lim = (r < n_qb) ? (a.causal ? (int)min(max(qp0 + r, (int64_t)-1), (int64_t)INT32_MAX) : INT32_MAX)
                                 : -1;
      auto valid = [&](int KT, int i) {  // branch-free
        const int kp = s0 + 16 * KT + 4 * kg + i;
        return tok[KT] & (kp >= kb) & (kp < ke) & (kp <= lim);
      };
      float mx = -INFINITY;
      if (full) {
#pragma unroll
        for (int KT = 0; KT < 4; ++KT)
#pragma unroll
          for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sc[rt][KT][i]);
        mx *= qs;
      } else {
#pragma unroll
        for (int KT = 0; KT < 4; ++KT)
#pragma unroll
          for (int i = 0; i < 4; ++i) mx = fmaxf(mx, valid(KT, i) ? sc[rt][KT][i] * qs : -INFINITY);
      }
      mx = xrow_max(mx);
      const bool grow = mx > m[rt] + PF_LAZY;  // a row with no key yet grows at its first key
      const float mn = grow ? mx : m[rt];
      const float ms = mn == -INFINITY ? 0.0f : mn;  // a row with no key yet keeps p = 0
      alpha[rt] = grow ? __builtin_amdgcn_exp2f(m[rt] - ms) : 1.0f;
      grow_any |= grow;
      m[rt] = mn;
      // exponent s qs - m, -inf for the masked (row, key) pairs (qs >= 0 keeps the
      // unmasked exponents <= PF_LAZY; with qs < 0 every step takes the masked branch,
      // where the maximum was taken over s qs itself)
      float xe[4][4];
#pragma unroll
      for (int KT = 0; KT < 4; ++KT)
#pragma unroll
        for (int i = 0; i < 4; ++i) xe[KT][i] = __builtin_fmaf(sc[rt][KT][i], qs, p_shift - ms);
      if (!full) {
#pragma unroll
        for (int KT = 0; KT < 4; ++KT)
#pragma unroll
          for (int i = 0; i < 4; ++i) xe[KT][i] = valid(KT, i) ? xe[KT][i] : -INFINITY;
      }
#pragma unroll
      for (int KT = 0; KT < 4; ++KT)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float p0 = __builtin_amdgcn_exp2f(xe[KT][2 * j]), p1 = __builtin_amdgcn_exp2f(xe[KT][2 * j + 1]);
          const uint32_t hw = F16 ? pack_f16(p0, p1) : pack_bf16(p0, p1);
          ph[rt][KT >> 1][2 * (KT & 1) + j] = hw;
          if constexpr (EXACT)
            pl[rt][KT >> 1][2 * (KT & 1) + j] =
                pack_bf16(p0 - __uint_as_float(hw << 16), p1 - __uint_as_float(hw & 0xFFFF0000u));
        }
    }
    // rescale O only when some row's maximum was raised
    if (__builtin_amdgcn_ballot_w64(grow_any)) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
        for (int jt = 0; jt < 8; ++jt) o[rt][jt] *= alpha[rt];
        ol[rt] *= alpha[rt];
      }
    }
    // the next step's K/V goes into the other LDS buffer (free since the last barrier), one
    // store piece per P.V tile, so that its VALU and LDS work sit beside the products (2%
    // on the ring workload against storing it whole before them)
    uint32_t nv0[8], nv1[8];  // the next step's V, decoded by store piece 2
    // A operand per 16-channel tile and k-block: V^T[channel 16 jt + n][k 8 kg ..+8],
    // read PVD tiles ahead of its products (the scheduling barrier keeps the compiler
    // from sinking the reads next to their use: 2% on the ring workload; one tile ahead
    // measured 2% faster than two once the blocks were launched longest first)
    constexpr int PVD = 1;
    att_u32x4 avr[PVD + 1][2];
    auto ld_av = [&](int jt, att_u32x4 (&dst)[2]) {
      const int ch = 16 * jt + n;
#pragma unroll
      for (int kbk = 0; kbk < 2; ++kbk)
        dst[kbk] = *reinterpret_cast<const att_u32x4 *>(&vtl[buf][ch * PF_VROW + ((((kbk << 2) + kg) ^ jt) << 4)]);
    };
#pragma unroll
    for (int jt = 0; jt < PVD; ++jt) ld_av(jt, avr[jt]);
    if constexpr (!EXACT) __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int jt = 0; jt < 8; ++jt) {
      if (jt + PVD < 8) ld_av(jt + PVD, avr[(jt + PVD) % (PVD + 1)]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kbk = 0; kbk < 2; ++kbk) {
        const att_u32x4 av = avr[jt % (PVD + 1)][kbk];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          if constexpr (F16) {
            o[rt][jt] = pf_mfma_f16(av, ph[rt][kbk], o[rt][jt]);
          } else {
            o[rt][jt] = pf_mfma_bf16(av, ph[rt][kbk], o[rt][jt]);
            if constexpr (EXACT) o[rt][jt] = pf_mfma_bf16(av, pl[rt][kbk], o[rt][jt]);
          }
        }
      }
      store_piece(buf ^ 1, jt, kc, vc, nv0, nv1);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int kbk = 0; kbk < 2; ++kbk)
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        if constexpr (F16) {
          ol[rt] = pf_mfma_f16(ones, ph[rt][kbk], ol[rt]);
        } else {
          ol[rt] = pf_mfma_bf16(ones, ph[rt][kbk], ol[rt]);
          if constexpr (EXACT) ol[rt] = pf_mfma_bf16(ones, pl[rt][kbk], ol[rt]);
        }
      }
    if constexpr (!EXACT) __builtin_amdgcn_s_setprio(1);
  };

  // steps: data of step s + 1 loaded into registers and the page of step s + 2 looked up
  // while step s computes; one barrier per step (the LDS buffers alternate).  The steps of
  // the ranges follow each other (the step after a range's last one is the next non-empty
  // range's first), with the running row maxima, O and row sums carried in registers from
  // range to range.  The last step also loads and stores a step after it (zero-length
  // loads; that buffer is never read).  Positions: p0 the step being computed, p1 the next
  // one (K/V loading), p2 the one after (page looked up); a position past the last range
  // stays there (s = 0, ke = 0).
  struct Pos {
    int s, rc;
    Range g;
  };
  auto advance = [&](const Pos &p) -> Pos {
    Pos q = p;
    if (p.rc >= n_ranges) return q;
    q.s = p.s + PF_KEYS;
    if (q.s >= p.g.ke_blk) {
      q.rc = next_range(p.rc + 1, q.g);
      q.s = q.rc < n_ranges ? q.g.s_first : 0;
    }
    return q;
  };
  auto ke_of = [&](const Pos &p) { return p.rc < n_ranges ? p.g.ke : 0; };
  att_u32x4 kc[2], vc[2];
  Pos p0 = {cur.s_first, rc, cur};
  // the pages of the first two steps and Q are read together, then the first step's K/V
  // and the block-table check
  StepPage pg0 = {0, 0, 0u, 0};
  if (p0.rc < n_ranges) pg0 = lookup_step(p0.s, p0.g.ke);
  Pos p1 = advance(p0);
  StepPage pg1 = lookup_step(p1.s, ke_of(p1));
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int r = wrow0 + 16 * rt + n;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      att_u32x4 w = {0u, 0u, 0u, 0u};
      if (r < n_qb) {
        const uint4 x =
            *reinterpret_cast<const uint4 *>(a.q + ((q_lo + r) * a.n_q_heads + hq) * D + kg * 32 + c * 8);
        w = att_u32x4{x.x, x.y, x.z, x.w};
      }
      qa[rt][c] = __builtin_bit_cast(att_bf16x8, w);
    }
  }
  if (p0.rc < n_ranges) issue_step(pg0, kc, vc);
  {
    bool bad = false;
    int64_t at = 0;
    for (int r = 0; r < n_ranges; ++r) {
      Range g = range(r);
      if constexpr (PARTS) cut(g, at);
      if (g.s_first >= g.ke) continue;
      const int p_lo = (int)pf_page_of(a, (uint32_t)g.s_first), p_hi = (int)pf_page_of(a, (uint32_t)(g.ke - 1));
      for (int pi = p_lo + (int)threadIdx.x; pi <= p_hi; pi += PF_THREADS) {
        const int64_t pg = bt[pi];
        bad |= pg < 0 || pg >= a.n_pages;
      }
    }
    all_ok = !__syncthreads_or(bad);
  }
  if (p0.rc < n_ranges) store_step(0, kc, vc);
  __syncthreads();
  int buf = 0;
  while (p0.rc < n_ranges) {
    const Pos p2 = advance(p1);
    issue_step(pg1, kc, vc);
    const StepPage pg2 = lookup_step(p2.s, ke_of(p2));
    compute_step(buf, p0.s, p0.g.kb, p0.g.ke, kc, vc);
    __syncthreads();
    buf ^= 1;
    p0 = p1;
    p1 = p2;
    pg1 = pg2;
  }

  // rows: normalise; merge; store channels 16 jt + 4 kg ..+4.  The running output and
  // log-sum-exp being merged into are read first, all at once (rows past the sequence's
  // end read its last row and discard it).
  const bool merge_old = (a.mode & PF_MERGE) && !(a.mode & PF_INIT);
  // the merged rows go back into the running output unless this is a ring's last step
  const bool keep = (a.mode & PF_MERGE) && !(a.mode & PF_LAST);
  float lse_prev[2];
  float4 o_prev[2][8];
  if (merge_old) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const int64_t row = (q_lo + min(wrow0 + 16 * rt + n, n_qb - 1)) * a.n_q_heads + hq;
      lse_prev[rt] = a.lse2[row];
#pragma unroll
      for (int jt = 0; jt < 8; ++jt) o_prev[rt][jt] = *reinterpret_cast<const float4 *>(a.o_acc + row * D + 16 * jt + 4 * kg);
    }
  }
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int r = wrow0 + 16 * rt + n;
    const float lt = ol[rt][0];
    if (r >= n_qb) continue;
    // FINAL: rows below kv_begin were finished by an earlier step (there is none before
    // the first); rows below kv_end (all rows on the last step) are finished by this one
    // and go to out only
    const int64_t pos = qp0 + r;
    const bool fin_mode = (a.mode & PF_FINAL) != 0;
    if (fin_mode && !(a.mode & PF_INIT) && pos < kb0) continue;
    const bool fin = fin_mode && (pos < ke0 || (a.mode & PF_LAST));
    const bool keep_row = keep && !fin;
    const bool bf16_row = (a.mode & PF_WRITE_BF16) && (!fin_mode || fin);
    const float lse_new = lt > 0.0f ? m[rt] + (__builtin_amdgcn_logf(lt) - p_shift) : -INFINITY;
    const float inv = lt > 0.0f ? vscale / lt : 0.0f;  // V's dequant scale applied once, here
    const int64_t row = (q_lo + r) * a.n_q_heads + hq;
    float wa = 0.0f, wb = 1.0f, lse = lse_new;
    if (merge_old) {
      const float lse_old = lse_prev[rt];
      const float mm = fmaxf(lse_old, lse_new);
      if (mm == -INFINITY) {
        wa = 0.0f;
        wb = 0.0f;
        lse = -INFINITY;
      } else {
        const float ea = __builtin_amdgcn_exp2f(lse_old - mm), eb = __builtin_amdgcn_exp2f(lse_new - mm);
        const float den = ea + eb;
        wa = ea / den;
        wb = eb / den;
        lse = mm + __builtin_amdgcn_logf(den);
      }
    }
#pragma unroll
    for (int jt = 0; jt < 8; ++jt) {
      const int64_t idx = row * D + 16 * jt + 4 * kg;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = o[rt][jt][i] * inv * wb;
      if (merge_old) {  // also at weight 0, so that a NaN of an earlier step stays (0 x NaN)
        const float4 old = o_prev[rt][jt];
        v[0] += wa * old.x;
        v[1] += wa * old.y;
        v[2] += wa * old.z;
        v[3] += wa * old.w;
      }
      if (keep_row) *reinterpret_cast<float4 *>(a.o_acc + idx) = make_float4(v[0], v[1], v[2], v[3]);
      if (bf16_row)
        *reinterpret_cast<uint2 *>(a.out + idx) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
    }
    if (keep_row && kg == 0) a.lse2[row] = lse;
  }
  if (e && a.err) atomicOr(a.err, e);
}

// ---------------------------------------------------------------- 64 rows per wave
//
// The same problem for large prefills that write their rows as bf16 (no running output):
// 64 query rows per wave (two groups of 32), 32x32x16 matrix tiles, one wave per SIMD with
// the registers of two.  The kernel above is bound by latencies that two waves per SIMD do
// not hide and reads every K/V operand from LDS for 32 rows (LDS active 56% of the cycles, 21%
// here); with 64 rows the operand traffic halves, and one instruction stream is laid out by
// hand:
//   * S^T of step j (32 matrix instructions) beside the decode and store of step j + 1's K
//     and V and the weights of the step's first 32 keys;
//   * P.V of step j - 1 beside the weights of the last 32 keys and the packing of P, each
//     chunk of P right after the products that read its predecessor.
// Counters of 4 x 8,192 causal (2.16 ms): matrix cores busy 43% of the SIMD cycles, vector
// instructions issued in 42%, waits 27%; a step of 64 keys takes about 4,800 cycles, start and
// end of a block included, 2,048 of them matrix time.
// No running maximum is computed in these steps: the weights are taken under the maxima the
// rows have, and only if a lane's sum of 16 weights exceeds 2^PF_LAZY (a score has outgrown
// its maximum by PF_LAZY, or many have by 4 and more), or where masks apply or a row has no
// key yet, the step's S^T is made again and the maxima are looked at; a repeated step
// raises every maximum that a score exceeds, after which no sum can trip the test until
// scores grow again (4 x 8,192 causal, all keys but the first 64 at 6 above those: 3,430
// us where only scores beyond PF_LAZY raised it, 2,081 so).  (K has three buffers in LDS for that, V^T four: a wave may be one
// step ahead of another).  Looking at the maxima in every step cost 12% (2.17 against 2.10
// ms); leaving its exponentials in one half of the step, with scalar page lookups between
// the halves, 2.22 ms.
// 4 x 8,192 causal, Hq 32 / Hkv 8 (one launch): 2.31 -> 2.18 ms on one box (2.10 on another,
// 1,045 TFLOP/s); 2 x 4,096 not causal 620 -> 572 us; 2,048 rows on 8,192 cached 387 -> 365 us.
typedef _Float16 pw_f16x2 __attribute__((ext_vector_type(2)));
typedef float att_f32x16 __attribute__((ext_vector_type(16)));
constexpr int PW_ROWS = 64;                   // query rows per wave and per block
constexpr int PW_KBYTES = PF_KEYS * PF_KROW;  // one K buffer (of 3)
constexpr int PW_VBYTES = 128 * PF_VROW;      // one V^T buffer (of 4)

__device__ __forceinline__ att_f32x16 pw_mfma_bf16(att_u32x4 a, att_u32x4 b, att_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(att_bf16x8, a), __builtin_bit_cast(att_bf16x8, b),
                                                 c, 0, 0, 0);
}
__device__ __forceinline__ att_f32x16 pw_mfma_f16(att_u32x4 a, att_u32x4 b, att_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(att_f16x8, a), __builtin_bit_cast(att_f16x8, b), c,
                                                0, 0, 0);
}

// V^T in LDS: row 8 (c % 16) + c / 16 holds channel c, so that a store of a wave (lanes'
// channels 16 apart) falls on rows next to each other and no swizzle is needed: the operand
// reads are one base plus constants.  Within a row the 64 keys are in the order in which
// the S^T tiles leave them: chunk kc (16 keys), lane half hl, element j (8) is key
// 16 kc + 8 (j / 4) + 4 hl + j % 4, at byte 32 kc + 16 hl + 2 j.
__device__ __forceinline__ int pw_vslot_byte(int c, int key) {
  const int kc = key >> 4, y = key & 15;
  return (8 * (c & 15) + (c >> 4)) * PF_VROW + 32 * kc + 16 * ((y >> 2) & 1) + 2 * (4 * (y >> 3) + (y & 3));
}

template <int PM>
__global__ void __launch_bounds__(PF_THREADS, 1) paged_prefill_wide_kernel(PrefillArgs a) {
  constexpr bool F16 = PM == PF_P_F16;
  constexpr int D = 128;
  constexpr int G = 4, QT = PW_ROWS;  // query heads (one per wave) and rows per block
  const int n_hg = a.n_q_heads / G;
  const int64_t per_rank = (int64_t)n_hg * a.n_seqs;
  const int64_t qt_rev = (int64_t)blockIdx.x / per_rank;
  const int rem = (int)((int64_t)blockIdx.x - qt_rev * per_rank);
  const int hg = rem % n_hg, b = rem / n_hg;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, hl = lane >> 5;
  const int grp = a.n_q_heads / a.n_kv_heads;
  const int hq = hg * G + wave;
  const int h = (hg * G) / grp;
  const int32_t cq0 = a.cu_q[b], cq1 = a.cu_q[b + 1], qp0_32 = a.q_pos0[b];
  const int32_t kb0 = a.kv_begin[b], ke0 = a.kv_end[b];
  const float sk = a.scales[h], sv = a.scales[a.n_kv_heads + h];
  // (together: see the kernel above)
  asm volatile("" ::"s"(cq0), "s"(cq1), "s"(qp0_32), "s"(kb0), "s"(ke0), "s"(sk), "s"(sv));
  const int64_t qp0 = qp0_32;
  const int64_t q_lo = cq0;
  // rows past max_rows (max_q_per_seq too small) are not computed: flagged below
  const bool rows_left_out = a.max_rows < cq1 - cq0;
  const int n_qb = rows_left_out ? (int)a.max_rows : cq1 - cq0;
  const int64_t row0_64 = ((int64_t)a.n_qt - 1 - qt_rev) * QT;
  if (row0_64 >= n_qb) return;
  const int row0_blk = (int)row0_64;
  const int wrow0 = row0_blk;  // all waves: the same rows of their own head
  const int64_t page_bytes = 2LL * a.n_kv_heads * a.page_size * D;
  const int64_t head_off = (int64_t)h * a.page_size * D;
  const int64_t v_off = (int64_t)a.n_kv_heads * a.page_size * D;
  const int32_t *bt = a.bt + (int64_t)b * a.max_blocks;
  int32_t e = 0;
  if (qt_rev == 0 && rows_left_out) e |= ZX_KERR_POS_RANGE;
  const int kmax = a.max_blocks * a.page_size;
  const int last_row = min(row0_blk + QT, n_qb) - 1;
  // Range r of this sequence: keys [kb, ke) (ke clipped to the block table), walked in
  // 64-key steps from s_first (kb rounded down to a 16-key tile) while below ke_blk (ke, or
  // the block's last causal key + 1).  All block-uniform.  Ranges that follow each other
  // without a gap (the shards of a ring) are walked as one.
  struct Range {
    int kb, ke, s_first, ke_blk;
  };
  __shared__ int32_t rtab[2][PF_RTAB];
  const int n_tab = a.n_ranges > 1 ? min(a.n_ranges, PF_RTAB) : 0;
  int n_ranges = a.n_ranges, ke_one = ke0;
  if (n_tab) {  // block-uniform
    bool gap = a.n_ranges > PF_RTAB;
    for (int r = threadIdx.x; r < n_tab; r += PF_THREADS) {
      const int64_t i = (int64_t)r * a.n_seqs + b;
      const int32_t kbr = a.kv_begin[i], ker = a.kv_end[i];
      rtab[0][r] = kbr;
      rtab[1][r] = ker;
      gap |= kbr < 0 || ker < kbr || (r > 0 && a.kv_end[i - a.n_seqs] != kbr);
    }
    if (!__syncthreads_or(gap)) {
      n_ranges = 1;
      ke_one = __builtin_amdgcn_readfirstlane(rtab[1][n_tab - 1]);
    }
  }
  auto range = [&](int r) -> Range {
    Range g;
    int32_t kbr, ker;
    if (r == 0) {
      kbr = kb0;
      ker = ke_one;
    } else if (r < n_tab) {
      kbr = __builtin_amdgcn_readfirstlane(rtab[0][r]);
      ker = __builtin_amdgcn_readfirstlane(rtab[1][r]);
    } else {
      const int64_t i = (int64_t)r * a.n_seqs + b;
      kbr = a.kv_begin[i];
      ker = a.kv_end[i];
    }
    g.kb = kbr > 0 ? kbr : 0;
    g.ke = ker;
    if (g.ke > kmax) {
      e |= ZX_KERR_POS_RANGE;
      g.ke = kmax;
    }
    g.ke_blk = a.causal ? (int)max((int64_t)-1, min((int64_t)g.ke, qp0 + last_row + 1)) : g.ke;
    g.s_first = (g.kb / 16) * 16;
    return g;
  };
  // the first range with a step at or after r (n_ranges if none)
  auto next_range = [&](int r, Range &g) -> int {
    for (; r < n_ranges; ++r) {
      g = range(r);
      if (g.s_first < g.ke_blk) return r;
    }
    return n_ranges;
  };
  Range g;
  int rc = next_range(0, g);
  __shared__ __attribute__((aligned(16))) uint8_t kst[3 * PW_KBYTES];
  __shared__ __attribute__((aligned(16))) uint8_t vtl[4 * PW_VBYTES];

  const float qs = sk * a.sm_log2e;
  const float vscale = sv;
  att_f32x16 o[2][4];  // [rg][ct]: channels 32 ct + 8 t + 4 hl ..+4 of row 32 rg + n
  float m[2], l[2];
#pragma unroll
  for (int rg = 0; rg < 2; ++rg) {
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[rg][ct][i] = 0.0f;
    m[rg] = -INFINITY;
    l[rg] = 0.0f;
  }
  const float p_shift = F16 ? PF_F16_SHIFT : 0.0f;
  const int kp2 = threadIdx.x >> 3, g8 = threadIdx.x & 7;
  const int kk0 = 2 * kp2;
  struct Codes {
    att_u32x4 k[2], v[2];
  };
  // Where the codes of 64 steps' tiles are (this wave's 16-key tile of each step): lane i
  // holds step base + i's byte offset in the pool and its bytes of valid rows, so that a
  // step costs three readlanes instead of a page lookup and its scalar arithmetic.
  uint32_t tab_lo = 0, tab_hi = 0;
  int tab_n = 0;
  auto fill_table = [&](int base) {
    const int64_t at = (int64_t)g.s_first + (int64_t)(base + lane) * PF_KEYS, tp = at + 16 * wave;
    const int n_live = at < g.ke_blk ? (int)max((int64_t)0, min((int64_t)16, g.ke - tp)) : 0;
    const uint32_t tc = n_live ? (uint32_t)tp : 0u;
    const uint32_t bi = pf_page_of(a, tc);
    const int64_t page = n_live ? bt[bi] : 0;
    const bool ok = page >= 0 && page < a.n_pages;
    e |= ok ? 0 : ZX_KERR_PAGE_RANGE;
    const uint64_t off =
        ok ? (uint64_t)(page * page_bytes + head_off + (int64_t)(tc - bi * (uint32_t)a.page_size) * D) : 0;
    tab_lo = (uint32_t)off;
    tab_hi = (uint32_t)(off >> 32);
    tab_n = ok ? n_live * D : 0;
  };
  const int ld_off = (kk0 & 15) * D + 16 * g8;
  // K and V codes of step i of the range into registers (past the block's last step: nothing
  // is read)
  auto issue_step = [&](int i, Codes &c) {
    const uint64_t off = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)tab_lo, i & 63) |
                         (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)tab_hi, i & 63) << 32;
    const int nrec = __builtin_amdgcn_readlane(tab_n, i & 63);
    const uint8_t *src = a.pool + off;
    const __amdgpu_buffer_rsrc_t rk =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(src), (short)0, nrec, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(src + v_off), (short)0, nrec, 0x00020000);
    c.k[0] = __builtin_amdgcn_raw_buffer_load_b128(rk, ld_off, 0, 0);
    c.k[1] = __builtin_amdgcn_raw_buffer_load_b128(rk, ld_off + D, 0, 0);
    c.v[0] = __builtin_amdgcn_raw_buffer_load_b128(rv, ld_off, 0, 0);
    c.v[1] = __builtin_amdgcn_raw_buffer_load_b128(rv, ld_off + D, 0, 0);
  };
  const int kst_off = kk0 * PF_KROW + 32 * g8;
  const int vst_off = pw_vslot_byte(16 * g8, kk0);
  auto store_k = [&](int kbuf, int j, const Codes &c) {
    uint32_t kb8[8];
    decode16_bf16(make_uint4(c.k[j].x, c.k[j].y, c.k[j].z, c.k[j].w), kb8);
    uint4 *kd = reinterpret_cast<uint4 *>(&kst[kbuf + kst_off + j * PF_KROW]);
    kd[0] = make_uint4(kb8[0], kb8[1], kb8[2], kb8[3]);
    kd[1] = make_uint4(kb8[4], kb8[5], kb8[6], kb8[7]);
  };
  // V^T of channels 16 g8 + 4 q ..+4 (q < 4): two code words of each key
  auto store_v = [&](int vbuf, int q, const Codes &c) {
    uint32_t v0[2], v1[2];
    const int w0 = (int)c.v[0][q], w1 = (int)c.v[1][q];
    if constexpr (F16) {
      v0[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 1.0f, false));
      v0[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 1.0f, true));
      v1[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 1.0f, false));
      v1[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 1.0f, true));
    } else {
      v0[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, false));
      v0[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, true));
      v1[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, false));
      v1[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, true));
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      uint8_t *row = &vtl[vbuf + vst_off + (4 * q + 2 * p) * 8 * PF_VROW];
      *reinterpret_cast<uint32_t *>(row) = __builtin_amdgcn_perm(v1[p], v0[p], 0x05040100u);
      *reinterpret_cast<uint32_t *>(row + 8 * PF_VROW) = __builtin_amdgcn_perm(v1[p], v0[p], 0x07060302u);
    }
  };

  att_u32x4 qa[2][8];
#pragma unroll
  for (int rg = 0; rg < 2; ++rg) {
    const int r = min(wrow0 + 32 * rg + n, n_qb - 1);  // rows past the last repeat it, and are not stored
#pragma unroll
    for (int c = 0; c < 8; ++c)
      qa[rg][c] =
          *reinterpret_cast<const att_u32x4 *>(a.q + ((q_lo + r) * a.n_q_heads + hq) * D + c * 16 + hl * 8);
  }
  Codes ca, cb;
  if (rc < n_ranges) {
    fill_table(0);
    issue_step(0, ca);
    issue_step(1, cb);
  }
  bool all_ok;
  {
    bool bad = false;
    for (int r = 0; r < n_ranges; ++r) {
      const Range w = range(r);
      if (w.s_first >= w.ke) continue;
      const int p_lo = (int)pf_page_of(a, (uint32_t)w.s_first), p_hi = (int)pf_page_of(a, (uint32_t)(w.ke - 1));
      for (int pi = p_lo + (int)threadIdx.x; pi <= p_hi; pi += PF_THREADS) {
        const int64_t pg = bt[pi];
        bad |= pg < 0 || pg >= a.n_pages;
      }
    }
    all_ok = !__syncthreads_or(bad);
  }
  auto tile_ok = [&](int tp, int ke) -> bool {
    if (tp >= ke) return false;
    if (all_ok) return true;
    const int64_t page = bt[pf_page_of(a, (uint32_t)tp)];
    return page >= 0 && page < a.n_pages;
  };
  att_u32x4 ph[2][4];  // [rg][kc] P^T as 16-bit pairs
  const int k_lane = n * PF_KROW + hl * 16;
  const int v_lane = n * PF_VROW + hl * 16;
  auto ld_k = [&](int kbuf, int t) -> att_u32x4 {  // t = 8 KT + c
    return *reinterpret_cast<const att_u32x4 *>(&kst[kbuf + k_lane + (t >> 3) * 32 * PF_KROW + (t & 7) * 32]);
  };
  auto ld_v = [&](int vbuf, int t) -> att_u32x4 {  // t = 4 kc + ct
    return *reinterpret_cast<const att_u32x4 *>(&vtl[vbuf + v_lane + (t & 3) * 32 * PF_VROW + (t >> 2) * 32]);
  };
  constexpr int FD = 3;  // operand reads ahead
  // the last key position a row may see, and the last step start at which every row of this
  // wave sees every key (of a range)
  auto row_lim = [&](int r) {
    return a.causal ? (int)min(max(qp0 + min(r, n_qb - 1), (int64_t)-1), (int64_t)INT32_MAX) : INT32_MAX;
  };
  const int lim[2] = {row_lim(wrow0 + n), row_lim(wrow0 + 32 + n)};
  const int s_full = all_ok ? row_lim(wrow0) - (PF_KEYS - 1) : -1;
  // P.V of a step that starts past the last key of the first 32 rows leaves them out: their
  // weights are 0, and a NaN V there would reach rows up to 126 positions before its key
  // instead of 94 (the 32-row kernel does not walk such steps for these rows)
  const int lim_first = row_lim(wrow0 + 31);
  bool pv_both = true;  // the step whose P.V is next has keys for the first 32 rows
  att_u32x4 kf[FD + 1], vf[FD + 1];
  auto pv_tile = [&](int t, int rg0 = 0) {
    const att_u32x4 av = vf[t % (FD + 1)];
    const int kc = t >> 2, ct = t & 3;
#pragma unroll
    for (int rg = rg0; rg < 2; ++rg) {
      if constexpr (F16) o[rg][ct] = pw_mfma_f16(av, ph[rg][kc], o[rg][ct]);
      else o[rg][ct] = pw_mfma_bf16(av, ph[rg][kc], o[rg][ct]);
    }
  };
  auto pv_rest = [&](int vrd) {  // tiles whose first FD operands are read
    auto tiles = [&](int rg0) {
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        if (t + FD < 16) vf[(t + FD) % (FD + 1)] = ld_v(vrd, t + FD);
        pv_tile(t, rg0);
      }
    };
    if (pv_both) tiles(0);
    else tiles(1);
  };
  using Scores = att_f32x16[2][2];  // [rg][KT]
  // word w of the weights of key chunk kc as 16-bit pairs, and the chunk's sum
  auto pack_p = [&](const Scores &s, float (&ls)[2][2], int kc, int w) {
#pragma unroll
    for (int rg = 0; rg < 2; ++rg) {
      const int i = 8 * (kc & 1) + 2 * w;
      const float x = s[rg][kc >> 1][i], y = s[rg][kc >> 1][i + 1];
      // (a scalar first: with this compiler __builtin_bit_cast of a vector's element reads
      // element 0)
      const uint32_t pw = F16 ? pack_f16(x, y) : pack_bf16(x, y);
      ph[rg][kc][w] = pw;
      if constexpr (F16)
        ls[rg][w & 1] = __builtin_amdgcn_fdot2(__builtin_bit_cast(pw_f16x2, pw), pw_f16x2{(_Float16)1, (_Float16)1},
                                               ls[rg][w & 1], false);
      else
        ls[rg][w & 1] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(att_bf2, pw),
                                                        __builtin_bit_cast(att_bf2, 0x3F803F80u), ls[rg][w & 1], false);
    }
  };
  // keeps a chunk's weights where they are made: beside the products, not sunk past them
  auto pin_p = [&](float (&ls)[2][2], int kc) {
    asm volatile("" : "+v"(ph[0][kc]), "+v"(ph[1][kc]), "+v"(ls[0][0]), "+v"(ls[0][1]), "+v"(ls[1][0]), "+v"(ls[1][1]));
  };
  auto qk_tile = [&](Scores &s, int t) {  // t = 8 KT + c
    const int KT = t >> 3, c = t & 7;
#pragma unroll
    for (int rg = 0; rg < 2; ++rg) {
      if (c == 0) {
        att_f32x16 z;
#pragma unroll
        for (int i = 0; i < 16; ++i) z[i] = 0.0f;
        s[rg][KT] = pw_mfma_bf16(kf[t % (FD + 1)], qa[rg][c], z);
      } else {
        s[rg][KT] = pw_mfma_bf16(kf[t % (FD + 1)], qa[rg][c], s[rg][KT]);
      }
    }
  };
  // exponents, then weights, of elements i0 ..+n_e of key tile KT (a weight right after its
  // own exponent would wait for it)
  auto weights = [&](Scores &s, int KT, int i0, int n_e, float q, const float (&cst)[2]) {
    float x[2][8];
#pragma unroll
    for (int rg = 0; rg < 2; ++rg)
#pragma unroll
      for (int u = 0; u < n_e; ++u) x[rg][u] = __builtin_fmaf(s[rg][KT][i0 + u], q, cst[rg]);
#pragma unroll
    for (int u = 0; u < n_e; ++u) asm volatile("" : "+v"(x[0][u]), "+v"(x[1][u]));
#pragma unroll
    for (int rg = 0; rg < 2; ++rg)
#pragma unroll
      for (int u = 0; u < n_e; ++u) s[rg][KT][i0 + u] = __builtin_amdgcn_exp2f(x[rg][u]);
  };
  constexpr float L_MOST = F16 ? 32768.0f : 256.0f;  // 2^(p_shift + PF_LAZY)
  float cst[2] = {-INFINITY, -INFINITY};
  bool m_ok = false;  // every row of the wave has a running maximum

  while (rc < n_ranges) {  // a range: its steps j = 0 .. n_steps - 1
    store_k(0, 0, ca);
    store_k(0, 1, ca);
#pragma unroll
    for (int q = 0; q < 4; ++q) store_v(0, q, ca);
    // the V^T buffer that the first step's (empty) P.V reads
    for (int i = threadIdx.x; i < PW_VBYTES / 16; i += PF_THREADS)
      *reinterpret_cast<uint4 *>(&vtl[3 * PW_VBYTES + 16 * i]) = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
    for (int rg = 0; rg < 2; ++rg)
#pragma unroll
      for (int kc = 0; kc < 4; ++kc) ph[rg][kc] = att_u32x4{0u, 0u, 0u, 0u};
    pv_both = true;
    __syncthreads();
    int kbuf = 0, vrd = 3 * PW_VBYTES, vnext = PW_VBYTES;
#pragma unroll
    for (int t = 0; t < FD; ++t) kf[t] = ld_k(0, t);
    const int s_hi = min(g.ke - PF_KEYS, s_full);
    const int n_steps = (g.ke_blk - g.s_first + PF_KEYS - 1) / PF_KEYS;
    for (int j = 0; j < n_steps;) {
      // the steps that every row of the wave sees whole, under the running maxima it has
      int kb_n = kbuf == 2 * PW_KBYTES ? 0 : kbuf + PW_KBYTES;
      float ls[2][2];
      bool grown = false;
      auto next_step = [&]() {
#pragma unroll
        for (int rg = 0; rg < 2; ++rg) l[rg] += ls[rg][0] + ls[rg][1];
        kbuf = kb_n;
        kb_n = kbuf == 2 * PW_KBYTES ? 0 : kbuf + PW_KBYTES;
        vrd = vrd == 3 * PW_VBYTES ? 0 : vrd + PW_VBYTES;
        vnext = vnext == 3 * PW_VBYTES ? 0 : vnext + PW_VBYTES;
        ++j;
      };
      while (m_ok && j < n_steps) {
        const int s0 = g.s_first + j * PF_KEYS;
        if (s0 < g.kb || s0 > s_hi) break;
        if (((j + 2) & 63) == 0) fill_table(j + 2);
        ls[0][0] = ls[0][1] = ls[1][0] = ls[1][1] = 0.0f;
        Scores s;
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          if (t + FD < 16) kf[(t + FD) % (FD + 1)] = ld_k(kbuf, t + FD);
          else vf[t + FD - 16] = ld_v(vrd, t + FD - 16);
          qk_tile(s, t);
          if (t == 0) store_k(kb_n, 0, cb);
          if (t == 2) store_k(kb_n, 1, cb);
          if (t >= 3 && t < 7) store_v(vnext, t - 3, cb);
          if (t >= 9 && t < 14) weights(s, 0, 3 * (t - 9), 3, qs, cst);
          if (t == 14) weights(s, 0, 15, 1, qs, cst);
          __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          if (t + FD < 16) vf[(t + FD) % (FD + 1)] = ld_v(vrd, t + FD);
          else kf[t + FD - 16] = ld_k(kb_n, t + FD - 16);
          pv_tile(t);
          if (t == 0) issue_step(j + 2, cb);
          if (t < 8) weights(s, 1, 2 * t, 2, qs, cst);
          if (t >= 4) {  // P of kc is free after tile 4 kc + 3
            pack_p(s, ls, (t >> 2) - 1, t & 3);
            if ((t & 3) == 3) pin_p(ls, (t >> 2) - 1);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int w = 0; w < 4; ++w) pack_p(s, ls, 3, w);
        pin_p(ls, 3);
        const bool big = fmaxf(fmaxf(ls[0][0], ls[0][1]), fmaxf(ls[1][0], ls[1][1])) > L_MOST;
        if (__builtin_amdgcn_ballot_w64(big)) {
          grown = true;
          break;
        }
        next_step();
      }
      if (j >= n_steps) break;
      const int s0 = g.s_first + j * PF_KEYS;
      if (!grown) {
        if (((j + 2) & 63) == 0) fill_table(j + 2);
        store_k(kb_n, 0, cb);
        store_k(kb_n, 1, cb);
#pragma unroll
        for (int q = 0; q < 4; ++q) store_v(vnext, q, cb);
#pragma unroll
        for (int t = 0; t < FD; ++t) vf[t] = ld_v(vrd, t);
        __syncthreads();
        issue_step(j + 2, cb);
        pv_rest(vrd);
      }
      {
        // (a negative scale: the maximum of s qs is not qs times that of s.  The steps above
        // take no maximum and any sign: 4 x 8,192 causal 4,243 us where they did not, 2,210 so)
        const bool full = s0 >= g.kb && s0 <= s_hi && qs >= 0.0f;
        pv_both = s0 <= lim_first;
        // the step with its running maxima looked at and the masks applied: the first step, the
        // steps that cross a boundary, and one whose weights outgrew the maxima (its S^T made
        // again; this step's K is still in LDS)
        Scores s;
#pragma unroll
        for (int t = 0; t < FD; ++t) kf[t] = ld_k(kbuf, t);
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          if (t + FD < 16) kf[(t + FD) % (FD + 1)] = ld_k(kbuf, t + FD);
          qk_tile(s, t);
        }
#pragma unroll
        for (int t = 0; t < FD; ++t) kf[t] = ld_k(kb_n, t);
        float qe = qs;
        if (!full) {  // scores times qs, -inf where the (row, key) does not count
          uint32_t tk = 0;
#pragma unroll
          for (int T = 0; T < 4; ++T) tk |= tile_ok(s0 + 16 * T, g.ke) ? 1u << T : 0u;
#pragma unroll
          for (int i = 0; i < 32; ++i) {
            const int kp = s0 + 8 * (i >> 2) + 4 * hl + (i & 3);
            const bool in = ((tk >> (i >> 3)) & 1u) != 0 && kp >= g.kb && kp < g.ke;
#pragma unroll
            for (int rg = 0; rg < 2; ++rg)
              s[rg][i >> 4][i & 15] = in && kp <= lim[rg] ? s[rg][i >> 4][i & 15] * qs : -INFINITY;
          }
          qe = 1.0f;
        }
        bool grow_any = false, ok = true;
        float alpha[2];
#pragma unroll
        for (int rg = 0; rg < 2; ++rg) {
          float mx = -INFINITY, x, y;
#pragma unroll
          for (int i = 0; i < 32; i += 2) mx = fmaxf(fmaxf(mx, s[rg][i >> 4][i & 15]), s[rg][i >> 4][(i & 15) + 1]);
          xrow_pair32(mx * qe, x, y);
          const float w = fmaxf(x, y);
          // (after a repeat by as little as it takes: left where it is, a maximum 4 to 8 below
          // the scores would have every further step repeated)
          const bool grow = w > m[rg] + (grown ? 0.0f : PF_LAZY);
          const float mn = grow ? w : m[rg];
          const float ms = mn == -INFINITY ? 0.0f : mn;  // a row with no key yet keeps p = 0
          alpha[rg] = grow ? __builtin_amdgcn_exp2f(m[rg] - ms) : 1.0f;
          grow_any |= grow;
          ok &= mn != -INFINITY;
          m[rg] = mn;
          l[rg] *= alpha[rg];
          cst[rg] = p_shift - ms;
          ls[rg][0] = ls[rg][1] = 0.0f;
        }
        m_ok = __builtin_amdgcn_ballot_w64(!ok) == 0;
#pragma unroll
        for (int KT = 0; KT < 2; ++KT)
#pragma unroll
          for (int i = 0; i < 16; i += 8) weights(s, KT, i, 8, qe, cst);
#pragma unroll
        for (int kc = 0; kc < 4; ++kc)
#pragma unroll
          for (int w = 0; w < 4; ++w) pack_p(s, ls, kc, w);
          // rescale O only when some row's maximum was raised
        if (__builtin_amdgcn_ballot_w64(grow_any)) {
#pragma unroll
          for (int rg = 0; rg < 2; ++rg)
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) o[rg][ct] *= alpha[rg];
        }
      }
      next_step();
    }
    // P.V of the last step
#pragma unroll
    for (int t = 0; t < FD; ++t) vf[t] = ld_v(vrd, t);
    pv_rest(vrd);
    rc = next_range(rc + 1, g);
    if (rc < n_ranges) {
      fill_table(0);
      issue_step(0, ca);
      issue_step(1, cb);
      __syncthreads();
    }
  }

  // rows: normalise; store.  O^T row 32 ct + 8 t + 4 hl + i is channel
  // 16 (4 hl + i) + 4 ct + t: 16 channels in a row per i.
#pragma unroll
  for (int rg = 0; rg < 2; ++rg) {
    const int r = wrow0 + 32 * rg + n;
    float lx, ly;
    xrow_pair32(l[rg], lx, ly);
    const float lt = lx + ly;
    if (r >= n_qb) continue;
    const float inv = lt > 0.0f ? vscale / lt : 0.0f;  // V's dequant scale applied once, here
    uint4 *out = reinterpret_cast<uint4 *>(a.out + ((q_lo + r) * a.n_q_heads + hq) * D + 64 * hl);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t w[8];
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        w[2 * ct] = pack_bf16(o[rg][ct][i] * inv, o[rg][ct][4 + i] * inv);
        w[2 * ct + 1] = pack_bf16(o[rg][ct][8 + i] * inv, o[rg][ct][12 + i] * inv);
      }
      out[2 * i] = make_uint4(w[0], w[1], w[2], w[3]);
      out[2 * i + 1] = make_uint4(w[4], w[5], w[6], w[7]);
    }
  }
  if (e && a.err) atomicOr(a.err, e);
}

// Rows whose keys several blocks shared: out = sum_s 2^(lse_s - M) o_s / sum_s 2^(lse_s - M)
// over the parts (normalised fp32 rows and their log2 sums), as bf16.  A block takes a query
// tile of a head group, as the parts' blocks did (rows no tile holds are left alone), half a
// wave a row, 4 channels per lane; the lanes of a half hold the parts' sums.  Parts of weight
// 0 are added too (0 x NaN: a NaN key or value makes its rows NaN whichever part held it).
constexpr int PC_MAX = 32;  // parts
__global__ void __launch_bounds__(256) prefill_combine_kernel(PrefillArgs a, int32_t G, int32_t qt_rows) {
  const int n_hg = a.n_q_heads / G;
  const int64_t per_rank = (int64_t)n_hg * a.n_seqs;
  const int64_t qt_rev = (int64_t)blockIdx.x / per_rank;
  const int rem = (int)((int64_t)blockIdx.x - qt_rev * per_rank);
  const int hg = rem % n_hg, b = rem / n_hg;
  const int32_t cq0 = a.cu_q[b], n_qb = a.cu_q[b + 1] - cq0;
  const int64_t row0 = ((int64_t)a.n_qt - 1 - qt_rev) * qt_rows;
  if (row0 >= n_qb) return;
  const int n_rows = (int)min((int64_t)qt_rows, n_qb - row0) * G;  // (row, head) pairs
  const int lane = threadIdx.x & 63, s_l = lane & 31;
  const int S = a.parts[blockIdx.x];
  if (S == 1) return;  // its block has written the rows
  for (int i = 8 * blockIdx.y + (threadIdx.x >> 5); i < n_rows; i += 8 * gridDim.y) {  // uniform in half a wave, where the shuffles stay
    const int64_t row = (cq0 + row0 + i / G) * a.n_q_heads + hg * G + i % G;
    const float ls = s_l < S ? a.lse2[s_l * a.part_stride + row] : -INFINITY;
    float M = ls;
#pragma unroll
    for (int off = 1; off < 32; off <<= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
    const float w = M == -INFINITY || s_l >= S ? 0.0f : __builtin_amdgcn_exp2f(ls - M);
    float L = w;
#pragma unroll
    for (int off = 1; off < 32; off <<= 1) L += __shfl_xor(L, off, 64);
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float *src = a.o_acc + row * 128 + 4 * s_l;
    for (int s = 0; s < S; s += 4) {
      float4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        v[u] = *reinterpret_cast<const float4 *>(src + min(s + u, S - 1) * a.part_stride * 128);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float ws = __shfl(w, ((lane & 32) + s + u) & 63, 64);
        if (s + u < S) {
          acc.x += ws * v[u].x;
          acc.y += ws * v[u].y;
          acc.z += ws * v[u].z;
          acc.w += ws * v[u].w;
        }
      }
    }
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    *reinterpret_cast<uint2 *>(a.out + row * 128 + 4 * s_l) =
        make_uint2(pack_bf16(acc.x * inv, acc.y * inv), pack_bf16(acc.z * inv, acc.w * inv));
  }
}

}  // namespace zx

using namespace zx;

namespace {
// How a call is cut into blocks.
struct PrefillPlan {
  int G, pm, n_split;
  bool wide;
  int QT;           // rows per block
  int32_t n_qt;     // tiles per sequence
  int64_t max_rows; // rows per sequence that are computed (a wide block's 64 rows may hold fewer)
  int64_t n_tiles;  // blocks that share no rows
};
PrefillPlan prefill_plan(int64_t n_q, int32_t n_q_heads, int32_t n_kv_heads, int32_t page_size, int32_t max_blocks,
                         int32_t n_seqs, int32_t max_q_per_seq, int32_t causal, int32_t flags) {
  PrefillPlan p;
  // a loose bound (a model's longest context) launches no tiles that no sequence can have: 64
  // rows on 8,128 keys under a bound of 131,072 390 us, 36 so
  max_q_per_seq = (int32_t)std::min<int64_t>(max_q_per_seq, n_q);
  const int grp = n_q_heads / n_kv_heads;
  p.G = grp % 4 == 0 ? 4 : (grp % 2 == 0 ? 2 : 1);
  p.pm = (flags & ZX_PREFILL_EXACT_P) ? PF_P_EXACT : ((flags & ZX_PREFILL_FAST_P) ? PF_P_BF16 : PF_P_F16);
  const int64_t cap = (int64_t)max_blocks * page_size;  // positions a sequence can have
  const bool rows_only = !(flags & ZX_PREFILL_MERGE);
  // blocks of `qt` rows that hold any (sequences differ in length)
  auto blocks = [&](int64_t qt) {
    return std::min(ceil_div(max_q_per_seq, qt) * n_seqs, ceil_div(n_q, qt) + n_seqs) * (n_q_heads / p.G);
  };
  // 64 rows per wave where nothing is merged, four query heads share a KV head, there is a
  // block per CU and contexts can be long.  Its blocks start and end more slowly, one to a CU,
  // so sequences need rows enough: 900 on average, or 320 where four rounds of blocks hold the
  // call.  (The host does not know the keys; new sequences have the fewest.  Tables of 8,192
  // positions, 32 rows against 64: 256 x 100 rows 213 us, 239; 64 x 256 150, 184; 25 x 630 188,
  // 200; 16 x 1,000 245, 240; 23 x 2,048 1,118, 1,014; in four rounds 16 x 250 52, 47; 21 x 380
  // 88, 88; 10 x 768 115, 105.  With 32 rows and fewer half of a tile is empty: 64 x 32 on 4k-8k
  // 300, 487.  Few keys without a mask are not kept out: 2 x 4,096 rows on 300 86, 97.)  One or
  // two heads per KV head gained nothing (2 x 4,096: 150 against 140, 175 against 175), and the
  // exact mode's second set of weights does not fit its registers.
  const int64_t wide_blocks = blocks(PW_ROWS), rows = n_q / n_seqs;
  p.wide = p.G == 4 && rows_only && p.pm != PF_P_EXACT && cap >= 4096 && wide_blocks >= num_cus() &&
           (rows >= 900 || (rows >= 320 && wide_blocks <= 4LL * num_cus()));
  // Few blocks: several share a tile's keys (2 x 300-700 rows on 4k-12k cached 467 -> 229 us,
  // 256 rows on 16k 436 -> 103, 4 x 4-8 rows on 4k-8k 397 -> 50).  One round of resident blocks
  // where that gives at least four parts a tile, else two, which even out sequences of
  // different lengths; none where the tiles fill the round as they are (64 x 32 rows on 6,000
  // cached 254 against 279 us in two parts, 32 x 64 on 4k-8k 299 against 325; 16 x 128 on
  // 500-16k the other way, 481 against 366); at least 8 steps each by the table's width.  (The
  // other lines were drawn while one block combined a tile: 256 rows on 16k 169 us with two
  // rounds against 134, 2 x 300-700 290 with one against 254, 1,024 rows of a new sequence 56 in
  // parts of 4 to 8 steps against 45.)
  p.n_split = 1;
  const int64_t nb = blocks(32 * 4 / p.G), slots = 2LL * num_cus();
  if (rows_only && !p.wide && nb > 0) {
    const int64_t steps = (cap - (causal ? std::min<int64_t>(max_q_per_seq, cap) / 2 : 0)) / PF_KEYS;
    const int64_t parts = slots / nb >= 4 ? slots / nb : (nb * 8 > slots * 7 ? 1 : 2 * slots / nb);
    p.n_split = (int)std::max<int64_t>(1, std::min({parts, steps / 8, (int64_t)PC_MAX}));
  }
  p.QT = p.wide ? PW_ROWS : 32 * 4 / p.G;
  p.n_qt = (int32_t)ceil_div(max_q_per_seq, p.QT);
  p.max_rows = ceil_div(max_q_per_seq, 128 / p.G) * (128 / p.G);
  p.n_tiles = (int64_t)p.n_qt * (n_q_heads / p.G) * n_seqs;
  return p;
}
size_t prefill_part_bytes(const PrefillPlan &p, int64_t n_q, int32_t n_q_heads) {
  return p.n_split > 1 ? (size_t)p.n_split * n_q * n_q_heads * (128 + 1) * sizeof(float) + p.n_tiles * sizeof(int32_t)
                       : 0;
}

int prefill_impl(const uint16_t *q, int64_t n_q, const int32_t *cu_q, const int32_t *q_pos0, int32_t n_q_heads,
                 const uint8_t *pool, int64_t n_pages, int32_t n_kv_heads, int32_t head_dim, int32_t page_size,
                 const float *scales, const int32_t *block_tables, int32_t max_blocks, const int32_t *kv_begin,
                 const int32_t *kv_end, int32_t n_ranges, int32_t n_seqs, int32_t max_q_per_seq, int32_t causal,
                 float sm_scale, int32_t flags, float *o_acc, float *lse2, uint16_t *out, int32_t *err,
                 void *workspace, size_t workspace_bytes, zx_stream_t stream) {
  ZX_REQUIRE(q && cu_q && q_pos0 && pool && scales && block_tables && kv_begin && kv_end,
             "paged_attention_prefill: null pointer");
  ZX_REQUIRE(n_ranges >= 1, "paged_attention: n_ranges must be positive");
  ZX_REQUIRE(n_q >= 0 && n_q_heads > 0 && n_kv_heads > 0 && n_pages > 0 && page_size > 0 && max_blocks > 0 &&
                 n_seqs > 0 && max_q_per_seq >= 0,
             "paged_attention_prefill: sizes must be positive");
  ZX_REQUIRE(n_q_heads % n_kv_heads == 0, "paged_attention_prefill: n_q_heads must be a multiple of n_kv_heads");
  ZX_REQUIRE((flags & ~(ZX_PREFILL_MERGE | ZX_PREFILL_INIT | ZX_PREFILL_BF16 | ZX_PREFILL_FAST_P | ZX_PREFILL_EXACT_P |
                        ZX_PREFILL_LAST | ZX_PREFILL_FINAL)) == 0,
             "paged_attention_prefill: unknown flags");
  ZX_REQUIRE(!(flags & ZX_PREFILL_FINAL) ||
                 ((flags & ZX_PREFILL_MERGE) && (flags & ZX_PREFILL_BF16) && causal && n_ranges == 1),
             "paged_attention_prefill: ZX_PREFILL_FINAL needs ZX_PREFILL_MERGE, ZX_PREFILL_BF16, causal and one key "
             "range (zx_paged_attention_prefill)");
  ZX_REQUIRE(!(flags & ZX_PREFILL_LAST) || ((flags & ZX_PREFILL_MERGE) && (flags & ZX_PREFILL_BF16)),
             "paged_attention_prefill: ZX_PREFILL_LAST needs ZX_PREFILL_MERGE and ZX_PREFILL_BF16");
  ZX_REQUIRE(!((flags & ZX_PREFILL_FAST_P) && (flags & ZX_PREFILL_EXACT_P)),
             "paged_attention_prefill: ZX_PREFILL_FAST_P and ZX_PREFILL_EXACT_P together");
  ZX_REQUIRE(!(flags & ZX_PREFILL_MERGE) || (o_acc && lse2), "paged_attention_prefill: merging needs o_acc and lse2");
  ZX_REQUIRE(!(flags & ZX_PREFILL_BF16) || out, "paged_attention_prefill: bf16 output requested without out");
  ZX_REQUIRE(flags & (ZX_PREFILL_MERGE | ZX_PREFILL_BF16), "paged_attention_prefill: nothing to write");
  ZX_REQUIRE(aligned16(q) && aligned16(pool) && (!(flags & ZX_PREFILL_MERGE) || aligned16(o_acc)) &&
                 (!(flags & ZX_PREFILL_BF16) || aligned16(out)),
             "paged_attention_prefill: q, pool, o_acc and out must be 16-byte aligned");
  if (head_dim != 128 || page_size % 16)
    return fail(ZX_ERR_UNSUPPORTED, "paged_attention_prefill: needs head_dim 128 and pages of a multiple of 16 tokens "
                                    "(got %d, %d)", head_dim, page_size);
  if (n_q == 0 || max_q_per_seq == 0) return ZX_OK;
  if ((int64_t)max_blocks * page_size >= (1LL << 31))
    return fail(ZX_ERR_UNSUPPORTED, "paged_attention_prefill: sequences too long");
  PrefillPlan p = prefill_plan(n_q, n_q_heads, n_kv_heads, page_size, max_blocks, n_seqs, max_q_per_seq, causal, flags);
  if (!workspace || workspace_bytes < prefill_part_bytes(p, n_q, n_q_heads)) p.n_split = 1;  // no room for parts
  const int G = p.G, pm = p.pm;
  PrefillArgs a;
  a.q = q;
  a.cu_q = cu_q;
  a.q_pos0 = q_pos0;
  a.pool = pool;
  a.scales = scales;
  a.bt = block_tables;
  a.kv_begin = kv_begin;
  a.kv_end = kv_end;
  a.n_ranges = n_ranges;
  a.n_seqs = n_seqs;
  a.o_acc = o_acc;
  a.lse2 = lse2;
  a.out = out;
  a.err = err;
  a.n_pages = n_pages;
  a.n_q_heads = n_q_heads;
  a.n_kv_heads = n_kv_heads;
  a.page_size = page_size;
  a.max_blocks = max_blocks;
  a.mode = ((flags & ZX_PREFILL_MERGE) ? PF_MERGE : 0) | ((flags & ZX_PREFILL_INIT) ? PF_INIT : 0) |
           ((flags & ZX_PREFILL_BF16) ? PF_WRITE_BF16 : 0) | ((flags & ZX_PREFILL_LAST) ? PF_LAST : 0) |
           ((flags & ZX_PREFILL_FINAL) ? PF_FINAL : 0);
  a.causal = causal ? 1 : 0;
  a.sm_log2e = sm_scale * ATT_LOG2E;
  {  // t / page_size = (t * magic) >> (31 + shift) for t < 2^31
    int shift = 0;
    while ((1LL << shift) < page_size) ++shift;
    a.p_shift = shift;
    a.p_magic = (uint32_t)(((1ULL << (31 + shift)) + page_size - 1) / page_size);
  }
  a.n_qt = p.n_qt;
  a.max_rows = p.max_rows;
  const int64_t n_blocks = p.n_tiles * p.n_split;
  ZX_REQUIRE(n_blocks < (1LL << 31), "paged_attention_prefill: too many query tiles or sequences");
  const dim3 grid((unsigned)n_blocks);
  hipStream_t st = as_stream(stream);
  if (p.wide) {
    if (pm == PF_P_F16) paged_prefill_wide_kernel<PF_P_F16><<<grid, PF_THREADS, 0, st>>>(a);
    else paged_prefill_wide_kernel<PF_P_BF16><<<grid, PF_THREADS, 0, st>>>(a);
    return check_launch("paged_prefill_wide");
  }
  a.n_split = p.n_split;
  a.part_stride = n_q * n_q_heads;
  if (p.n_split > 1) {
    a.o_acc = static_cast<float *>(workspace);
    a.lse2 = a.o_acc + (int64_t)p.n_split * a.part_stride * 128;
    a.parts = reinterpret_cast<int32_t *>(a.lse2 + p.n_split * a.part_stride);
  }
  switch (G * 4 + pm) {
#define ZX_PF_CASE(g, m)                                                                     \
  case g * 4 + m:                                                                            \
    if (p.n_split > 1) paged_prefill_mfma_kernel<g, m, true><<<grid, PF_THREADS, 0, st>>>(a); \
    else paged_prefill_mfma_kernel<g, m, false><<<grid, PF_THREADS, 0, st>>>(a);              \
    break;
#define ZX_PF_CASES(g) ZX_PF_CASE(g, PF_P_F16) ZX_PF_CASE(g, PF_P_BF16) ZX_PF_CASE(g, PF_P_EXACT)
    ZX_PF_CASES(4)
    ZX_PF_CASES(2)
    ZX_PF_CASES(1)
#undef ZX_PF_CASES
#undef ZX_PF_CASE
    default: return fail(ZX_ERR_INVALID, "paged_attention_prefill: internal dispatch");
  }
  int rc = check_launch("paged_prefill_mfma");
  if (rc || p.n_split == 1) return rc;
  // a tile's 128 (row, head) pairs over up to 16 blocks (one block a tile: 64 rows on 8,128
  // keys 81 us against 33, 2 x 300 on 4,000 113 against 90)
  const unsigned gy = (unsigned)std::min<int64_t>(16, std::max<int64_t>(1, 8LL * num_cus() / p.n_tiles));
  prefill_combine_kernel<<<dim3((unsigned)p.n_tiles, gy), 256, 0, st>>>(a, G, p.QT);
  return check_launch("prefill_combine");
}
}  // namespace

extern "C" size_t zx_paged_attention_ring_workspace_bytes(int64_t n_q, int32_t n_q_heads, int32_t n_kv_heads,
                                                          int32_t page_size, int32_t max_blocks, int32_t n_seqs,
                                                          int32_t max_q_per_seq, int32_t causal, int32_t flags) {
  if (n_q <= 0 || n_q_heads <= 0 || n_kv_heads <= 0 || n_q_heads % n_kv_heads || page_size <= 0 || max_blocks <= 0 ||
      n_seqs <= 0 || max_q_per_seq <= 0)
    return 0;
  return prefill_part_bytes(
      prefill_plan(n_q, n_q_heads, n_kv_heads, page_size, max_blocks, n_seqs, max_q_per_seq, causal, flags), n_q,
      n_q_heads);
}

extern "C" int zx_paged_attention_ring_ws(const uint16_t *q, int64_t n_q, const int32_t *cu_q, const int32_t *q_pos0,
                                          int32_t n_q_heads, const uint8_t *pool, int64_t n_pages, int32_t n_kv_heads,
                                          int32_t head_dim, int32_t page_size, const float *scales,
                                          const int32_t *block_tables, int32_t max_blocks, const int32_t *kv_begin,
                                          const int32_t *kv_end, int32_t n_ranges, int32_t n_seqs,
                                          int32_t max_q_per_seq, int32_t causal, float sm_scale, int32_t flags,
                                          float *o_acc, float *lse2, uint16_t *out, int32_t *err, void *workspace,
                                          size_t workspace_bytes, zx_stream_t stream) {
  clear_error();
  ZX_REQUIRE(!workspace || aligned16(workspace), "paged_attention_ring_ws: workspace must be 16-byte aligned");
  return prefill_impl(q, n_q, cu_q, q_pos0, n_q_heads, pool, n_pages, n_kv_heads, head_dim, page_size, scales,
                      block_tables, max_blocks, kv_begin, kv_end, n_ranges, n_seqs, max_q_per_seq, causal, sm_scale,
                      flags, o_acc, lse2, out, err, workspace, workspace_bytes, stream);
}

extern "C" int zx_paged_attention_prefill(const uint16_t *q, int64_t n_q, const int32_t *cu_q, const int32_t *q_pos0,
                                          int32_t n_q_heads, const uint8_t *pool, int64_t n_pages, int32_t n_kv_heads,
                                          int32_t head_dim, int32_t page_size, const float *scales,
                                          const int32_t *block_tables, int32_t max_blocks, const int32_t *kv_begin,
                                          const int32_t *kv_end, int32_t n_seqs, int32_t max_q_per_seq,
                                          int32_t causal, float sm_scale, int32_t flags, float *o_acc, float *lse2,
                                          uint16_t *out, int32_t *err, zx_stream_t stream) {
  clear_error();
  return prefill_impl(q, n_q, cu_q, q_pos0, n_q_heads, pool, n_pages, n_kv_heads, head_dim, page_size, scales,
                      block_tables, max_blocks, kv_begin, kv_end, 1, n_seqs, max_q_per_seq, causal, sm_scale, flags,
                      o_acc, lse2, out, err, nullptr, 0, stream);
}

extern "C" int zx_paged_attention_ring(const uint16_t *q, int64_t n_q, const int32_t *cu_q, const int32_t *q_pos0,
                                       int32_t n_q_heads, const uint8_t *pool, int64_t n_pages, int32_t n_kv_heads,
                                       int32_t head_dim, int32_t page_size, const float *scales,
                                       const int32_t *block_tables, int32_t max_blocks, const int32_t *kv_begin,
                                       const int32_t *kv_end, int32_t n_ranges, int32_t n_seqs, int32_t max_q_per_seq,
                                       int32_t causal, float sm_scale, int32_t flags, float *o_acc, float *lse2,
                                       uint16_t *out, int32_t *err, zx_stream_t stream) {
  clear_error();
  return prefill_impl(q, n_q, cu_q, q_pos0, n_q_heads, pool, n_pages, n_kv_heads, head_dim, page_size, scales,
                      block_tables, max_blocks, kv_begin, kv_end, n_ranges, n_seqs, max_q_per_seq, causal, sm_scale,
                      flags, o_acc, lse2, out, err, nullptr, 0, stream);
}
