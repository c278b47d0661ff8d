// zx_attention.hip -- decode attention straight from the paged FP8 pool.
//
// One query token per sequence attends to its K/V pages without materialising bf16 K/V
// (the attention that consumes FP8 pages directly, QuantizedRingAttention README.md:344):
//   s_t = sm_scale * q . K_t,  K_t = decode(code) * scale_k     (t < seq_len)
//   out = sum_t softmax(s)_t V_t,  V_t = decode(code) * scale_v
// HBM traffic is 1 B per K/V element (the gather + dequant path moves 3 B and then the
// attention reads 2 B more).
//
// Split-K flash decoding with the work dealt evenly.  The positions of all sequences are cut
// into units (what the four waves of a block take per step), laid end to end, and every
// block of a (kv head, group of query heads) takes an equal run of units (att_locate), so
// sequences of different lengths leave no block empty and none late.  A run may end one
// sequence and begin the next: each part of it that lies in one sequence is a segment, with
// its own running softmax.  A segment that is a whole sequence is finished by its block;
// others leave a partial (m, l, acc[D]) per query head in the workspace, and pass 2
// (paged_decode_combine_kernel) merges a sequence's partials and writes bf16.  Many short
// sequences are dealt whole instead (att_take_whole).  Which it is, and where a run begins,
// follows from the lengths on the device, not from the width of the block tables: up to 64
// sequences every wave finds it in its lanes, for more paged_decode_plan_kernel writes it
// into the workspace.
//
// paged_decode_partial_kernel (any head_dim and page size): lane l of a wave owns 16
// channels (dc = l % LPT, LPT = D / 16 lanes per token) of token slot l / LPT, so K and V
// rows are read as 16-byte loads that cover whole page rows.  Scale factors fold into the
// score (scale_k * sm_scale * log2 e) and into the end (scale_v), so the inner loop works on
// decoded codes.  Each wave keeps an online softmax (running max m, sum l, accumulator
// acc[G][16] per lane, exp2 domain) over steps of ATT_U passes; at the end the token slots
// and the block's 4 waves are combined.  paged_decode_mfma_kernel does the same on the
// matrix cores where its tiles fit.
//
// Bound by HBM reads of the codes (1 B per element) once contexts are long, by the chain of
// a block's first loads before.  One layer, Hq 32 / Hkv 8, D = 128, pages of 16, on the GPU,
// against fixed splits of at least 1,024 positions (most of them empty or alone in a last
// round when lengths differ): 1 x 2,048 20.8 -> 9.9 us; 16 x 1k-8k 50 -> 29 us (4.1 TB/s);
// 64 x 512-4k 90 -> 59 us; 1,024 x 600 273 -> 225 us; 64 x 32k 673 -> 663 us (6.5 TB/s).
#include <algorithm>

#include "zx_attn_common.h"

namespace zx {

constexpr int ATT_THREADS = 256;  // 4 waves
constexpr int ATT_WAVES = ATT_THREADS / 64;
constexpr int ATT_U = 4;          // passes per online-softmax step
constexpr int AM_ROWS = 16;  // query heads a block of the matrix-core variant can hold (the M rows of a tile)

struct AttnGeom {
  int32_t n_q_heads, n_kv_heads, head_dim, page_size, max_blocks, n_seqs;
  int32_t n_run;        // equal runs, one block per head group each
  uint32_t unit, cap;   // positions per unit (a power of two); positions a block table holds
  uint32_t tail;        // see att_take_whole
  int32_t whole;        // every sequence is taken whole: known to the host
  int32_t group, n_group;       // query heads per block; groups of them
  uint32_t p_magic;  // t / page_size = (t * p_magic) >> (31 + p_shift) for t < 2^31
  int32_t p_shift;
  int64_t n_pages;
  float sm_scale;
};

__device__ __forceinline__ uint32_t page_of(const AttnGeom &g, uint32_t t) {
  return (uint32_t)(((uint64_t)t * g.p_magic) >> (31 + g.p_shift));
}

// Positions of a sequence that are attended to (lengths are int32).
__device__ __forceinline__ uint32_t att_live_len(const AttnGeom &g, int32_t len) {
  return len > 0 ? min((uint32_t)len, g.cap) : 0u;
}
__device__ __forceinline__ uint32_t att_units(const AttnGeom &g, int32_t len) {
  return (att_live_len(g, len) + (g.unit - 1)) / g.unit;  // unit: a power of two
}

// The U units of all sequences dealt to n_run runs: run x takes q = U / n_run of them, the
// first r = U % n_run one more.  T: 32 bits where U fits.
template <typename T> struct AttnDeal {
  T q, r;
  __device__ AttnDeal(T q_, T r_) : q(q_), r(r_) {}
  __device__ T begin(T x) const { return x * q + min(x, r); }
  __device__ T run_of(T u) const { return u < r * (q + 1) ? u / (q + 1) : r + (u - r * (q + 1)) / q; }
};

// Whole sequences instead of equal runs?  A run starts anew in every sequence that it touches
// (q, the first page ids, K and V one after the other: about as long as four units) and its
// parts are merged; whole sequences leave blocks idle while the longest one ends.  With as many
// sequences as runs or more, where most runs would start anew anyway: if the longest one has
// at most ATT_TAIL_MANY positions and an eighth of an equal share.  Else if it exceeds a share
// by at most ATT_TAIL_ONE units.  (g.tail: that slack in units; a call whose longest sequence
// is within it needs no sums.)  In a graph, Hq 32 / Hkv 8, D = 128, tables of 32k positions:
// 512 x 100-500 139 us in runs, 90 whole; 4 x 100-500 10.9 in runs, 16.3 whole; 64 x 512-4k
// 59 in runs, 73 whole.
constexpr uint32_t ATT_TAIL_ONE = 2, ATT_TAIL_MANY = 1024;
__device__ __forceinline__ bool att_take_whole(const AttnGeom &g, uint64_t most, uint64_t share) {
  return most <= g.tail + (g.n_seqs < g.n_run ? share : share / 8);
}

// Inclusive sum over the lanes below n (n <= 64, uniform).
__device__ __forceinline__ uint32_t att_scan(uint32_t v, int n) {
  const int lane = threadIdx.x & 63;
  for (int off = 1; off < n; off <<= 1) {
    const uint32_t y = __shfl_up(v, off, 64);
    if (lane >= off) v += y;
  }
  return v;
}

// More than 64 sequences: what every block needs to know, computed once by att_plan_kernel.
struct AttnTable {
  uint64_t *head;   // [4]: whole sequences?, q, r
  uint64_t *first;  // [n_seqs] a sequence's first unit
  int32_t *x0, *n_live;  // [n_seqs] the first run that holds a part of it, and how many do
  int32_t *run_b;        // [n_run] the sequence in which a run begins
  __host__ __device__ AttnTable(void *at, int64_t n_seqs) {
    head = static_cast<uint64_t *>(at);
    first = head + 4;
    x0 = reinterpret_cast<int32_t *>(first + n_seqs);
    n_live = x0 + n_seqs;
    run_b = n_live + n_seqs;
  }
  static size_t bytes(int64_t n_seqs, int64_t n_run) {
    return 4 * sizeof(uint64_t) + (size_t)n_seqs * (sizeof(uint64_t) + 2 * sizeof(int32_t)) +
           (size_t)n_run * sizeof(int32_t);
  }
};

// The run of block x: units [u, u_end), unit u in sequence b, whose first unit is b_first.
// All block-uniform; an empty run has u == u_end.  Up to 64 sequences every lane keeps one
// sequence's length, so that stepping to the next sequence reads no memory.
struct AttnRun {
  uint64_t u, u_end, b_first;
  int32_t b, lane_len;
  int32_t x, y;  // the run (or sequence) and the group of query heads
};
__device__ __forceinline__ int32_t att_len(const AttnGeom &g, const int32_t *seq_lens, const AttnRun &r) {
  return g.n_seqs <= 64 ? __builtin_amdgcn_readlane(r.lane_len, r.b) : seq_lens[r.b];
}
// Lane b's units, and how up to 64 sequences are dealt: whole, or units [begin(x), begin(x +
// 1)) to run x, where incl is the inclusive sum over the sequences.
struct AttnLanes {
  uint32_t n, incl = 0;
  bool whole;
  AttnDeal<uint32_t> deal;
  __device__ AttnLanes(const AttnGeom &g, int32_t lane_len) : n(att_units(g, lane_len)), deal(0, 0) {
    whole = __ballot(n > g.tail) == 0;
    if (whole) return;
    incl = att_scan(n, g.n_seqs);
    const uint32_t all = __builtin_amdgcn_readlane(incl, g.n_seqs - 1);
    deal = AttnDeal<uint32_t>(all / (uint32_t)g.n_run, all % (uint32_t)g.n_run);
    whole = __ballot(!att_take_whole(g, n, deal.q)) == 0;
  }
};
// Block `at` of a one-dimensional grid: the groups of a run (or sequence) are neighbours, so
// that blocks that read the same pages run together, and the blocks without one come last
// (between the others they left three quarters of the CUs idle).
__device__ __forceinline__ AttnRun att_locate(const AttnGeom &g, const int32_t *seq_lens, const AttnTable &t,
                                              uint32_t at) {
  AttnRun r;
  const int lane = threadIdx.x & 63;
  r.lane_len = lane < g.n_seqs ? seq_lens[lane] : 0;
  r.x = (int)(at / (uint32_t)g.n_group);
  r.y = (int)(at - (uint32_t)r.x * (uint32_t)g.n_group);
  const int x = r.x;
  r.b = x;
  r.u = r.u_end = r.b_first = 0;
  bool whole = g.whole;
  uint64_t q = 0, rem = 0;
  if (!whole && g.n_seqs <= 64) {  // every wave by itself
    const AttnLanes l(g, r.lane_len);
    whole = l.whole;
    if (!whole && x < g.n_run) {
      const uint32_t u = l.deal.begin((uint32_t)x), u_end = l.deal.begin((uint32_t)x + 1);
      r.u = u;
      r.u_end = u_end;
      const uint64_t after = __ballot(l.incl > u);  // sequences that end after u; the first holds it
      r.b = after ? __ffsll((long long)after) - 1 : 0;
      r.b_first = __builtin_amdgcn_readlane(l.incl - l.n, r.b);
    }
  } else if (!whole) {
    whole = t.head[0] != 0;
    q = t.head[1];
    rem = t.head[2];
    if (!whole && x < g.n_run) {
      const AttnDeal<uint64_t> deal(q, rem);
      r.u = deal.begin((uint64_t)x);
      r.u_end = deal.begin((uint64_t)x + 1);
      if (r.u < r.u_end) {
        r.b = t.run_b[x];
        r.b_first = t.first[r.b];
      }
    }
  }
  if (whole && x < g.n_seqs) r.u_end = __builtin_amdgcn_readfirstlane(att_units(g, att_len(g, seq_lens, r)));
  return r;
}

// One block: the table of a call of more than 64 sequences.  (Each block of the two passes
// scanned all lengths for itself before, work that grows with the square of the sequences:
// 4,096 x 600 positions 4,580 us, 876 so.)
constexpr int AP_THREADS = 1024;
__global__ void __launch_bounds__(AP_THREADS)
paged_decode_plan_kernel(AttnGeom g, const int32_t *__restrict__ seq_lens, void *table) {
  const AttnTable t(table, g.n_seqs);
  constexpr int WAVES = AP_THREADS / 64;
  __shared__ uint64_t wsum[WAVES];
  __shared__ uint32_t wmax[WAVES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint64_t sum = 0;
  uint32_t most = 0;
  for (int b = threadIdx.x; b < g.n_seqs; b += AP_THREADS) {
    const uint32_t n = att_units(g, seq_lens[b]);
    sum += n;
    most = max(most, n);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    sum += __shfl_xor(sum, off, 64);
    most = max(most, (uint32_t)__shfl_xor((int)most, off, 64));
  }
  if (lane == 0) wsum[wave] = sum, wmax[wave] = most;
  __syncthreads();
  uint64_t U = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    U += wsum[w];
    most = max(most, wmax[w]);
  }
  const AttnDeal<uint64_t> deal(U / (uint64_t)g.n_run, U % (uint64_t)g.n_run);
  const bool whole = att_take_whole(g, most, deal.q);
  if (threadIdx.x == 0) {
    t.head[0] = whole;
    t.head[1] = deal.q;
    t.head[2] = deal.r;
  }
  uint64_t carry = 0;
  for (int b0 = 0; b0 < g.n_seqs; b0 += AP_THREADS) {  // block-uniform
    const int b = b0 + threadIdx.x;
    const uint64_t n = b < g.n_seqs ? att_units(g, seq_lens[b]) : 0;
    uint64_t incl = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint64_t y = __shfl_up(incl, off, 64);
      if (lane >= off) incl += y;
    }
    __syncthreads();  // the sums of the round before have been read
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    uint64_t before = carry;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      if (w < wave) before += wsum[w];
      carry += wsum[w];
    }
    if (b >= g.n_seqs) continue;
    const uint64_t first = before + incl - n;
    t.first[b] = first;
    if (whole || n == 0) {
      t.x0[b] = 0;
      t.n_live[b] = n != 0;
      continue;
    }
    const uint64_t xa = deal.run_of(first), xz = deal.run_of(first + n - 1);
    t.x0[b] = (int32_t)xa;
    t.n_live[b] = (int32_t)(xz - xa + 1);
    for (uint64_t x = deal.begin(xa) < first ? xa + 1 : xa; x <= xz; ++x) t.run_b[x] = b;
  }
}

// Merges the block's four waves' (m, l, acc[G][D]) (in LDS, after a barrier) and stores the
// segment's rows: bf16 rows when the segment is its whole sequence (zeros when no position
// had a page), else partial x + b of the row's n_run + n_seqs (moving along the runs, x or
// b or both grow from one segment to the next, so x + b names a segment).
template <int D, int ROWS>
__device__ __forceinline__ void att_store(const AttnGeom &g, const float (&sm_m)[ATT_WAVES][ROWS],
                                          const float (&sm_l)[ATT_WAVES][ROWS], const float *const (&acc)[ATT_WAVES],
                                          float *part, uint16_t *out, int G, int hq0, int b, int x, bool whole,
                                          float sv) {
  for (int idx = threadIdx.x; idx < G * D; idx += ATT_THREADS) {
    const int j = idx / D, d = idx % D;
    float M = sm_m[0][j];
#pragma unroll
    for (int w = 1; w < ATT_WAVES; ++w) M = fmaxf(M, sm_m[w][j]);
    float a = 0.0f, ll = 0.0f;
#pragma unroll
    for (int w = 0; w < ATT_WAVES; ++w) {
      const float f = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(sm_m[w][j] - M);
      a += f * acc[w][j * D + d];
      ll += f * sm_l[w][j];
    }
    if (whole) {
      const float o = ll == 0.0f ? 0.0f : a / ll * sv;
      out[((int64_t)b * g.n_q_heads + hq0 + j) * D + d] = (uint16_t)(pack_bf16(o, 0.0f) & 0xFFFFu);
    } else {
      float *pp = part + ((int64_t)(hq0 + j) * ((int64_t)g.n_run + g.n_seqs) + x + b) * (2 + D);
      pp[2 + d] = a;
      if (d == 0) {
        pp[0] = M;
        pp[1] = ll;
      }
    }
  }
}

// Zero rows of sequence b (a block that takes whole sequences meets an empty one).
__device__ __forceinline__ void att_zero_rows(const AttnGeom &g, uint16_t *out, int G, int hq0, int b, int D) {
  for (int i = threadIdx.x; i < G * D; i += ATT_THREADS) out[((int64_t)b * g.n_q_heads + hq0) * D + i] = 0;
}

// 16 e4m3 codes -> 16 fp32 values (exact).
__device__ __forceinline__ void decode16(uint4 c, float (&f)[16]) {
  e4m3x4_decode(c.x, f[0], f[1], f[2], f[3]);
  e4m3x4_decode(c.y, f[4], f[5], f[6], f[7]);
  e4m3x4_decode(c.z, f[8], f[9], f[10], f[11]);
  e4m3x4_decode(c.w, f[12], f[13], f[14], f[15]);
}

// Across 16-lane rows: the lane 16 and 32 positions away (ds_bpermute).  (The
// v_permlane16/32_swap builtins return one of their two outputs twice with this
// compiler, so they are not used.)
__device__ __forceinline__ float rows_sum(float v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}
__device__ __forceinline__ float rows_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16, 64));
  return fmaxf(v, __shfl_xor(v, 32, 64));
}
// Max / sum over the token slots of a wave for each channel group: lanes l, l + LPT,
// l + 2 LPT, ... (row_ror by 4 and 8 inside a 16-lane row keeps l % LPT, then the row
// pairs).
template <int LPT> __device__ __forceinline__ float slots_max(float v) {
  if (LPT <= 4) v = fmaxf(v, dpp<0x124>(v));  // row_ror:4
  if (LPT <= 8) v = fmaxf(v, dpp<0x128>(v));  // row_ror:8
  return rows_max(v);
}
template <int LPT> __device__ __forceinline__ float slots_sum(float v) {
  if (LPT <= 4) v += dpp<0x124>(v);
  if (LPT <= 8) v += dpp<0x128>(v);
  return rows_sum(v);
}

// Partial layout in the workspace: [Hq][n_run + B][2 + D] fp32 = (m, l, acc[D]) with m in
// the exp2 domain; a segment without valid positions writes m = -inf, l = 0, acc = 0.
template <int G, int D, bool FAST>
__global__ void __launch_bounds__(ATT_THREADS)
paged_decode_partial_kernel(const uint16_t *__restrict__ q, AttnGeom g, const uint8_t *__restrict__ pool,
                            const float *__restrict__ scales, const int32_t *__restrict__ block_tables,
                            const int32_t *__restrict__ seq_lens, float *__restrict__ part,
                            uint16_t *__restrict__ out, int32_t *err, void *table) {
  constexpr int LPT = D / 16;   // lanes per token
  constexpr int TPW = 64 / LPT;  // token slots per wave pass
  constexpr int STEP = ATT_U * TPW;
  AttnRun run = att_locate(g, seq_lens, AttnTable(table, g.n_seqs), blockIdx.x);
  const int grp_blocks = g.n_q_heads / g.n_kv_heads / G;  // query-head groups per kv head
  const int h = run.y / grp_blocks;
  const int hq0 = h * (g.n_q_heads / g.n_kv_heads) + (run.y % grp_blocks) * G;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: scalar addressing
  const int ts = lane / LPT, dc = lane % LPT;
  const int64_t page_bytes = 2LL * g.n_kv_heads * g.page_size * D;
  const uint8_t *kbase = pool + (int64_t)h * g.page_size * D + dc * 16;
  const int64_t v_off = (int64_t)g.n_kv_heads * g.page_size * D;
  const float qs = scales[h] * g.sm_scale * ATT_LOG2E;
  __shared__ float sm_m[ATT_WAVES][G], sm_l[ATT_WAVES][G];
  __shared__ float sm_acc[ATT_WAVES][G][D];
  int32_t e = 0;
  if (g.whole && run.u == run.u_end) att_zero_rows(g, out, G, hq0, run.b, D);
  while (run.u < run.u_end) {
    const int b = run.b;
    const int32_t len = att_len(g, seq_lens, run);
    const uint32_t b_units = att_units(g, len);
    const uint32_t seg_end = (uint32_t)min(run.u_end - run.b_first, (uint64_t)b_units);
    const bool whole_seq = run.u == run.b_first && seg_end == b_units;
    const uint32_t t_begin = (uint32_t)(run.u - run.b_first) * g.unit;
    const uint32_t t_end = min(att_live_len(g, len), seg_end * g.unit);
    if (t_begin < t_end) {
      const int32_t *bt = block_tables + (int64_t)b * g.max_blocks;

      // q as bf16 pairs for this lane's 16 channels; the score scale (scale_k * sm_scale *
      // log2 e) multiplies the reduced dot product
      uint32_t qb[G][8];
#pragma unroll
      for (int j = 0; j < G; ++j) {
        const uint4 *qp = reinterpret_cast<const uint4 *>(q + ((int64_t)b * g.n_q_heads + hq0 + j) * D + dc * 16);
        const uint4 a = qp[0], c = qp[1];
        qb[j][0] = a.x; qb[j][1] = a.y; qb[j][2] = a.z; qb[j][3] = a.w;
        qb[j][4] = c.x; qb[j][5] = c.y; qb[j][6] = c.z; qb[j][7] = c.w;
      }

      float m[G], l[G], acc[G][16];
#pragma unroll
      for (int j = 0; j < G; ++j) {
        m[j] = -INFINITY;
        l[j] = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[j][i] = 0.0f;
      }
      // positions past the block table are not attended to, and flagged
      if (threadIdx.x == 0 && (int64_t)len > (int64_t)g.max_blocks * g.page_size) e |= ZX_KERR_POS_RANGE;

      // K/V of one step (ATT_U passes of TPW positions) into registers.  FAST (page size a
      // multiple of TPW): the TPW positions of a pass share one page, so the page id is a
      // scalar load and the loads go through a resource whose num_records ends at the last
      // valid row; otherwise every lane looks its page up.  ok marks positions with data.
      auto load_step = [&](int64_t t0, uint4 (&kc)[ATT_U], uint4 (&vc)[ATT_U], bool (&ok)[ATT_U]) {
#pragma unroll
        for (int u = 0; u < ATT_U; ++u) {
          if constexpr (FAST) {
            const int64_t tp = t0 + u * TPW;  // uniform
            const int64_t rows = min((int64_t)TPW, t_end - tp);
            int nrec = 0;
            const uint8_t *src = pool;
            if (rows > 0) {
              const uint32_t bi = page_of(g, (uint32_t)tp);
              const int64_t page = bt[bi];
              if (page < 0 || page >= g.n_pages) e |= ZX_KERR_PAGE_RANGE;
              else {
                src = pool + page * page_bytes + (int64_t)h * g.page_size * D + (tp - (int64_t)bi * g.page_size) * D;
                nrec = (int)rows * D;
              }
            }
            const __amdgpu_buffer_rsrc_t rk =
                __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(src), (short)0, nrec, 0x00020000);
            const __amdgpu_buffer_rsrc_t rv =
                __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(src + (nrec ? v_off : 0)), (short)0, nrec, 0x00020000);
            typedef unsigned int v4u __attribute__((ext_vector_type(4)));
            const v4u a = __builtin_amdgcn_raw_buffer_load_b128(rk, ts * D + dc * 16, 0, 2);
            const v4u c = __builtin_amdgcn_raw_buffer_load_b128(rv, ts * D + dc * 16, 0, 2);
            kc[u] = make_uint4(a.x, a.y, a.z, a.w);
            vc[u] = make_uint4(c.x, c.y, c.z, c.w);
            ok[u] = ts * D < nrec;
          } else {
            // branch-free (positions clamped into the segment, bad pages read the pool's first):
            // with a branch per pass the loop over segments kept 286 registers with four heads,
            // one wave per SIMD (64 x 2k-8k, D = 64, pages of 24: 189 us, 113 so)
            const uint32_t t = (uint32_t)t0 + u * TPW + ts, tc = min(t, t_end - 1);
            const uint32_t bi = page_of(g, tc);
            const int32_t page = bt[bi];
            const bool live = t < t_end, good = page >= 0 && page < g.n_pages;
            e |= live && !good ? ZX_KERR_PAGE_RANGE : 0;
            ok[u] = live && good;
            const uint8_t *kp =
                kbase + (ok[u] ? page * page_bytes + (int64_t)(tc - bi * (uint32_t)g.page_size) * D : 0);
            kc[u] = *reinterpret_cast<const uint4 *>(kp);
            const uint4 v = *reinterpret_cast<const uint4 *>(kp + v_off);
            vc[u] = ok[u] ? v : make_uint4(0, 0, 0, 0);  // (weight 0 times a NaN code)
          }
        }
      };

      auto compute_step = [&](const uint4 (&kc)[ATT_U], const uint4 (&vc)[ATT_U], const bool (&ok)[ATT_U]) {
        float s[ATT_U][G];
#pragma unroll
        for (int u = 0; u < ATT_U; ++u) {
          uint32_t kb[8];
          decode16_bf16(kc[u], kb);
#pragma unroll
          for (int j = 0; j < G; ++j) {
            float a = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i)
              a = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(att_bf2, qb[j][i]), __builtin_bit_cast(att_bf2, kb[i]),
                                                  a, false);
            a = group_sum<LPT>(a);
            s[u][j] = ok[u] ? a * qs : -INFINITY;
          }
        }
        // running max per head (the same in every lane); the accumulators are rescaled only
        // on the steps where some head's max grew (a scalar branch: rare after the first
        // steps of a split)
        float m_new[G];
        bool grew = false;
#pragma unroll
        for (int j = 0; j < G; ++j) {
          float mx = s[0][j];
#pragma unroll
          for (int u = 1; u < ATT_U; ++u) mx = fmaxf(mx, s[u][j]);
          mx = slots_max<LPT>(mx);
          m_new[j] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, fmaxf(m[j], mx))));
          grew = grew || m_new[j] > m[j];
        }
        if (grew) {
#pragma unroll
          for (int j = 0; j < G; ++j) {
            const float alpha = m_new[j] == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m[j] - m_new[j]);
            m[j] = m_new[j];
            l[j] *= alpha;
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[j][i] *= alpha;
          }
        }
#pragma unroll
        for (int j = 0; j < G; ++j) {
#pragma unroll
          for (int u = 0; u < ATT_U; ++u) s[u][j] = m[j] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(s[u][j] - m[j]);
        }
#pragma unroll
        for (int u = 0; u < ATT_U; ++u) {
          float v[16];
          decode16(vc[u], v);
#pragma unroll
          for (int j = 0; j < G; ++j) {
            l[j] += s[u][j];
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[j][i] = __builtin_fmaf(s[u][j], v[i], acc[j][i]);
          }
        }
      };

      // wave w takes steps w, w + 4, ...; the next step's loads are issued before the
      // current step is computed
      const int64_t stride = (int64_t)ATT_WAVES * STEP;
      int64_t t0 = t_begin + (int64_t)wave * STEP;
      uint4 ka[ATT_U], va[ATT_U], kb2[ATT_U], vb2[ATT_U];
      bool oka[ATT_U], okb[ATT_U];
      if (t0 < t_end) load_step(t0, ka, va, oka);
      while (t0 < t_end) {
        if (t0 + stride < t_end) load_step(t0 + stride, kb2, vb2, okb);
        compute_step(ka, va, oka);
        t0 += stride;
        if (t0 >= t_end) break;
        if (t0 + stride < t_end) load_step(t0 + stride, ka, va, oka);
        compute_step(kb2, vb2, okb);
        t0 += stride;
      }

      // token slots of the wave -> one value per (head, channel) in every lane of slot 0
#pragma unroll
      for (int j = 0; j < G; ++j) {
        l[j] = slots_sum<LPT>(l[j]);
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[j][i] = slots_sum<LPT>(acc[j][i]);
      }
      // the block's waves meet in LDS
      if (ts == 0) {
#pragma unroll
        for (int j = 0; j < G; ++j) {
#pragma unroll
          for (int i = 0; i < 16; ++i) sm_acc[wave][j][dc * 16 + i] = acc[j][i];
          if (dc == 0) {
            sm_m[wave][j] = m[j];
            sm_l[wave][j] = l[j];
          }
        }
      }
    }
    __syncthreads();
    const float *const accs[ATT_WAVES] = {&sm_acc[0][0][0], &sm_acc[1][0][0], &sm_acc[2][0][0], &sm_acc[3][0][0]};
    if (t_begin < t_end)
      att_store<D, G>(g, sm_m, sm_l, accs, part, out, G, hq0, b, run.x, whole_seq, scales[g.n_kv_heads + h]);
    run.u = run.b_first + seg_end;
    run.b_first += b_units;
    ++run.b;
    __syncthreads();
  }
  if (e && err) atomicOr(err, e);
}

// Matrix-core variant of pass 1 for D = 64 and 128 and page sizes that are a multiple of 16:
// q.K^T and P.V run on v_mfma_f32_16x16x32_bf16 with the (up to 16) query heads of the
// block as the M rows (padded to 16), so up to 16 query heads of a kv head read its pages
// once.  A wave takes steps of 32 positions (two 16-token
// tiles, each inside one page).  The K and V codes of a tile arrive as two contiguous
// 1 KiB loads per run (lane l: token 8 i + l / 8, channels 16 (l % 8) ..+16: whole cache
// lines per instruction) and are rearranged on chip:
//   * K codes go through a staging area (144-byte token rows) and come back as lane
//     (n, kg) = token n, channels 32 kg ..+32, converted to bf16 exactly: the B operand
//     of q.K^T (k = channel; any channel permutation shared with q's A operand works,
//     since the product sums over channels);
//   * V values go into LDS as bf16 token rows (288-byte rows: the four rows a 16-lane
//     group reads fall on distinct banks) with two 16-byte stores per load, and the B
//     operand of P.V (8 consecutive tokens of one channel per lane) comes back through
//     gfx950's transposing LDS read, ds_read_b64_tr_b16 (2% faster than storing V^T with
//     64 two-byte stores per lane and step).
// P goes through LDS as fp32 into the A-operand layout and is split into bf16 terms: for
// D = 128 hi + lo (two MFMAs), which keeps the products at ~2^-17 relative error; for D = 64
// the rest as well (three MFMAs: all 24 bits of P, as in the fp32 products of the kernel
// above: where values nearly cancel the error against 64 bits is 2^-24 max|V| as there, and
// 2^-18.5 with two terms; 16 x 1k-8k, Hq 32 / Hkv 8: 24.2 us against 23.3).  Scores land in the C
// layout: lane row kg (16 lanes) holds heads 4 kg ..+4 of token l % 16, so the softmax
// bookkeeping is a 16-lane DPP reduction per head; the O accumulators (8 tiles of 16
// channels) live in MFMA results, rows = heads.
typedef short att_i16x4 __attribute__((ext_vector_type(4)));
constexpr int AM_STEP = 32;                       // positions per wave and step
constexpr int AM_PROW = 36;                       // floats per head row of P (32 tokens + 4 pad)
constexpr int AM_PBYTES = AM_ROWS * AM_PROW * 4;  // one wave's P (16 heads x 32 tokens fp32)
template <int D> struct AmLds {
  static constexpr int VROW = 2 * D + 32;        // bytes per token row of V (bf16 + pad)
  static constexpr int VBYTES = AM_STEP * VROW;  // one wave's V (32 tokens)
  static constexpr int KROW = D + 16;            // bytes per token row of the K staging (codes + pad)
  static constexpr int KBYTES = AM_STEP * KROW;  // one wave's K codes (32 tokens)
  static constexpr int WAVE = VBYTES + AM_PBYTES + KBYTES;
};

template <int D>
__global__ void __launch_bounds__(ATT_THREADS, 2)
paged_decode_mfma_kernel(const uint16_t *__restrict__ q, AttnGeom g, const uint8_t *__restrict__ pool,
                         const float *__restrict__ scales, const int32_t *__restrict__ block_tables,
                         const int32_t *__restrict__ seq_lens, float *__restrict__ part,
                         uint16_t *__restrict__ out, int32_t *err, void *table) {
  using Lds = AmLds<D>;
  constexpr int LPT = D / 16;   // lanes per token of a 16-byte load
  constexpr int TPL = 64 / LPT;  // tokens per load
  constexpr int NL = 16 / TPL;   // loads per 16-token tile
  constexpr int CPK = D / 4;     // channels per lane row kg of the q.K^T operands
  constexpr int NC = D / 32;     // q.K^T products per tile
  constexpr int NT = D / 16;     // 16-channel tiles of O
  constexpr bool P3 = D == 64;   // P in three bf16 terms
  const int G = g.group;
  AttnRun run = att_locate(g, seq_lens, AttnTable(table, g.n_seqs), blockIdx.x);
  const int grp_blocks = g.n_q_heads / g.n_kv_heads / G;
  const int h = run.y / grp_blocks;
  const int hq0 = h * (g.n_q_heads / g.n_kv_heads) + (run.y % grp_blocks) * G;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, kg = lane >> 4;  // MFMA column / k-group
  const int64_t page_bytes = 2LL * g.n_kv_heads * g.page_size * D;
  const int64_t head_off = (int64_t)h * g.page_size * D;
  const int64_t v_off = (int64_t)g.n_kv_heads * g.page_size * D;
  const float qs = scales[h] * g.sm_scale * ATT_LOG2E;
  __shared__ __attribute__((aligned(16))) uint8_t lds[ATT_WAVES][Lds::WAVE];
  __shared__ float sm_m[ATT_WAVES][AM_ROWS], sm_l[ATT_WAVES][AM_ROWS];
  uint8_t *vt = lds[wave];
  float *pl = reinterpret_cast<float *>(lds[wave] + Lds::VBYTES);
  uint8_t *ks = lds[wave] + Lds::VBYTES + AM_PBYTES;
  int32_t e = 0;
  if (g.whole && run.u == run.u_end) att_zero_rows(g, out, G, hq0, run.b, D);
  while (run.u < run.u_end) {
    const int b = run.b;
    const int32_t len = att_len(g, seq_lens, run);
    const uint32_t b_units = att_units(g, len);
    const uint32_t seg_end = (uint32_t)min(run.u_end - run.b_first, (uint64_t)b_units);
    const bool whole_seq = run.u == run.b_first && seg_end == b_units;
    const uint32_t t_begin = (uint32_t)(run.u - run.b_first) * g.unit;
    const uint32_t t_end = min(att_live_len(g, len), seg_end * g.unit);
    if (t_begin < t_end) {
      // positions past the block table are not attended to, and flagged
      if (threadIdx.x == 0 && (int64_t)len > (int64_t)g.max_blocks * g.page_size) e |= ZX_KERR_POS_RANGE;
      const int32_t *bt = block_tables + (int64_t)b * g.max_blocks;

      // q rows (heads) as the A operand: lane l holds head n, channels CPK kg + 8 c .. +8
      att_bf16x8 qa[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        att_u32x4 w = {0u, 0u, 0u, 0u};
        if (n < G) {
          const uint4 x = *reinterpret_cast<const uint4 *>(q + ((int64_t)b * g.n_q_heads + hq0 + n) * D + kg * CPK + c * 8);
          w = att_u32x4{x.x, x.y, x.z, x.w};
        }
        qa[c] = __builtin_bit_cast(att_bf16x8, w);
      }

      att_f32x4 o[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) o[t] = att_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      float m[4], l[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        m[j] = -INFINITY;
        l[j] = 0.0f;
      }

      // one 16-token tile: K and V codes of token tp + n, channels CPK kg ..+CPK; rows = valid tokens.
      // Branch-free: the block-table entry is read for a position clamped into the split
      // (always a valid index), validity is a select, and a tile past the end or on a bad
      // page loads through resources with num_records = 0 (zeros, no memory traffic).  Every
      // step therefore issues the same loads, so the compiler's s_waitcnt counts only wait
      // for the step being computed and the next step's loads stay in flight.
      const uint32_t t_last = t_end - 1;
      // page id of the tile at tp (position clamped into the split: always a valid index)
      auto tile_page = [&](uint32_t tp) -> int32_t {
        return bt[page_of(g, min(tp, t_last))];
      };
      auto load_tile = [&](uint32_t tp, int32_t page, uint4 (&kc)[NL], uint4 (&vc)[NL], int &rows) {
        const int live = tp < t_end ? (int)min(16u, t_end - tp) : 0;
        const uint32_t tc = min(tp, t_last);
        const uint32_t bi = page_of(g, tc);
        const bool ok = page >= 0 && page < g.n_pages;
        e |= (live > 0 && !ok) ? ZX_KERR_PAGE_RANGE : 0;
        rows = ok ? live : 0;
        const int nrec = rows * D;
        const uint8_t *src = pool + (ok ? (int64_t)page * page_bytes + head_off + (int64_t)(tc - bi * (uint32_t)g.page_size) * D : 0);
        const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(src), (short)0, nrec,
                                                                            0x00020000);
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t *>(src + (ok ? v_off : 0)), (short)0, nrec, 0x00020000);
        // contiguous: load i gives lane l the 16 codes of token TPL i + l / LPT, channels
        // 16 (l % LPT) ..+16, so one instruction reads 1 KiB of whole cache lines (the mapping
        // that gives each lane its MFMA operand directly touches half lines and was ~20%
        // slower on the same bytes); the operand layout is made on chip
#pragma unroll
        for (int i = 0; i < NL; ++i) {
          const att_u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(rk, 16 * lane + 1024 * i, 0, 2);
          const att_u32x4 c = __builtin_amdgcn_raw_buffer_load_b128(rv, 16 * lane + 1024 * i, 0, 2);
          kc[i] = make_uint4(a.x, a.y, a.z, a.w);
          vc[i] = make_uint4(c.x, c.y, c.z, c.w);
        }
      };

      auto compute_step = [&](const uint4 (&kc)[2][NL], const uint4 (&vc)[2][NL], const int (&rows)[2]) {
        // K codes through the staging rows: written as loaded, read back as lane (n, kg) =
        // token n, channels CPK kg ..+CPK (D = 128: 144-byte rows, the 16 rows of a read hit distinct banks)
#pragma unroll
        for (int T = 0; T < 2; ++T)
#pragma unroll
          for (int i = 0; i < NL; ++i)
            *reinterpret_cast<uint4 *>(ks + (T * 16 + TPL * i + lane / LPT) * Lds::KROW + 16 * (lane % LPT)) = kc[T][i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // scores: S[head][token] for both tiles
        float sv[2][4];
#pragma unroll
        for (int T = 0; T < 2; ++T) {
          uint32_t kb[4 * NC];
          const uint8_t *kr = ks + (T * 16 + n) * Lds::KROW + kg * CPK;
#pragma unroll
          for (int i = 0; i < CPK / 16; ++i)
            decode16_bf16(*reinterpret_cast<const uint4 *>(kr + 16 * i), *reinterpret_cast<uint32_t (*)[8]>(&kb[8 * i]));
          att_f32x4 sc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int c = 0; c < NC; ++c)
            sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                qa[c], __builtin_bit_cast(att_bf16x8, att_u32x4{kb[4 * c], kb[4 * c + 1], kb[4 * c + 2], kb[4 * c + 3]}),
                sc, 0, 0, 0);
#pragma unroll
          for (int j = 0; j < 4; ++j)
            sv[T][j] = (4 * kg + j < G && n < rows[T]) ? sc[j] * qs : -INFINITY;
        }
        float m_new[4];
        bool grew = false;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          m_new[j] = fmaxf(m[j], row16_max(fmaxf(sv[0][j], sv[1][j])));
          grew = grew || m_new[j] > m[j];
        }
        // the accumulators are rescaled only on the steps where some head's max grew
        if (__builtin_amdgcn_ballot_w64(grew)) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float alpha = m_new[j] == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m[j] - m_new[j]);
            m[j] = m_new[j];
            l[j] *= alpha;
#pragma unroll
            for (int t = 0; t < NT; ++t) o[t][j] *= alpha;
          }
        }
        // P (fp32) into LDS as [head][token]
#pragma unroll
        for (int T = 0; T < 2; ++T)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float p = m[j] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(sv[T][j] - m[j]);
            l[j] += p;
            if (4 * kg + j < G) pl[(4 * kg + j) * AM_PROW + T * 16 + n] = p;
          }
        // V into LDS as token rows (VROW bytes, channels in order, bf16): load i of tile T
        // gave lane l token t = 16 T + TPL i + l / LPT, channels 16 (l % LPT) ..+16: 32 bytes
#pragma unroll
        for (int T = 0; T < 2; ++T)
#pragma unroll
          for (int i = 0; i < NL; ++i) {
            uint32_t vb[8];
            decode16_bf16(vc[T][i], vb);
            const int t = T * 16 + TPL * i + lane / LPT;
            uint4 *row = reinterpret_cast<uint4 *>(vt + t * Lds::VROW + 32 * (lane % LPT));
            row[0] = make_uint4(vb[0], vb[1], vb[2], vb[3]);
            row[1] = make_uint4(vb[4], vb[5], vb[6], vb[7]);
          }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // A operand: P[head n][tokens 8 kg ..+8], split into bf16 hi + lo (+ the rest)
        att_bf16x8 ah, al, ar;
        {
          float pr[8];
          if (n < G) {
            const float4 a = *reinterpret_cast<const float4 *>(pl + n * AM_PROW + kg * 8);
            const float4 c = *reinterpret_cast<const float4 *>(pl + n * AM_PROW + kg * 8 + 4);
            pr[0] = a.x; pr[1] = a.y; pr[2] = a.z; pr[3] = a.w; pr[4] = c.x; pr[5] = c.y; pr[6] = c.z; pr[7] = c.w;
          } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) pr[i] = 0.0f;
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            ah[i] = (__bf16)pr[i];
            const float rest = pr[i] - (float)ah[i];
            al[i] = (__bf16)rest;
            if constexpr (P3) ar[i] = (__bf16)(rest - (float)al[i]);
          }
        }
        // B operand per 16-channel tile: V^T[channel 16 jt + n][tokens 8 kg ..+8]
#pragma unroll
        for (int jt = 0; jt < NT; ++jt) {
          // two transposing reads (ds_read_b64_tr_b16): within each 16-lane group kg, lane L
          // reads channels 16 jt + 4 (L % 4) ..+4 of token 8 kg + L / 4 (+4), and lane n
          // receives channel 16 jt + n of the four tokens, the B operand's k = 8 kg ..+4 (+4)
          const uint8_t *src = vt + (8 * kg + (n >> 2)) * Lds::VROW + 2 * (16 * jt + 4 * (n & 3));
          const att_i16x4 w0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) att_i16x4 *)(src));
          const att_i16x4 w1 =
              __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) att_i16x4 *)(src + 4 * Lds::VROW));
          const att_bf16x8 bv = __builtin_bit_cast(
              att_bf16x8, att_u32x4{__builtin_bit_cast(uint2, w0).x, __builtin_bit_cast(uint2, w0).y,
                                    __builtin_bit_cast(uint2, w1).x, __builtin_bit_cast(uint2, w1).y});
          o[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bv, o[jt], 0, 0, 0);
          o[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bv, o[jt], 0, 0, 0);
          if constexpr (P3) o[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ar, bv, o[jt], 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      };

      // steps of 32 positions: wave w takes steps w, w + 4, ...; a step's K/V loads are issued
      // one step ahead and its two page ids one step before that, so no step waits on a
      // block-table read before it can issue its loads.  (Two steps ahead, in a third register
      // buffer, needs the running maxima in scalar registers: 253 VGPRs and 48 SGPRs spilled,
      // 5-10% slower on everything but the longest batch, where it was 1% slower.)
      constexpr uint32_t stride = ATT_WAVES * AM_STEP;
      uint32_t t0 = t_begin + (uint32_t)wave * AM_STEP;
      uint4 k0[2][NL], v0[2][NL], k1[2][NL], v1[2][NL];
      int r0[2], r1[2];
      int32_t p0[2], p1[2];
      auto pages_of_step = [&](uint32_t ts0, int32_t (&p)[2]) {
        p[0] = tile_page(ts0);
        p[1] = tile_page(ts0 + 16);
      };
      auto load_step = [&](uint32_t ts0, const int32_t (&p)[2], uint4 (&kc)[2][NL], uint4 (&vc)[2][NL],
                           int (&rows)[2]) {
        load_tile(ts0, p[0], kc[0], vc[0], rows[0]);
        load_tile(ts0 + 16, p[1], kc[1], vc[1], rows[1]);
      };
      // past the end the loads are zero-length
      pages_of_step(t0, p0);
      load_step(t0, p0, k0, v0, r0);
      pages_of_step(t0 + stride, p1);
      while (t0 < t_end) {
        load_step(t0 + stride, p1, k1, v1, r1);
        pages_of_step(t0 + 2 * stride, p0);
        compute_step(k0, v0, r0);
        t0 += stride;
        if (t0 >= t_end) break;
        load_step(t0 + stride, p0, k0, v0, r0);
        pages_of_step(t0 + 2 * stride, p1);
        compute_step(k1, v1, r1);
        t0 += stride;
      }

      // l over the 16 token lanes; then the block's waves meet in LDS (a wave's O rows take the
      // place of its own V rows, which it has read)
#pragma unroll
      for (int j = 0; j < 4; ++j) l[j] = group_sum<16>(l[j]);
      static_assert(AM_ROWS * D * 4 <= Lds::VBYTES, "a wave's O fits where its V was");
      float *acc_w = reinterpret_cast<float *>(vt);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * kg + j < G) {
#pragma unroll
          for (int t = 0; t < NT; ++t) acc_w[(4 * kg + j) * D + 16 * t + n] = o[t][j];
          if (n == 0) {
            sm_m[wave][4 * kg + j] = m[j];
            sm_l[wave][4 * kg + j] = l[j];
          }
        }
    }
    __syncthreads();
    const float *const accs[ATT_WAVES] = {reinterpret_cast<const float *>(lds[0]), reinterpret_cast<const float *>(lds[1]),
                                          reinterpret_cast<const float *>(lds[2]), reinterpret_cast<const float *>(lds[3])};
    if (t_begin < t_end)
      att_store<D, AM_ROWS>(g, sm_m, sm_l, accs, part, out, G, hq0, b, run.x, whole_seq, scales[g.n_kv_heads + h]);
    run.u = run.b_first + seg_end;
    run.b_first += b_units;
    ++run.b;
    __syncthreads();
  }
  if (e && err) atomicOr(err, e);
}

// Pass 2: out[b][hq][:] = scale_v * sum_s 2^(m_s - M) acc_s / sum_s 2^(m_s - M) l_s over
// the segments of sequence b.  A wave owns 64 channels of one row; its lanes hold the
// maxima and sums of 64 segments at a time, whose weights reach the channels by readlane,
// so there is no LDS and no barrier, and several segments' values are loaded
// before the first is used (1 x 2,048 positions, both passes: 20.4 -> 9.5 us, this one's
// share 4.0 -> 3.0; before, a block-wide table and one load at a time).
constexpr int CB_U = 8;  // segments whose values are loaded together
__global__ void __launch_bounds__(256)
paged_decode_combine_kernel(const float *__restrict__ part, AttnGeom g, const float *__restrict__ scales,
                            const int32_t *__restrict__ seq_lens, uint16_t *__restrict__ out, void *table) {
  const int D = g.head_dim;
  const int lane = threadIdx.x & 63;
  const int64_t row = blockIdx.x;  // b * Hq + hq
  const int d = threadIdx.x;
  const int b = (int)(row / g.n_q_heads);
  const int h = (int)(row % g.n_q_heads) / (g.n_q_heads / g.n_kv_heads);
  // the sequence's first run, and how many hold a part of it
  int32_t x0 = 0, n_live = 0;
  if (g.n_seqs <= 64) {
    const AttnLanes l(g, lane < g.n_seqs ? seq_lens[lane] : 0);
    const uint32_t nb = __builtin_amdgcn_readlane(l.n, b);
    if (l.whole) {
      n_live = nb != 0;
    } else if (nb) {
      const uint32_t last = __builtin_amdgcn_readlane(l.incl, b) - 1;
      x0 = (int32_t)l.deal.run_of(last + 1 - nb);
      n_live = (int32_t)l.deal.run_of(last) - x0 + 1;
    }
  } else {
    const AttnTable t(table, g.n_seqs);
    x0 = t.x0[b];
    n_live = t.n_live[b];
  }
  if (n_live == 1) return;  // the sequence was one segment: its block has written the row
  const float sv = scales[g.n_kv_heads + h];
  const int64_t hq = row % g.n_q_heads;
  const float *pp = part + (hq * ((int64_t)g.n_run + g.n_seqs) + x0 + b) * (2 + D);
  float M = -INFINITY, L = 0.0f, A = 0.0f;
  for (int base = 0; base < n_live; base += 64) {
    const int cnt = min(64, n_live - base);
    const float *p0 = pp + (int64_t)base * (2 + D);
    const float ms = lane < cnt ? p0[lane * (2 + D)] : -INFINITY;
    const float ls = lane < cnt ? p0[lane * (2 + D) + 1] : 0.0f;
    float v[CB_U];
#pragma unroll
    for (int u = 0; u < CB_U; ++u) v[u] = p0[min(u, cnt - 1) * (2 + D) + 2 + d];
    const float Mn = fmaxf(M, xrow_max(row16_max(ms)));
    const float alpha = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(M - Mn);
    const float w = Mn == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ms - Mn);
    M = Mn;
    L = L * alpha + rows_sum(group_sum<16>(w * ls));
    A *= alpha;
    for (int s = 0; s < cnt; s += CB_U) {
      float nx[CB_U];
      if (s + CB_U < cnt) {
#pragma unroll
        for (int u = 0; u < CB_U; ++u) nx[u] = p0[min(s + CB_U + u, cnt - 1) * (2 + D) + 2 + d];
      }
#pragma unroll
      for (int u = 0; u < CB_U; ++u)
        if (s + u < cnt)
          A += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), s + u)) * v[u];
#pragma unroll
      for (int u = 0; u < CB_U; ++u) v[u] = nx[u];
    }
  }
  // a sequence without positions (L = 0) gives zeros
  const float o = L == 0.0f ? 0.0f : A / L * sv;
  out[row * D + d] = (uint16_t)(pack_bf16(o, 0.0f) & 0xFFFFu);
}

}  // namespace zx

using namespace zx;

// Query heads per block.  The matrix-core variant (head_dim 64 and 128, pages of a multiple of
// 16) takes all query heads of a kv head in one block, up to its 16 rows, so their pages are
// read once; with one head per block (one per kv head, or a prime number of more than 16) 15
// of the 16 rows would be padding and the other variant is faster (64 sequences of 2k-8k, 8
// heads: D = 128 109 against 112 us, D = 64 59 against 69; 16 x 1k-8k, 19 heads per kv head,
// D = 64: 221 against 244, D = 128 371 against 384).  That one takes up to four heads per
// block.
static int32_t att_group(int32_t grp, bool mfma) {
  if (!mfma) return grp % 4 == 0 ? 4 : (grp % 2 == 0 ? 2 : 1);
  int g = grp < AM_ROWS ? grp : AM_ROWS;
  while (grp % g) --g;
  return g;
}
static bool att_mfma(int32_t grp, int32_t head_dim, int32_t page_size) {
  return head_dim <= 128 && page_size % 16 == 0 && att_group(grp, true) > 1;
}

// The head_dims the kernels are built for; the plan below holds for these only.
static bool att_dim_ok(int32_t head_dim) { return head_dim == 64 || head_dim == 128 || head_dim == 256; }

// Blocks per group of query heads, and how the sequences are dealt to them.
struct AttnPlan {
  bool mfma, whole;
  int32_t group, unit;
  uint32_t tail;
  int64_t n_run, n_blk;
};
static AttnPlan att_plan(int32_t n_seqs, int32_t n_q_heads, int32_t n_kv_heads, int32_t head_dim, int32_t max_blocks,
                         int32_t page_size) {
  AttnPlan p;
  const int32_t grp = n_q_heads / n_kv_heads;
  p.mfma = att_mfma(grp, head_dim, page_size);
  p.group = att_group(grp, p.mfma);
  p.unit = ATT_WAVES * (p.mfma ? AM_STEP : ATT_U * 64 / (head_dim / 16));
  const int64_t groups = n_q_heads / p.group;
  // units of the longest sequence there can be (lengths are int32)
  const int64_t seq_units = ceil_div(std::min((int64_t)max_blocks * page_size, (int64_t)INT32_MAX), p.unit);
  // resident blocks per group, one equal run each: two per CU (registers, and LDS at D = 128),
  // three where they fit (64 x 2k-8k, D = 64: 65 against 72 us; one head per block 64 against
  // 80, 71 heads on one kv head 297 against 337; at D = 256 1,412 against 1,326 the other way).
  // More runs than resident blocks leave a second, partly filled round: 16 x 1k-8k 37 against
  // 31 us at three per CU.  A number of groups that leaves a part of the CUs without a run takes
  // up to four rounds of shorter ones where those fill the chip by 5% more (152 groups: 3 runs
  // on 456 of 512, or 10 in three rounds: 16 x 1k-8k, 19 heads per kv head, D = 128 371 -> 311
  // us, D = 64 221 -> 164).
  const int64_t resident = ((p.mfma ? head_dim == 64 : p.group == 1 && head_dim < 256) ? 3LL : 2LL) * num_cus();
  int64_t slots = std::max<int64_t>(1, resident / groups);
  double per_round = (double)slots;
  for (int64_t rounds = 2; rounds <= 4; ++rounds) {
    const int64_t n = rounds * resident / groups;
    if ((double)n / rounds > 1.05 * per_round) {
      slots = n;
      per_round = (double)n / rounds;
    }
  }
  p.n_run = std::min(seq_units * n_seqs, slots);
  p.tail = n_seqs >= p.n_run ? std::max<uint32_t>(1, ATT_TAIL_MANY / p.unit) : ATT_TAIL_ONE;
  // Whole sequences whatever their lengths, without the merge's launch: one unit each, or at
  // most 512 positions where they fill half the chip (32 x 100-500: 10.2 us, in runs 17), or
  // so short that att_take_whole() says so anyway (128 x 100-600, 12 heads, D = 64: 26 -> 19).
  p.whole = seq_units == 1 || (seq_units * p.unit <= 512 && n_seqs >= slots / 2) ||
            seq_units <= p.tail;
  p.n_blk = p.whole ? n_seqs : std::max<int64_t>(p.n_run, n_seqs);  // room for either way of dealing
  return p;
}

extern "C" size_t zx_paged_attention_decode_workspace_bytes(int32_t n_seqs, int32_t n_q_heads, int32_t n_kv_heads,
                                                            int32_t head_dim, int32_t max_blocks, int32_t page_size) {
  if (n_seqs <= 0 || n_q_heads <= 0 || n_kv_heads <= 0 || n_q_heads % n_kv_heads || !att_dim_ok(head_dim) ||
      max_blocks <= 0 || page_size <= 0)
    return 0;
  const AttnPlan p = att_plan(n_seqs, n_q_heads, n_kv_heads, head_dim, max_blocks, page_size);
  // partials, then the table (read by 8 bytes: 2 + head_dim is even)
  return (size_t)(n_q_heads * (p.n_run + n_seqs) * (2 + head_dim)) * sizeof(float) +
         (n_seqs > 64 ? AttnTable::bytes(n_seqs, p.n_run) : 0);
}

template <int G, int D>
static int launch_partial(dim3 grid, hipStream_t st, const uint16_t *q, const AttnGeom &g, const uint8_t *pool,
                          const float *scales, const int32_t *bt, const int32_t *sl, float *part, uint16_t *out,
                          int32_t *err, void *table) {
  constexpr int TPW = 64 / (D / 16);
  // (D = 64 with several heads: such pages take the matrix-core variant)
  if ((G == 1 || D > 64) && g.page_size % TPW == 0)
    paged_decode_partial_kernel<G, D, (G == 1 || D > 64)><<<grid, ATT_THREADS, 0, st>>>(q, g, pool, scales, bt, sl, part, out, err, table);
  else
    paged_decode_partial_kernel<G, D, false><<<grid, ATT_THREADS, 0, st>>>(q, g, pool, scales, bt, sl, part, out, err, table);
  return check_launch("paged_decode_partial");
}

template <int D>
static int launch_g(const AttnPlan &p, dim3 grid, hipStream_t st, const uint16_t *q, const AttnGeom &g,
                    const uint8_t *pool, const float *scales, const int32_t *bt, const int32_t *sl, float *part,
                    uint16_t *out, int32_t *err, void *table) {
  if constexpr (D <= 128)
    if (p.mfma) {
      paged_decode_mfma_kernel<D><<<grid, ATT_THREADS, 0, st>>>(q, g, pool, scales, bt, sl, part, out, err, table);
      return check_launch("paged_decode_mfma");
    }
  switch (p.group) {
    case 1: return launch_partial<1, D>(grid, st, q, g, pool, scales, bt, sl, part, out, err, table);
    case 2: return launch_partial<2, D>(grid, st, q, g, pool, scales, bt, sl, part, out, err, table);
    default: return launch_partial<4, D>(grid, st, q, g, pool, scales, bt, sl, part, out, err, table);
  }
}

extern "C" int zx_paged_attention_decode(const uint16_t *q, int32_t n_q_heads, const uint8_t *pool, int64_t n_pages,
                                         int32_t n_kv_heads, int32_t head_dim, int32_t page_size,
                                         const float *scales, const int32_t *block_tables, int32_t max_blocks,
                                         const int32_t *seq_lens, int32_t n_seqs, float sm_scale, uint16_t *out,
                                         int32_t *err, void *workspace,
                                         size_t workspace_bytes, zx_stream_t stream) {
  clear_error();
  ZX_REQUIRE(q && pool && scales && block_tables && seq_lens && out, "paged_attention_decode: null pointer");
  ZX_REQUIRE(aligned16(q) && aligned16(pool) && aligned16(out),
             "paged_attention_decode: q, pool and out must be 16-byte aligned");
  ZX_REQUIRE(n_q_heads > 0 && n_kv_heads > 0 && n_pages > 0 && page_size > 0 && max_blocks > 0 && n_seqs > 0,
             "paged_attention_decode: sizes must be positive");
  ZX_REQUIRE(n_q_heads % n_kv_heads == 0, "paged_attention_decode: n_q_heads must be a multiple of n_kv_heads");
  if (!att_dim_ok(head_dim))
    return fail(ZX_ERR_UNSUPPORTED, "paged_attention_decode: head_dim %d not in {64, 128, 256}", head_dim);
  if (n_seqs > 65535) return fail(ZX_ERR_UNSUPPORTED, "paged_attention_decode: more than 65535 sequences");
  const size_t need =
      zx_paged_attention_decode_workspace_bytes(n_seqs, n_q_heads, n_kv_heads, head_dim, max_blocks, page_size);
  if (!workspace || workspace_bytes < need)
    return fail(ZX_ERR_WORKSPACE, "paged_attention_decode: workspace %zu < %zu bytes", workspace_bytes, need);
  const AttnPlan p = att_plan(n_seqs, n_q_heads, n_kv_heads, head_dim, max_blocks, page_size);
  AttnGeom g;
  g.n_q_heads = n_q_heads;
  g.n_kv_heads = n_kv_heads;
  g.head_dim = head_dim;
  g.page_size = page_size;
  g.max_blocks = max_blocks;
  g.n_seqs = n_seqs;
  g.n_run = (int32_t)p.n_run;
  g.tail = p.tail;
  g.unit = (uint32_t)p.unit;
  g.cap = (uint32_t)std::min((int64_t)max_blocks * page_size, (int64_t)INT32_MAX);
  g.whole = p.whole ? 1 : 0;
  g.group = p.group;
  g.n_pages = n_pages;
  g.sm_scale = sm_scale;
  {  // magic division by the page size for positions below 2^31
    int sh = 0;
    while ((1LL << sh) < page_size) ++sh;
    g.p_shift = sh;
    g.p_magic = (uint32_t)(((1ULL << (31 + sh)) + (uint64_t)page_size - 1) / (uint64_t)page_size);
  }
  const int64_t gy = n_q_heads / p.group;
  if (gy > 65535) return fail(ZX_ERR_UNSUPPORTED, "paged_attention_decode: too many heads");
  ZX_REQUIRE(p.n_blk * gy < (1LL << 31), "paged_attention_decode: too many sequences or heads");
  g.n_group = (int32_t)gy;
  hipStream_t st = as_stream(stream);
  float *part = static_cast<float *>(workspace);
  void *table = part + n_q_heads * (p.n_run + n_seqs) * (2 + head_dim);
  if (n_seqs > 64 && !p.whole) {
    paged_decode_plan_kernel<<<1, AP_THREADS, 0, st>>>(g, seq_lens, table);
    const int prc = check_launch("paged_decode_plan");
    if (prc) return prc;
  }
  const dim3 grid((unsigned)(p.n_blk * gy));
  int rc;
  switch (head_dim) {
    case 64: rc = launch_g<64>(p, grid, st, q, g, pool, scales, block_tables, seq_lens, part, out, err, table); break;
    case 128: rc = launch_g<128>(p, grid, st, q, g, pool, scales, block_tables, seq_lens, part, out, err, table); break;
    default: rc = launch_g<256>(p, grid, st, q, g, pool, scales, block_tables, seq_lens, part, out, err, table); break;
  }
  if (rc || p.whole) return rc;  // every row is written
  paged_decode_combine_kernel<<<(unsigned)((int64_t)n_seqs * n_q_heads), head_dim, 0, st>>>(part, g, scales, seq_lens,
                                                                                            out, table);
  return check_launch("paged_decode_combine");
}
