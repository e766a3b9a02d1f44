// Paged causal GQA attention for the verify pass (T = k+1 queries per row), 1-token decode and
// prefill, reading keys/values straight from the block pool.
//
// Reference: paged.py:80-81 (gather every table block) + model.py:70-76 (repeat_interleave GQA,
// key_pos <= query_pos mask, scaled_dot_product_attention with scale 1/sqrt(D)).
//
// Work split (all kernels): the keys of a row are cut into fixed chunks of `split` absolute positions
// (512 for the float32 and generic kernels, FS_ATTN_SPLIT (default 16384) for the MFMA kernels; fixed for the life
// of the process); chunk s covers keys
// [s*split, (s+1)*split). Each workgroup produces the softmax partial
// (running max m, sum l, unnormalised output acc) of its chunk, and attn_combine merges the chunks of
// a query in increasing chunk order. A query at position p only ever reads the chunks that hold
// keys <= p, and inside a chunk keys above p contribute exact zeros, so the output of a query does
// not depend on T, on the other rows of the batch, or on how far the other queries of its row reach:
// the verify pass and a 1-token decode at the same position give bit-identical outputs.
//
// Fast path (bf16, head_dim 64/128, block_size % 16 == 0, fs_kv_layout with slot-major keys and
// dim-major values): one wavefront per (chunk, batch row, kv head, 32-row query tile). The query
// tile is the (token, group-head) pairs of one KV head: rows = T * (n_heads / n_kv_heads).
//   S^T[key, row] = K . Q^T    v_mfma_f32_16x16x32_bf16, A = 16 keys x 32 dims straight from HBM
//   O^T[dim, row] += V^T . P^T v_mfma_f32_16x16x32_bf16, A = 16 dims x 4 keys of each tile of a pair
// With the transposed products every lane owns whole query rows (row = lane % 16), so the softmax
// statistics, the P operand and the O rescale stay in the lane's own registers.
// float32 in such a layout takes the same products on v_mfma_f32_16x16x4_f32; any other type or layout the
// scalar kernel.
#include <math.h>
#include <stdlib.h>

#include "common.h"

namespace {

constexpr int QTILE = 32;            // query rows per MFMA wave
constexpr int PLAN_THREADS = 256, PLAN_THREADS_PREFILL = 1024;   // (a prompt's positions are many loads)
constexpr int SPLIT_UNITS_MAX = 128;  // calls with at most this many units (half the CUs) may split each
// workspace: item count (bytes 0..255), the split units' arrival counters (one unsigned each), then
// the item list, the chunk partials and the split units' published partials
constexpr int64_t WS_COUNTERS = 256;
constexpr int64_t WS_HEADER = WS_COUNTERS + 4 * SPLIT_UNITS_MAX;
constexpr float LOG2E = 1.4426950408889634f;
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

struct AttnParams {
  const void* q;
  int64_t q_sb, q_st, q_sh;
  fs_kv_layout kv;
  const int32_t* table;
  int64_t table_stride;
  int32_t max_blocks;
  const int32_t* pos;
  int32_t B, T, H, G;                // G = n_heads / n_kv_heads
  float scale_log2;                  // scale * log2(e): scores are kept in the log2 domain
  float* ws_acc;                     // [B*T*H][nsplit][D]
  float* ws_ml;                      // [B*T*H][nsplit][2]
  int32_t nsplit;
  int32_t split;                     // keys per chunk: a multiple of 16
  struct AttnItem* items;            // MFMA path: the work list written by attn_plan_kernel
  int32_t* n_items;                  // its length
  // MFMA path: a query that sees one chunk only (position < split, or nsplit == 1) has its output
  // written by that chunk's workgroup, and attn_combine leaves it alone
  int32_t direct;
  void* out;
  int64_t o_sb, o_st, o_sh;
  // packed (varlen) rows: when set, row b's token t is token row_start[b] + t of q and out (strides
  // q_st/q_sh, o_st/o_sh; q_sb and o_sb unused), and only tokens t < row_start[b+1] - row_start[b]
  // exist: the others (positions -1) are neither read nor written
  const int32_t* row_start;
  // query tiles per plan item: 1 for the unit kernel, PF_WAVES for the prefill kernel (item.z is then
  // the index of a group of zgroup consecutive tiles, item.qmax the group's furthest query)
  int32_t zgroup;
  // split units (attn_unit_part_kernel): one arrival counter per unit (zero between launches) and
  // SPLIT_SLOTS published partials per unit
  unsigned* split_cnt;
  float* split_ws;
};

// Reductions over the four 16-lane groups of a wave (lanes l, l^16, l^32, l^48) with the gfx950
// row swaps: permlane16_swap of (x, x) yields {rows 0,0,2,2 ; rows 1,1,3,3} of x, permlane32_swap
// yields {lanes 0-31 twice ; lanes 32-63 twice}. Both steps are symmetric, so every lane ends with
// the same value, and the sum adds (g0 + g1) + (g2 + g3) in every lane.
// 2^x with the bare v_exp_f32 (no denormal-result scaling): the same value as exp2f wherever the
// result is a normal float.
FS_DEVICE float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// The maxima over the lanes l, l ^ 16, l ^ 32, l ^ 48 of x0 and of x1, in three swaps:
// permlane16_swap of (x0, x1) yields {x0 rows 0,1 ; x1 rows 0,1 ; x0 rows 2,3 ; x1 rows 2,3} as pairs,
// so one maximum leaves x0's groups 0/1 and 2/3 in rows 0 and 2 and x1's in rows 1 and 3;
// permlane32_swap and a maximum complete both (x0's in rows 0 and 2, x1's in rows 1 and 3), and a last
// permlane16_swap hands every lane both. Every lane gets max(max(g0, g1), max(g2, g3)). IEEE maximum
// (v_maximum3_f32, one instruction) rather than fmaxf, which needs its permuted operands canonicalised
// first; the two agree on every non-NaN input (the scores are finite or -inf) up to the sign of a
// zero maximum, which no result depends on.
FS_DEVICE void max_across_groups2(float x0, float x1, float& m0, float& m1) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x0), __float_as_uint(x1), false, false);
  const float y = __builtin_elementwise_maximum(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(y), __float_as_uint(y), false, false);
  const float z = __builtin_elementwise_maximum(__uint_as_float(b[0]), __uint_as_float(b[1]));
  auto c = __builtin_amdgcn_permlane16_swap(__float_as_uint(z), __float_as_uint(z), false, false);
  m0 = __uint_as_float(c[0]);
  m1 = __uint_as_float(c[1]);
}

FS_DEVICE float sum_across_groups(float x) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Four floats to bf16 (round to nearest even) with gfx950's packed conversion, as MFMA operand bits.
FS_DEVICE short4_t bf16_rne4(const float (&v)[4]) {
  typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2;
  typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
  const bf16x2 a = __builtin_convertvector((f32x2){v[0], v[1]}, bf16x2);
  const bf16x2 b = __builtin_convertvector((f32x2){v[2], v[3]}, bf16x2);
  const uint32_t ua = __builtin_bit_cast(uint32_t, a), ub = __builtin_bit_cast(uint32_t, b);
  return short4_t{(short)(ua & 0xffff), (short)(ua >> 16), (short)(ub & 0xffff), (short)(ub >> 16)};
}

FS_DEVICE int64_t row_index(const AttnParams& P, int b, int t, int h) { return ((int64_t)b * P.T + t) * P.H + h; }

FS_DEVICE bool token_exists(const AttnParams& P, int b, int t) {
  return P.row_start == nullptr || t < P.row_start[b + 1] - P.row_start[b];
}
FS_DEVICE int64_t q_offset(const AttnParams& P, int b, int t) {
  return P.row_start ? (int64_t)(P.row_start[b] + t) * P.q_st : (int64_t)b * P.q_sb + (int64_t)t * P.q_st;
}
FS_DEVICE int64_t o_offset(const AttnParams& P, int b, int t, int64_t o_sb, int64_t o_st) {
  return P.row_start ? (int64_t)(P.row_start[b] + t) * o_st : (int64_t)b * o_sb + (int64_t)t * o_st;
}

// ------------------------------------------------------------------------------------------------
// work plan: the (query tile, chunk) items that hold visible keys
// ------------------------------------------------------------------------------------------------
struct AttnItem {
  int32_t b, z, s, qmax;   // batch row, query tile, chunk, furthest query position of the tile
};

// furthest query position of query rows [row0, row0 + n) of batch row b (-1 if none)
FS_DEVICE int rows_qmax(const AttnParams& P, int b, int row0, int n) {
  n = min(n, P.T * P.G - row0);
  if (n <= 0) return -1;
  const int t0 = row0 / P.G, t1 = (row0 + n - 1) / P.G;
  const int* posb = P.pos + (int64_t)b * P.T;
  int q = -1;
  for (int t = t0; t <= t1; ++t) q = max(q, posb[t]);
  return q;
}
FS_DEVICE int tile_qmax(const AttnParams& P, int b, int z) { return rows_qmax(P, b, z * QTILE, QTILE); }

// Chunks a query tile reads. With direct outputs a tile of padding queries still gets chunk 0, whose
// workgroup writes their zero outputs.
FS_DEVICE int tile_chunks(const AttnParams& P, int qmax) {
  return qmax < 0 ? (P.direct ? 1 : 0) : min(qmax / P.split + 1, P.nsplit);
}

constexpr int UNIT_WAVES = 8;                  // waves per unit workgroup
constexpr int SPLIT_SLOTS = 7;                  // published partials per split unit, at most (four parts)
// floats of one published partial: m and l of the 32 rows, then acc as the LDS holds it (2 * D/16
// (half, dim tile) pairs, 64 lanes, 4 values)
constexpr int64_t split_slot_floats(int D) { return 2 * QTILE + (int64_t)QTILE * D; }
constexpr int MAX_SPLIT = 2 * 64 * 16 * UNIT_WAVES;   // keys per chunk, at most: a wave's pairs fit one
                                                       // lane each

// Inclusive scan of one int per thread over the workgroup: lane scans inside each wave, then the
// wave totals (two barriers). `tot` receives the workgroup's total.
template <int NTH>
FS_DEVICE int block_scan(int x, int* sh, int& tot) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) sh[wv] = x;
  __syncthreads();
  int before = 0;
  tot = 0;
#pragma unroll
  for (int k = 0; k < NTH / 64; ++k) {
    const int t = sh[k];
    if (k < wv) before += t;
    tot += t;
  }
  __syncthreads();
  return x + before;
}

// One workgroup lists every item: first the chunks that lie wholly below their tile's furthest query (the full
// chunks), tile by tile, then the last chunk of each tile, longest first. Workgroups start in list order, so
// the short last chunks even out the finish (longest-first list scheduling). A prefill's groups of zgroup
// tiles are listed the same way: row after row, which keeps one row's keys in an XCD's L2, prompts of 128-700
// tokens (8 rows) took 85 us instead of 70, of 817-4096 (5 rows) 452 instead of 440, and four of 2048 each
// 261 instead of 249. Eight threads look through a group's positions, 1,024 threads in all: a thread per group
// took 18 us for the 5 rows, now 8.
template <int NTH>
__global__ void __launch_bounds__(NTH) attn_plan_kernel(AttnParams P) {
  // the split units' arrival counters start at zero (each unit's last part leaves its counter zero,
  // so calls that reuse this plan find them so too)
  for (int i = threadIdx.x; i < SPLIT_UNITS_MAX; i += NTH) st_ag(P.split_cnt + i, 0u);
  __shared__ int sh[NTH / 64];
  __shared__ int cursor[MAX_SPLIT / 16 + 1];   // last chunks by length in 16-key tiles
  const int tid = threadIdx.x;
  const int qtiles = ((P.T * P.G + QTILE - 1) / QTILE + P.zgroup - 1) / P.zgroup;   // tiles, or groups of tiles, per row
  const int U = P.B * qtiles;
  // A group's furthest query: eight lanes look through its positions. Kept where the attention kernels put
  // their partials later (at least one per row of every tile).
  int* group_qmax = reinterpret_cast<int*>(P.ws_acc);
  if (P.zgroup > 1) {
    for (int u0 = 0; u0 < U; u0 += NTH / 8) {
      const int u = u0 + (tid >> 3);
      int q = -1;
      if (u < U) {
        const int b = u / qtiles, row0 = (u - b * qtiles) * P.zgroup * QTILE;
        const int n = min(P.zgroup * QTILE, P.T * P.G - row0);
        const int* posb = P.pos + (int64_t)b * P.T;
        const int t1 = (row0 + n - 1) / P.G;
#pragma unroll 8
        for (int t = row0 / P.G + (tid & 7); t <= t1; t += 8) q = max(q, posb[t]);
      }
#pragma unroll
      for (int o = 1; o < 8; o <<= 1) q = max(q, __shfl_xor(q, o, 64));
      if (u < U && (tid & 7) == 0) group_qmax[u] = q;
    }
    __syncthreads();
  }
  auto unit_qmax = [&](int u) { return P.zgroup > 1 ? group_qmax[u] : tile_qmax(P, u / qtiles, u % qtiles); };
  const int nlen = P.split / 16;   // a last chunk holds 1..nlen tiles (an empty one counts as 1)
  for (int i = tid; i <= nlen; i += NTH) cursor[i] = 0;
  // the thread's first tile (u = tid) stays in registers; tiles past the first NTH are
  // recomputed when needed
  int qm0 = -1, nch0 = 0;
  if (tid < U) {
    qm0 = unit_qmax(tid);
    nch0 = tile_chunks(P, qm0);
  }
  auto tile = [&](int u, int& qm, int& nch) {
    if (u == tid) {
      qm = qm0;
      nch = nch0;
    } else {
      qm = unit_qmax(u);
      nch = tile_chunks(P, qm);
    }
  };
  auto last_tiles = [&](int qm, int nch) { return max(min((qm + 1 - (nch - 1) * P.split + 15) >> 4, nlen), 1); };
  __syncthreads();
  int nf = 0;
  for (int u = tid; u < U; u += NTH) {   // full chunks, and a histogram of the last chunks' lengths
    int qm, nch;
    tile(u, qm, nch);
    nf += max(nch - 1, 0);
    if (nch > 0) atomicAdd(&cursor[last_tiles(qm, nch)], 1);
  }
  int n_full;
  block_scan<NTH>(nf, sh, n_full);
  {   // exclusive scan from the longest length down: cursor[len] = first slot of that length
    constexpr int PER = (MAX_SPLIT / 16 + NTH - 1) / NTH;
    int c[PER], loc = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k) {   // thread tid owns lengths nlen - PER*tid - k
      const int len = nlen - PER * tid - k;
      c[k] = len >= 1 ? cursor[len] : 0;
      loc += c[k];
    }
    int n_last;
    int run = n_full + block_scan<NTH>(loc, sh, n_last) - loc;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int len = nlen - PER * tid - k;
      if (len >= 1) cursor[len] = run;
      run += c[k];
    }
    if (tid == 0) P.n_items[0] = n_full + n_last;
    __syncthreads();
  }
  int base_full = 0;
  for (int u0 = 0; u0 < U; u0 += NTH) {
    const int u = u0 + tid;
    int qm = -1, nch = 0;
    if (u < U) tile(u, qm, nch);
    const int b = u / qtiles, z = u - b * qtiles;
    const int f = max(nch - 1, 0);
    int n_round;
    const int ef = base_full + block_scan<NTH>(f, sh, n_round) - f;
    for (int c = 0; c < f; ++c) P.items[ef + c] = AttnItem{b, z, c, qm};
    // the slot order inside one length is whatever the atomics give: it only changes which
    // workgroup runs an item, never what the item computes
    if (nch > 0) P.items[atomicAdd(&cursor[last_tiles(qm, nch)], 1)] = AttnItem{b, z, nch - 1, qm};
    base_full += n_round;
  }
}

// ------------------------------------------------------------------------------------------------
// MFMA kernel (bf16)
// ------------------------------------------------------------------------------------------------
// ------------------------------------------------------------------------------------------------
// unit kernel: one workgroup of UNIT_WAVES waves per (plan item, KV head)
// ------------------------------------------------------------------------------------------------
// The item's keys [kbeg, kend) are cut into pairs of 16-key tiles; wave w takes pairs w, w + UNIT_WAVES, ...
// in increasing order and keeps its own softmax partial, and the waves' partials are merged through
// LDS in wave order. Which pairs a wave sees, and in what order, depends only on absolute key
// positions, and a pair wholly above a query's position leaves that query's partial exactly as it
// was; a query's result therefore does not depend on the other queries of its tile.

// Smallest position over the rows r < nrows of a wave's 32-row tile (-1 if nrows <= 0); the rows of
// lane l16 are l16 and 16 + l16, whose positions are rpos[0] and rpos[1].
FS_DEVICE int rows_min_pos(const int (&rpos)[2], int nrows) {
  if (nrows <= 0) return -1;
  const int l16 = threadIdx.x & 15;
  int v = min(l16 < nrows ? rpos[0] : 0x7fffffff, 16 + l16 < nrows ? rpos[1] : 0x7fffffff);
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) v = min(v, __shfl_xor(v, o, 64));
  return __builtin_amdgcn_readfirstlane(v);
}

constexpr float REF_SLACK = 8.f;   // log2 units a pair's maximum may exceed the reference by

// A pair of 16-key tiles (32 keys from j0 on) into a wave's online-softmax partial of up to 32 query rows (two
// 16-row halves; TWO: the second too, whatever rows of it exist), in two steps: the scores S^T = K.Q^T, tile
// by tile, and pair_step. The pair is one k = 32 product O^T += V^T.P^T: in the operands lane group g's eight k
// slots are keys 4g .. 4g+3 of the first tile, then of the second, so its probabilities (the S^T accumulators)
// and its values (8 bytes per dim and tile) lie in the lane as the product wants them. One product of 32 keys
// costs what one of 16 does, and the softmax's reductions and branches are paid once per 32 keys.
//
// ok: whether each tile is there (a mapped block, a tile the chunk has); fresh: acc is all zeros; rpos: the
// positions of the lane's two rows (-1: no query), rmin the smallest position over all 32 rows (-1 if any row
// is missing), qmax the furthest. A key above a row's position gets score -inf; values that must not reach the
// product (an absent tile, or a key past qmax, which may never have been written) are zeroed.
//
// The partial is (m, l, acc) with p = 2^(s - m): m is a reference maximum that moves only when a pair's
// maximum exceeds it by more than 8 (then to that maximum, and acc and l are rescaled), so p <= 2^8 and the
// rescale is rare once a row has seen a few pairs. A pair wholly above a row leaves that row's partial
// exactly as it was (m unchanged, alpha = 1, p = 0), and the part of a pair above it counts as exact zeros.
// A pair whose keys every row sees takes a path without the per-key masks; its arithmetic is the same. Every
// kernel that builds a partial calls these functions, so a row's partial does not depend on which kernel
// ran it.
template <int D, bool TWO>
FS_DEVICE void tile_scores(const bf16x8_t (&kf)[D / 32], const bf16x8_t (&qf)[2][D / 32], float4_t (&sc)[2]) {
  constexpr int KS = D / 32;
  sc[0] = float4_t{0.f, 0.f, 0.f, 0.f};
  sc[1] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    sc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks], qf[0][ks], sc[0], 0, 0, 0);
    if (TWO) sc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks], qf[1][ks], sc[1], 0, 0, 0);
  }
}

// Queries whose scale is negative are negated as they are loaded, and zeroed where it is 0 (both exact), so
// scores are scaled by a positive number: a maximum commutes with it, and a masked score stays -inf.
FS_DEVICE bf16x8_t signed_query(bf16x8_t q, float scale_log2) {
  const unsigned flip = scale_log2 < 0.f ? 0x80008000u : 0u, keep = scale_log2 == 0.f ? 0u : ~0u;
  return __builtin_bit_cast(bf16x8_t, (__builtin_bit_cast(u32x4, q) ^ flip) & keep);
}
FS_DEVICE float positive_scale(float scale_log2) { return scale_log2 == 0.f ? 1.f : fabsf(scale_log2); }

// The softmax step of one pair for the lane's two rows: the references, p = 2^(s - m) as bf16 operands, and
// l <- l * alpha + (the lane's sum of p), alpha = 2^(m_old - m_new) for a row that moved, else 1. Returns
// whether any row of the wave moved; alpha is for the caller's rescale of acc.
template <bool TWO>
FS_DEVICE bool pair_probs(const float (&sc)[2][2][4], float scale, float (&m_run)[2], float (&l_run)[2], float (&alpha)[2],
                          bf16x8_t (&pf)[2]) {
  constexpr int NT = TWO ? 2 : 1;
  float x[2];   // the lane's largest score of each row, unscaled
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    float a[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) a[e] = __builtin_elementwise_maximum(sc[0][nt][e], sc[1][nt][e]);
    x[nt] = __builtin_elementwise_maximum(__builtin_elementwise_maximum(a[0], a[1]), __builtin_elementwise_maximum(a[2], a[3]));
  }
  auto probs = [&](int nt, float m) {   // the lane's p of a row, into pf; returns their sum
    const float ref = m == -INFINITY ? 0.f : m;   // (a row that has seen nothing yet: every p is 0)
    float pv[2][4];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) pv[u][e] = fast_exp2(fmaf(sc[u][nt][e], scale, -ref));
    struct Halves { short4_t a, b; } h = {bf16_rne4(pv[0]), bf16_rne4(pv[1])};
    pf[nt] = __builtin_bit_cast(bf16x8_t, h);
    return ((pv[0][0] + pv[0][1]) + (pv[0][2] + pv[0][3])) + ((pv[1][0] + pv[1][1]) + (pv[1][2] + pv[1][3]));
  };
  // A row's maximum exceeds m + REF_SLACK exactly when one of its four lane groups' maxima does. When no
  // lane's does, no row moves (m_new = m, alpha = 1), and the reduction across the lane groups is skipped.
    const bool moved = __any(x[0] * scale > m_run[0] + REF_SLACK || (TWO && x[1] * scale > m_run[1] + REF_SLACK));
  if (moved) {
    float tmax[2];
    max_across_groups2(x[0], x[TWO ? 1 : 0], tmax[0], tmax[1]);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const float t = tmax[nt] * scale;
      const bool mv = t > m_run[nt] + REF_SLACK;   // (false for a row that sees nothing here)
      const float m_new = mv ? t : m_run[nt];
      alpha[nt] = mv ? fast_exp2(m_run[nt] - m_new) : 1.f;
      l_run[nt] *= alpha[nt];
      m_run[nt] = m_new;
    }
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) l_run[nt] += probs(nt, m_run[nt]);
  return moved;
}

// SEEN: every row sees every key of the pair (the caller knows; j0, ok and qmax are not looked at).
// value(mt): the pair's values of dims 16 mt .. as the product's operand.
template <int D, bool TWO, bool SEEN = false, class Value>
FS_DEVICE void pair_step(const float4_t (&sc)[2][2], Value value, int j0, const bool (&ok)[2], bool fresh, int qmax,
                         const int (&rpos)[2], int rmin, float scale, float4_t (&acc)[D / 16][2], float (&m_run)[2],
                         float (&l_run)[2]) {
  constexpr int MT = D / 16;
  constexpr int NT = TWO ? 2 : 1;
  const int g = (threadIdx.x & 63) >> 4;
  const bool full = SEEN || (ok[0] && ok[1] && j0 + 31 <= rmin);   // wave-uniform
  float s[2][2][4];   // (one by one: masked in place)
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[u][nt][e] = sc[u][nt][e];
  if (!full) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int last = (ok[u] ? rpos[nt] : -1) - j0 - 16 * u - 4 * g;   // the row sees the lane's keys e <= last
#pragma unroll
        for (int e = 0; e < 4; ++e) s[u][nt][e] = e <= last ? s[u][nt][e] : -INFINITY;
      }
  }
  bf16x8_t pf[2];
  float alpha[2];
  const bool moved = pair_probs<TWO>(s, scale, m_run, l_run, alpha, pf);
  if (moved && !fresh) {   // (alpha = 1 for every row that did not: skipping the rescale is exact)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[mt][nt][e] *= alpha[nt];
  }
  // zero bits for the values that must not reach the product (ands behind a branch that every group of dims
  // takes or skips: a second copy of the products took 50 registers more)
  const bool masked = !full && !(ok[0] && ok[1] && j0 + 31 <= qmax);
  u32x4 keep = {~0u, ~0u, ~0u, ~0u};
  if (masked) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int last = (ok[c >> 1] ? qmax : -1) - j0 - 16 * (c >> 1) - 4 * g, e = 2 * (c & 1);   // keys e, e + 1
      keep[c] = (e <= last ? 0xffffu : 0u) | (e < last ? 0xffff0000u : 0u);
    }
  }
  // two groups of dims at a time with the next two's values on their way (read sooner, they would need
  // registers of their own)
  __builtin_amdgcn_sched_barrier(0);
  bf16x8_t v[2][2];
  v[0][0] = value(0);
  v[0][1] = value(1);
#pragma unroll
  for (int mt = 0; mt < MT; mt += 2) {
    bf16x8_t(&now)[2] = v[mt / 2 & 1], (&next)[2] = v[(mt / 2 & 1) ^ 1];
    if (mt + 2 < MT) {
      next[0] = value(mt + 2);
      next[1] = value(mt + 3);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (masked) {
#pragma unroll
      for (int i = 0; i < 2; ++i) now[i] = __builtin_bit_cast(bf16x8_t, __builtin_bit_cast(u32x4, now[i]) & keep);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      acc[mt + i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(now[i], pf[0], acc[mt + i][0], 0, 0, 0);
      if (TWO) acc[mt + i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(now[i], pf[1], acc[mt + i][1], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The operand of a pair's values: the first tile's four keys of the lane, then the second's.
FS_DEVICE bf16x8_t pair_value(short4_t a, short4_t b) {
  return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// A chunk's result for one query row is its 8 partials (class v: pairs p with p % 8 == v) folded in
// increasing v: (M, L, O) <- (max(M, m), L*2^(M-M') + l*2^(m-M'), O*2^(M-M') + a*2^(m-M')). An empty
// partial (m = -inf: no visible key) leaves the state as it is; the first non-empty one gets weight 1
// and the empty state weight 2^-inf = 0. fold_weights returns false for an empty partial.
FS_DEVICE bool fold_weights(float M, float m, float& Mn, float& cM, float& cm) {
  if (m == -INFINITY) return false;
  Mn = fmaxf(M, m);
  cM = fast_exp2(M - Mn);
  cm = fast_exp2(m - Mn);
  return true;
}
FS_DEVICE float fold_value(float x, float cM, float y, float cm) { return fmaf(x, cM, y * cm); }

// Pairs of tiles a wave holds in registers. One (a key buffer is refilled as soon as its scores are formed, a
// value buffer after its product, so about two tiles are in flight) keeps the unit kernel's 2,048 waves at what
// HBM delivers: with two, where the registers allow them, 64 rows of 1000-2000 keys take 75 us instead of 68.
// Two waves on a CU (four parts) want two (3 rows of 8000-30000 keys: 68 -> 64 us); four want one (16 rows of
// 128-1280 keys, 64 dims: 12.3 against 13.4). The last pair is consumed with nothing left to load: prefetching
// past the end cost 64 rows of 1000-2000 keys 7 us.
constexpr int UNIT_PAIRS = 1;
constexpr int part_pairs(int parts) { return parts == 4 ? 2 : 1; }

// TWO: the tile has a second 16-row half. NP: pair buffers in registers.
template <int D, int BSZ, bool TWO, int NP>
__device__ __attribute__((always_inline)) inline void attn_wave_tiles(const AttnParams& P, int b, int kbeg, int kend,
                                                                      int qmax, int row0, int nrows,
                                                                      const int (&rpos)[2], int hkv, int w,
                                                                      float4_t (*red_acc)[64], float* red_m,
                                                                      float* red_l) {
  constexpr int KS = D / 32;   // k-steps of the QK^T product
  constexpr int MT = D / 16;   // 16-dim tiles of the PV product
  constexpr int NT = TWO ? 2 : 1;
  const int lane = threadIdx.x & 63;
  const int l16 = lane & 15, g = lane >> 4;
  const int ntiles = (kend - kbeg + 15) >> 4;
  const int npairs = (ntiles + 1) >> 1;
  const int np_w = npairs > w ? (npairs - w + UNIT_WAVES - 1) / UNIT_WAVES : 0;   // <= 64 pairs
  auto pair_key = [&](int i) { return kbeg + 32 * (w + UNIT_WAVES * i); };   // the first key of the wave's pair i
  const int BS = BSZ ? BSZ : P.kv.block_size;
  const int64_t v_dim = BSZ ? BSZ : P.kv.v_dim;   // == block_size (dim-major values)

  // lane i: where the tiles of the wave's pair i start in the pool, in bytes from the head's base (64 bits: the
  // block stride is the caller's, and a pool that keeps every layer of a block together spans more than 64 GiB;
  // an unmapped block reads block 0 and is masked, a second tile that the chunk lacks reads the first), and
  // which of them are there
  typedef uint16_t u16;
  const u16* kpool = reinterpret_cast<const u16*>(P.kv.k) + (int64_t)hkv * P.kv.k_head;
  const u16* vpool = reinterpret_cast<const u16*>(P.kv.v) + (int64_t)hkv * P.kv.v_head;
  const int64_t k_slot = P.kv.k_slot;
  uint64_t k_at[2], v_at[2];
  uint64_t mapped[2];
  bool all_mapped = true;
  {
    int phys[2] = {-1, -1}, slot0[2] = {0, 0};
    bool exists[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int j0 = pair_key(lane) + 16 * u, blk = j0 / BS;
      exists[u] = lane < np_w && j0 < kend;
      if (exists[u]) {
        slot0[u] = j0 - blk * BS;
        if (blk < P.max_blocks) phys[u] = P.table[(int64_t)b * P.table_stride + blk];
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bool ok = phys[u] >= 0 && phys[u] < P.kv.num_blocks;
      mapped[u] = __ballot(ok);
      all_mapped &= mapped[u] == __ballot(exists[u]);
      const int64_t pb = ok ? phys[u] : 0;
      k_at[u] = (uint64_t)(2 * (pb * P.kv.k_block + slot0[u] * k_slot));
      v_at[u] = (uint64_t)(2 * (pb * P.kv.v_block + slot0[u]));
    }
    if (!exists[1]) {
      k_at[1] = k_at[0];
      v_at[1] = v_at[0];
    }
  }

  // Q fragments (B operand of S^T): Q[row][32*ks + 8*g .. +8]. Loaded before the first tiles: vmcnt counts in
  // order, so a wait for queries loaded after them would wait for every tile in flight, at each turn of
  // the loop (the compiler merges the first turn's state into all).
  const u16* qbase = reinterpret_cast<const u16*>(P.q);
  bf16x8_t qf[2][KS];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int r = row0 + 16 * nt + l16;
    const bool in_tile = (16 * nt + l16) < nrows;
    const bool ok = in_tile && token_exists(P, b, r / P.G);
    const int t = ok ? r / P.G : 0;
    const int h = hkv * P.G + (ok ? r - (r / P.G) * P.G : 0);
    const u16* qr = qbase + q_offset(P, b, t) + (int64_t)h * P.q_sh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ok)
        qf[nt][ks] = signed_query(*reinterpret_cast<const bf16x8_t*>(qr + 32 * ks + 8 * g), P.scale_log2);
      else
        qf[nt][ks] = bf16x8_t{};
    }
  }

  // NP pair buffers: a pair's keys are loaded once the scores that read the buffer are formed, its values once
  // the product is. Every load of a loop is unconditional and the loops have one back edge each, so that each wait before a product counts exactly the loads issued
  // after its operand.
  static_assert(NP * 2 * (KS + MT) < 64, "vmcnt counts every load in flight");
  bf16x8_t kb[NP][2][KS];
  short4_t vb[NP][2][MT];
  // a lane's byte offsets inside a tile; a tile adds its wave-uniform base. Key (slot, dims 8c .. 8c+7) is at
  // slot * k_slot + c * kgs: slot-major (k_slot = D, kgs = 8) or grouped (k_slot = 8, kgs = 8 * block_size:
  // one load of a tile's 32 dims is a contiguous 1 KB)
  const int64_t kgs = key_group_stride(P.kv);
  uint32_t k_lane[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) k_lane[ks] = (uint32_t)(2 * (l16 * k_slot + (g + 4 * ks) * kgs));
  const uint32_t v_lane = (uint32_t)(2 * (l16 * v_dim + 4 * g));
  // where a tile of the wave's pair i starts (a wave without pairs reads block 0 and consumes nothing)
  auto tile_at = [&](const u16* pool, uint64_t at, int i) {
    const int l = max(min(i, np_w - 1), 0);
    const uint32_t lo = __builtin_amdgcn_readlane((int)at, l), hi = __builtin_amdgcn_readlane((int)(at >> 32), l);
    uint64_t t = reinterpret_cast<uint64_t>(pool) + ((uint64_t)hi << 32 | lo);
    asm("" : "+s"(t));   // a scalar base and 32-bit lane offsets: no 64-bit vector adds per load
    return (__attribute__((address_space(1))) const char*)t;
  };
  typedef __attribute__((address_space(1))) const bf16x8_t GKey;
  typedef __attribute__((address_space(1))) const short4_t GVal;
  auto load_keys = [&](int pair, bf16x8_t (&kd)[2][KS]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      auto kt = tile_at(kpool, k_at[u], pair);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)   // read once per launch: nontemporal
        kd[u][ks] = __builtin_nontemporal_load((GKey*)(kt + k_lane[ks]));
    }
  };
  auto load_values = [&](int pair, short4_t (&vd)[2][MT]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      auto vt = tile_at(vpool, v_at[u], pair);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        vd[u][mt] = __builtin_nontemporal_load((GVal*)(vt + (v_lane + (uint32_t)(32 * mt * v_dim))));
    }
  };
#pragma unroll
  for (int j = 0; j < NP; ++j) {   // in the order that the loops' waits count
    load_keys(j, kb[j]);
    __builtin_amdgcn_sched_barrier(0);
    load_values(j, vb[j]);
    __builtin_amdgcn_sched_barrier(0);
  }

  float4_t acc[MT][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    acc[mt][0] = float4_t{0.f, 0.f, 0.f, 0.f};
    acc[mt][1] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
  float m_run[2] = {-INFINITY, -INFINITY};
  float l_run[2] = {0.f, 0.f};

  // The wave's first n_full pairs have every key mapped and seen by every row: they take a loop without masks
  // or lookups. The rest (the pairs around the rows' own positions, or all of them where a row is padding or
  // a block unmapped) follow; a pair past the wave's last is two absent tiles.
  const int rmin = rows_min_pos(rpos, nrows);
  const int n_seen = rmin + 1 > kbeg ? min((rmin + 1 - kbeg) >> 5, ntiles >> 1) : 0;   // pairs all rows see
  const int n_full = all_mapped && n_seen > w ? (n_seen - w + UNIT_WAVES - 1) / UNIT_WAVES : 0;
  const float scale = positive_scale(P.scale_log2);
  auto there = [&](int i, int u) { return i < np_w && ((mapped[u] >> (i & 63)) & 1) != 0; };
  int i = 0;
  auto refill_keys = [&](int j) {   // (moved up, they would need registers of their own)
    __builtin_amdgcn_sched_barrier(0);
    load_keys(i + j + NP, kb[j]);
  };
  auto refill_values = [&](int j) {
    __builtin_amdgcn_sched_barrier(0);
    load_values(i + j + NP, vb[j]);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto value = [&](int j) { return [&, j](int mt) { return pair_value(vb[j][0][mt], vb[j][1][mt]); }; };
  for (; i + NP <= n_full && i + NP < np_w; i += NP) {
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      float4_t sc[2][2];
      tile_scores<D, TWO>(kb[j][0], qf, sc[0]);
      tile_scores<D, TWO>(kb[j][1], qf, sc[1]);
      refill_keys(j);
      pair_step<D, TWO, true>(sc, value(j), 0, {true, true}, i + j == 0, 0, rpos, rmin, scale, acc, m_run, l_run);
      refill_values(j);
    }
  }
  auto masked_pair = [&](int j, bool refill) {
    const int p = i + j;
    float4_t sc[2][2];
    tile_scores<D, TWO>(kb[j][0], qf, sc[0]);
    tile_scores<D, TWO>(kb[j][1], qf, sc[1]);
    if (refill) refill_keys(j);
    pair_step<D, TWO>(sc, value(j), pair_key(p), {there(p, 0), there(p, 1)}, p == 0, qmax, rpos, rmin, scale, acc, m_run,
                      l_run);
    if (refill) refill_values(j);
  };
  for (; i + NP < np_w; i += NP) {
#pragma unroll
    for (int j = 0; j < NP; ++j) masked_pair(j, true);
  }
#pragma unroll
  for (int j = 0; j < NP; ++j) masked_pair(j, false);   // the last pairs, or absent ones: nothing is left to load
  // this wave's partial to LDS: acc by (query half, dim tile, lane), m and l by query row
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red_acc[nt * MT + mt][lane] = acc[mt][nt];
    const float lsum = sum_across_groups(l_run[nt]);
    if (g == 0) {
      red_m[16 * nt + l16] = m_run[nt];
      red_l[16 * nt + l16] = lsum;
    }
  }
}

// Row `rr` of the query rows (token rr / G, head hkv*G + rr % G), dims 16*(mt + i) + 4g .. +4 for i < N, from its
// folded chunk-s state (M, L, o): a query that sees one chunk only is finished here (a padding query,
// position < 0, gets zeros from chunk 0); any other query gets this chunk's partial for attn_combine
// if the chunk holds keys it sees.
template <int D, int N>
FS_DEVICE void attn_emit(const AttnParams& P, int b, int s, int kbeg, int hkv, int rr, int rp, int mt, float M,
                         float L, const float4_t (&o)[N]) {
  const int lane = threadIdx.x & 63, g = lane >> 4;
  const bool direct = P.direct && (rp < P.split || P.nsplit == 1);
  if (direct ? s != 0 : rp < kbeg) return;
  const int t = rr / P.G, h = hkv * P.G + (rr - t * P.G);
  if (direct) {
    if (!token_exists(P, b, t)) return;
    // o / L, rounded to bf16. o times L's reciprocal, which the row's outputs share, is within 2 ulps of it, and rounds
    // to the same bf16 unless a tie is that near: then the wave divides (one time in thirty for N = 1, in nine for
    // 4). Prompts of 817-4096 tokens: every output divided 402 us, products with N = 1 397, with N = 4 362.
    const float inv = 1.f / L;
    float f[N][4];
    uint16_t near = 0xffff;   // the products' smallest distance above four ulps below a tie
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        f[i][c] = o[i][c] * inv;
        near = min(near, (uint16_t)((uint16_t)__float_as_uint(f[i][c]) - 0x7ffc));
      }
    if (__any(near <= 8 || !(L > 0.f))) {
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) f[i][c] = L > 0.f ? o[i][c] / L : 0.f;
    }
    uint16_t* orow = reinterpret_cast<uint16_t*>(P.out) + o_offset(P, b, t, P.o_sb, P.o_st) + (int64_t)h * P.o_sh;
#pragma unroll
    for (int i = 0; i < N; ++i) *reinterpret_cast<short4_t*>(orow + 16 * (mt + i) + 4 * g) = bf16_rne4(f[i]);
    return;
  }
  const int64_t R = row_index(P, b, t, h);
#pragma unroll
  for (int i = 0; i < N; ++i)
    *reinterpret_cast<float4_t*>(P.ws_acc + (R * P.nsplit + s) * D + 16 * (mt + i) + 4 * g) = o[i];
  if (mt == 0 && g == 0) {
    float* pm = P.ws_ml + (R * P.nsplit + s) * 2;
    pm[0] = M;
    pm[1] = L;
  }
}

template <int D, int BSZ, bool TWO>
__global__ void __launch_bounds__(64 * UNIT_WAVES) __attribute__((amdgpu_waves_per_eu(2)))
attn_unit_kernel(AttnParams P) {
  constexpr int MT = D / 16, NG = (TWO ? 2 : 1) * MT;
  __shared__ float4_t red_acc[UNIT_WAVES][NG][64];
  __shared__ float red_m[UNIT_WAVES][QTILE], red_l[UNIT_WAVES][QTILE];
  const int nkv = P.kv.n_kv_heads;
  const int64_t e_idx = blockIdx.x / nkv;
  const int hkv = (int)(blockIdx.x - e_idx * nkv);
  if (e_idx >= P.n_items[0]) return;   // uniform over the workgroup
  typedef __attribute__((address_space(4))) const AttnItem ConstItem;   // read-only: scalar loads
  ConstItem* ep = (ConstItem*)(uintptr_t)(P.items + e_idx);
  const int b = ep->b, z = ep->z, s = ep->s, qmax = ep->qmax;
  const int lane = threadIdx.x & 63, l16 = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // wave-uniform, in a scalar register
  const int row0 = z * QTILE;
  const int nrows = min(QTILE, P.T * P.G - row0);
  const int* posb = P.pos + (int64_t)b * P.T;
  int rpos[2];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int r = 16 * nt + l16;
    rpos[nt] = (r < nrows) ? posb[(row0 + r) / P.G] : -1;
  }
  const int kbeg = s * P.split;
  const int kend = min(kbeg + P.split, qmax + 1);

  attn_wave_tiles<D, BSZ, TWO, UNIT_PAIRS>(P, b, kbeg, kend, qmax, row0, nrows, rpos, hkv, w, red_acc[w], red_m[w], red_l[w]);
  __syncthreads();

  // fold the waves' partials in wave order; wave w takes the (query half, 16-dim tile) pairs w,
  // w + UNIT_WAVES, ...
  for (int gi = w; gi < NG; gi += UNIT_WAVES) {
    const int nt = gi / MT, mt = gi - nt * MT;
    const int r = 16 * nt + l16;
    if (r >= nrows) continue;
    float M = -INFINITY, L = 0.f;
    float4_t o = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < UNIT_WAVES; ++v) {
      float Mn, cM, cm;
      if (!fold_weights(M, red_m[v][r], Mn, cM, cm)) continue;
      L = fold_value(L, cM, red_l[v][r], cm);
      const float4_t a = red_acc[v][gi][lane];
#pragma unroll
      for (int c = 0; c < 4; ++c) o[c] = fold_value(o[c], cM, a[c], cm);
      M = Mn;
    }
    attn_emit<D, 1>(P, b, s, kbeg, hkv, row0 + r, rpos[nt], mt, M, L, {o});
  }
}

// Device-coherent accesses to a split unit's published partials: buffer loads and stores with the sc1
// cache policy (coherent at device scope, the encoding agent-scope atomics get), four floats at a time
// where the data allows. Being plain accesses, the compiler issues a wave's loads together; the
// barrier and the arrival count order them against the other parts' stores.
constexpr int CPOL_SC1 = 16;
FS_DEVICE __amdgpu_buffer_rsrc_t slot_rsrc(float* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(base, (short)0, bytes, 0x00020000);
}
FS_DEVICE void st4_dev(__amdgpu_buffer_rsrc_t r, int off, float4_t v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, CPOL_SC1);
}
FS_DEVICE void st1_dev(__amdgpu_buffer_rsrc_t r, int off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, CPOL_SC1);
}
FS_DEVICE float4_t ld4_dev(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, CPOL_SC1));
}
FS_DEVICE float ld1_dev(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, CPOL_SC1));
}

// A unit split over PARTS workgroups: workgroup PARTS * u + part (UNIT_WAVES / PARTS waves) builds classes
// WPP * part + w of unit u, each with the unit kernel's attn_wave_tiles, so that a call with few units keeps
// more CUs streaming (a CU has about 40 KB of misses outstanding, 45 GB/s from HBM, however deep its waves
// prefetch). A row's result is the unit kernel's fold over classes 0..7 in increasing order: part 0 publishes
// its classes folded, (M, L, O), every other part its class partials one by one, and the part that arrives
// last folds them in order and emits the rows. The arrival is counted (an agent-scope atomic), never awaited;
// the published values cross XCDs through device-coherent accesses.
template <int D, int BSZ, bool TWO, int PARTS>
__global__ void __launch_bounds__(64 * UNIT_WAVES / PARTS) __attribute__((amdgpu_waves_per_eu(1)))
attn_unit_part_kernel(AttnParams P) {
  constexpr int WPP = UNIT_WAVES / PARTS;
  constexpr int MT = D / 16, GI = (TWO ? 2 : 1) * MT;
  constexpr int NSLOT = 1 + UNIT_WAVES - WPP;   // part 0's prefix, then classes WPP .. 7
  constexpr int64_t SLOT = split_slot_floats(D);
  static_assert(NSLOT <= SPLIT_SLOTS, "the workspace holds the published partials");
  __shared__ float4_t red_acc[WPP][GI][64];
  __shared__ float red_m[WPP][QTILE], red_l[WPP][QTILE];
  __shared__ int sh_last;
  const int nkv = P.kv.n_kv_heads;
  const int64_t unit = blockIdx.x / PARTS;
  const int part = blockIdx.x % PARTS;
  const int64_t e_idx = unit / nkv;
  const int hkv = (int)(unit - e_idx * nkv);
  if (e_idx >= P.n_items[0]) return;   // uniform over the workgroup (and over a unit's parts)
  typedef __attribute__((address_space(4))) const AttnItem ConstItem;
  ConstItem* ep = (ConstItem*)(uintptr_t)(P.items + e_idx);
  const int b = ep->b, z = ep->z, s = ep->s, qmax = ep->qmax;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = z * QTILE;
  const int nrows = min(QTILE, P.T * P.G - row0);
  const int* posb = P.pos + (int64_t)b * P.T;
  int rpos[2];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int r = 16 * nt + l16;
    rpos[nt] = (r < nrows) ? posb[(row0 + r) / P.G] : -1;
  }
  const int kbeg = s * P.split;
  const int kend = min(kbeg + P.split, qmax + 1);

  attn_wave_tiles<D, BSZ, TWO, part_pairs(PARTS)>(P, b, kbeg, kend, qmax, row0, nrows, rpos, hkv, WPP * part + w,
                                                         red_acc[w], red_m[w], red_l[w]);
  __syncthreads();

  // this unit's published partials, SLOT floats each
  const __amdgpu_buffer_rsrc_t scr =
      slot_rsrc(P.split_ws + unit * SPLIT_SLOTS * SLOT, (int)(SPLIT_SLOTS * SLOT * sizeof(float)));
  auto m_at = [&](int slot, int r) { return (int)((slot * SLOT + r) * sizeof(float)); };
  auto l_at = [&](int slot, int r) { return (int)((slot * SLOT + QTILE + r) * sizeof(float)); };
  auto acc_at = [&](int slot, int gi) { return (int)((slot * SLOT + 2 * QTILE + (gi * 64 + lane) * 4) * sizeof(float)); };
  if (part == 0) {
    for (int gi = w; gi < GI; gi += WPP) {
      const int nt = gi / MT, mt = gi - nt * MT, r = 16 * nt + l16;
      float M = -INFINITY, L = 0.f;
      float4_t o = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int v = 0; v < WPP; ++v) {
        float Mn, cM, cm;
        if (!fold_weights(M, red_m[v][r], Mn, cM, cm)) continue;
        L = fold_value(L, cM, red_l[v][r], cm);
        const float4_t a = red_acc[v][gi][lane];
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] = fold_value(o[c], cM, a[c], cm);
        M = Mn;
      }
      st4_dev(scr, acc_at(0, gi), o);
      if (mt == 0 && g == 0) {
        st1_dev(scr, m_at(0, r), M);
        st1_dev(scr, l_at(0, r), L);
      }
    }
  } else {   // this wave's class partial, as the unit kernel's LDS holds it
    const int slot = 1 + WPP * (part - 1) + w;
#pragma unroll
    for (int gi = 0; gi < GI; ++gi) st4_dev(scr, acc_at(slot, gi), red_acc[w][gi][lane]);
    if (lane < (TWO ? QTILE : 16)) {
      st1_dev(scr, m_at(slot, lane), red_m[w][lane]);
      st1_dev(scr, l_at(slot, lane), red_l[w][lane]);
    }
  }
  stores_done();
  __syncthreads();   // every wave's published values have completed
  if (threadIdx.x == 0) sh_last = count_in(P.split_cnt + unit, (unsigned)PARTS);
  __syncthreads();
  if (!sh_last) return;

  // the unit's last arrival: the prefix, then the remaining classes in order, then the rows. Every value a
  // (half, dim tile) pair needs is loaded at once.
  for (int gi = w; gi < GI; gi += WPP) {
    const int nt = gi / MT, mt = gi - nt * MT, r = 16 * nt + l16;
    float4_t a[NSLOT];
    float m[NSLOT], l[NSLOT];
#pragma unroll
    for (int v = 0; v < NSLOT; ++v) {
      a[v] = ld4_dev(scr, acc_at(v, gi));
      m[v] = ld1_dev(scr, m_at(v, r));
      l[v] = ld1_dev(scr, l_at(v, r));
    }
    float M = m[0], L = l[0];
    float4_t o = a[0];
#pragma unroll
    for (int v = 1; v < NSLOT; ++v) {
      float Mn, cM, cm;
      if (!fold_weights(M, m[v], Mn, cM, cm)) continue;
      L = fold_value(L, cM, l[v], cm);
#pragma unroll
      for (int c = 0; c < 4; ++c) o[c] = fold_value(o[c], cM, a[v][c], cm);
      M = Mn;
    }
    if (r < nrows) attn_emit<D, 1>(P, b, s, kbeg, hkv, row0 + r, nt ? rpos[1] : rpos[0], mt, M, L, {o});
  }
}

// ------------------------------------------------------------------------------------------------
// prefill kernel: one workgroup of PF_WAVES waves per (plan item of PF_WAVES query tiles, KV head)
// ------------------------------------------------------------------------------------------------
// A prompt's queries are many 32-row tiles per row. Here the PF_WAVES tiles of an item (256 query rows:
// wave w owns tile PF_WAVES * item.z + w) share every key and value tile through an LDS ring that
// direct global->LDS copies fill, so a key tile is read from memory once per 256 query rows instead of
// once per 32. Each wave computes, for its own rows, exactly what the unit kernel computes for them:
// the partial of the pairs p = v, v + 8, v + 16, ... (v = 0..7, increasing), with pair_step, folded in
// increasing v with fold_weights/fold_value. The ring therefore carries the chunk's pairs in that
// order (all pairs p % 8 == 0, then p % 8 == 1, ...), and a wave skips the pairs wholly above its
// furthest query (no-ops for every row of the wave). Output bits equal the unit kernel's.
//
// Bound by vector instructions and the waits between the steps of a pair (2 waves per SIMD, 244 registers at 128
// dims: no room to form one pair's scores under another's softmax): per pair and wave 32 products (512 cycles)
// against about 240 vector instructions, a quarter of them the folds of the 8 classes. Tile by tile instead of
// pair by pair it issued 360. Prompts of 4096, 1228, 1817, 1837 and 817 tokens (32/8 heads, 128 dims):
// 494 -> 437 us; raising the waves' priority around the products changes it by 1%.
constexpr int PF_WAVES = 8;      // query tiles (waves) per workgroup
// 16-key tiles per ring stage, and stages (PF_NS - 2 in flight behind the one awaited). Two long stages rather than four
// of half their length: half the barriers, each of which puts the eight waves in step again (prompts of 817-4096
// tokens 395 -> 390 us, four of 2048 246 -> 242; three short stages: 428).
constexpr int PF_TILES = 8;
constexpr int PF_NS = 2;
constexpr int PF_MIN_QTILES = 5; // a call with at least this many query tiles per row takes this kernel

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// One 16-byte copy per lane straight into LDS from sbase + voff (a wave-uniform base in SGPRs and a
// 32-bit unsigned per-lane byte offset; lane l lands at lds + 16 * l, the same base for the whole
// wave). The copy is counted by vmcnt like any vector load; the waits below are explicit.
FS_DEVICE void pf_dma16(const void* sbase, uint32_t voff, uint32_t lds) {
  const uint32_t l = __builtin_amdgcn_readfirstlane(lds);
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(l) : "memory", "m0");
}
#pragma clang diagnostic pop
template <int N>
FS_DEVICE void pf_wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The chunk's pairs of tiles (2p, 2p + 1) in the ring's order: class v = p % 8 in increasing v, increasing p inside
// a class. The pair after p (of n) is p + 8, or the next class's first pair (p % 8) + 1.
FS_DEVICE int pf_next_pair(int p, int n) {
  p += 8;
  return p < n ? p : (p & 7) + 1;
}
// The pair at place j (0 <= j < n): class v holds the n_v = ceil((n - v) / 8) pairs v, v + 8, ...
FS_DEVICE int pf_pair(int j, int n) {
  int first = 0, p = 0;
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    const int nv = n > v ? ((n - 1 - v) >> 3) + 1 : 0;
    if (j >= first && j < first + nv) p = v + 8 * (j - first);
    first += nv;
  }
  return p;
}

template <int D, int BSZ>
__global__ void __launch_bounds__(64 * PF_WAVES) __attribute__((amdgpu_waves_per_eu(2)))
attn_prefill_kernel(AttnParams P) {
  constexpr int KS = D / 32, MT = D / 16;
  constexpr int TK = 16 * D * 2;                    // bytes of a tile's keys (and of its values)
  constexpr int TB = 2 * TK;                        // a tile in LDS: keys, then values
  constexpr int CPT = TB / 1024;                    // 1 KB copies per tile
  constexpr int CPW = PF_TILES * CPT / PF_WAVES;    // copies per wave per stage
  constexpr int CPR = D / 8;                        // 16-byte chunks per key row
  constexpr int STAGE = PF_TILES * TB;
  static_assert(PF_WAVES % CPT == 0 && CPW >= 1, "every wave copies the same part of its tiles");
  static_assert(PF_NS >= 2 && PF_NS <= 4, "the waits below cover two stages in flight behind the awaited one");
  __shared__ __attribute__((aligned(1024))) char ring[PF_NS * STAGE];
  __shared__ int tbl[MAX_SPLIT / 16 + 1];           // the chunk's physical blocks (-1: unmapped)

  const int nkv = P.kv.n_kv_heads;
  const int64_t e_idx = blockIdx.x / nkv;
  const int hkv = (int)(blockIdx.x - e_idx * nkv);
  if (e_idx >= P.n_items[0]) return;   // uniform over the workgroup
  typedef __attribute__((address_space(4))) const AttnItem ConstItem;
  ConstItem* ep = (ConstItem*)(uintptr_t)(P.items + e_idx);
  const int b = ep->b, zb = ep->z, s = ep->s, qmax_item = ep->qmax;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int BS = BSZ ? BSZ : P.kv.block_size;
  const int64_t v_dim = BSZ ? BSZ : P.kv.v_dim;   // == block_size (dim-major values)
  const int kbeg = s * P.split;
  const int kend = min(kbeg + P.split, qmax_item + 1);
  const int ntiles = max((kend - kbeg + 15) >> 4, 0);
  const int npairs = (ntiles + 1) >> 1;
  const int nst = (2 * npairs + PF_TILES - 1) / PF_TILES;

  // this wave's query tile: the unit kernel's tile z, with its rows, positions and furthest query
  const int z = zb * PF_WAVES + w;
  const int row0 = z * QTILE;
  const int nrows = min(QTILE, P.T * P.G - row0);   // <= 0: a wave past the last tile (copies only)
  const int* posb = P.pos + (int64_t)b * P.T;
  int rpos[2];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int r = 16 * nt + l16;
    rpos[nt] = (r < nrows) ? posb[(row0 + r) / P.G] : -1;
  }
  const int qmax = nrows > 0 ? tile_qmax(P, b, z) : -1;
  const int rmin = rows_min_pos(rpos, nrows);
  const int ntiles_w = nrows > 0 ? min(max((min(kbeg + P.split, qmax + 1) - kbeg + 15) >> 4, 0), ntiles) : 0;

  typedef uint16_t u16;
  const u16* qbase = reinterpret_cast<const u16*>(P.q);
  bf16x8_t qf[2][KS];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int r = row0 + 16 * nt + l16;
    const bool in_tile = nrows > 0 && (16 * nt + l16) < nrows;
    const bool ok = in_tile && token_exists(P, b, r / P.G);
    const int t = ok ? r / P.G : 0;
    const int h = hkv * P.G + (ok ? r - (r / P.G) * P.G : 0);
    const u16* qr = qbase + q_offset(P, b, t) + (int64_t)h * P.q_sh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[nt][ks] = ok ? signed_query(*reinterpret_cast<const bf16x8_t*>(qr + 32 * ks + 8 * g), P.scale_log2) : bf16x8_t{};
  }

  // the chunk's table entries
  const int blk0 = kbeg / BS;
  const int nblk = ntiles > 0 ? (kbeg + 16 * ntiles - 1) / BS - blk0 + 1 : 0;
  int unmapped = 0;
  for (int i = tid; i < nblk; i += 64 * PF_WAVES) {
    const int blk = blk0 + i;
    int v = blk < P.max_blocks ? P.table[(int64_t)b * P.table_stride + blk] : -1;
    v = (v >= 0 && v < P.kv.num_blocks) ? v : -1;
    unmapped |= v < 0;
    tbl[i] = v;
  }
  // every load above has landed (the copies below are counted by the explicit waits only)
  __builtin_amdgcn_s_waitcnt(0);
  const bool all_mapped = !__syncthreads_or(unmapped);   // (the common case: no lookups per tile)

  // This wave copies part p = w % CPT of every tile it copies (keys for p < CPT/2, else values).
  // LDS layouts (16-byte slots; 16 consecutive slots are read without bank conflicts):
  //  * slot-major keys: row r's 16-byte chunk c at slot r * CPR + (c ^ f(r)), f(r) = r & 15 for 16
  //    chunks per row, (r >> 1) & 7 for 8, so the 16 rows of an MFMA operand read 16 different slots
  //    mod 16; grouped keys: chunk c of row r at slot 16 * c + r, the pool's own order (each copy is
  //    then one contiguous 1 KB of the pool, and an operand's 16 rows are 16 consecutive slots);
  //  * values: dim d's keys 8h .. 8h+7 at slot 2d + (h ^ ((d >> 3) & 1)), so dims d and d + 8 of an
  //    operand read different slots mod 16.
  const int p = w % CPT;
  const bool kpart = p < CPT / 2;
  const bool kgrp = P.kv.k_group != 0;
  const int64_t kgs = key_group_stride(P.kv);
  int64_t src_off;
  {
    const int P16 = (kpart ? p : p - CPT / 2) * 64 + lane;
    if (kpart && kgrp) {
      src_off = (int64_t)(P16 & 15) * 8 + (int64_t)(P16 >> 4) * kgs;
    } else if (kpart) {
      const int row = P16 / CPR, f = CPR == 16 ? (row & 15) : ((row >> 1) & 7);
      const int c = (P16 % CPR) ^ f;
      src_off = (int64_t)row * D + 8 * c;
    } else {
      const int d = P16 >> 1, h = (P16 & 1) ^ ((d >> 3) & 1);
      src_off = (int64_t)d * v_dim + 8 * h;
    }
  }
  // copies read pool_h + (a tile's offset) + coff: the head's base is wave-uniform, the lane's part of
  // a tile lies inside one block (a few KB), so it fits the 32-bit offset of the scalar-base form
  const char* pool_h = reinterpret_cast<const char*>(kpart ? P.kv.k : P.kv.v) +
                       2 * (int64_t)hkv * (kpart ? P.kv.k_head : P.kv.v_head);
  const uint32_t coff = (uint32_t)(2 * src_off);
  const int64_t blk_stride = kpart ? P.kv.k_block : P.kv.v_block;
  const int64_t slot_mul = kpart ? P.kv.k_slot : 1;
  const uint32_t ring0 = (uint32_t)(uintptr_t)ring;
  // this lane's operand reads inside a tile (bytes)
  const int fk = CPR == 16 ? (l16 & 15) : ((l16 >> 1) & 7);
  // (chunk 4ks + g of a row's keys lies at koff ^ (ks * kx): one register for the KS addresses)
  const int koff = (kgrp ? g * 16 + l16 : l16 * CPR + (g ^ fk)) * 16, kx = kgrp ? 1024 : 64;
  const int voff = TK + (2 * l16 + ((g >> 1) ^ ((l16 >> 3) & 1))) * 16 + 8 * (g & 1);

  // Copies walk the ring positions PF_TILES at a time; a position without a tile copies the last
  // tile again. Lane j holds the byte offset of the tile at ring position 64 * win + j (relative to
  // pool_h), refreshed when a stage enters the next 64 positions, so a copy reads its tile's offset
  // with two lane reads instead of walking the order and the table per copy.
  static_assert(64 % PF_TILES == 0, "a stage's positions lie in one 64-position window");
  uint32_t woff_lo = 0, woff_hi = 0;
  auto refresh = [&](int win) {
    const int j = min(64 * win + lane, 2 * npairs - 1);
    const int t = min(2 * pf_pair(j >> 1, npairs) + (j & 1), ntiles - 1);
    const int key0 = kbeg + 16 * t;
    const int bi = key0 / BS;
    const int ph = tbl[bi - blk0];
    const int64_t pb = ph >= 0 ? ph : 0;         // unmapped: block 0, masked in pair_step
    const uint64_t o = (uint64_t)(2 * (pb * blk_stride + (int64_t)(key0 - bi * BS) * slot_mul));
    woff_lo = (uint32_t)o;
    woff_hi = (uint32_t)(o >> 32);
  };
  auto issue = [&](int k) {
    if ((k & (64 / PF_TILES - 1)) == 0) refresh(k / (64 / PF_TILES));
    const uint32_t base = ring0 + (uint32_t)((k % PF_NS) * STAGE) + (uint32_t)(p * 1024);
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
      const int u = (w + PF_WAVES * i) / CPT;   // the stage's tile this copy fills
      const int j = (PF_TILES * k + u) & 63;
      const uint64_t o = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)woff_hi, j) << 32) |
                         (uint32_t)__builtin_amdgcn_readlane((int)woff_lo, j);
      pf_dma16(pool_h + o, coff, base + (uint32_t)(u * TB));
    }
  };
  auto wait_stages = [&](int later) {
    if (later >= 2) pf_wait_vm<2 * CPW>();
    else if (later == 1) pf_wait_vm<CPW>();
    else pf_wait_vm<0>();
  };

  float4_t acc[MT][2], O[MT][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      acc[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
      O[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
  float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};
  float Ms[2] = {-INFINITY, -INFINITY}, Ls[2] = {0.f, 0.f};
  // the finished partial of class v into the row state, then an empty partial for the next class
  auto fold = [&]() {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const float l = sum_across_groups(l_run[nt]);
      float Mn, cM, cm;
      if (fold_weights(Ms[nt], m_run[nt], Mn, cM, cm)) {
        Ls[nt] = fold_value(Ls[nt], cM, l, cm);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int c = 0; c < 4; ++c) O[mt][nt][c] = fold_value(O[mt][nt][c], cM, acc[mt][nt][c], cm);
        Ms[nt] = Mn;
      }
      m_run[nt] = -INFINITY;
      l_run[nt] = 0.f;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
  };

#pragma unroll
  for (int k = 0; k < PF_NS - 1; ++k)
    if (k < nst) issue(k);
  int next = 0;   // the pair consumed next
  bool fresh = true;   // acc is all zeros
  int cur_v = 0;
  const float scale = positive_scale(P.scale_log2);
  auto mapped = [&](int key0) { return all_mapped || tbl[key0 / BS - blk0] >= 0; };
  for (int k = 0; k < nst; ++k) {
    wait_stages(min(PF_NS - 2, nst - 1 - k));
    __syncthreads();   // stage k has landed for every wave; stage k-1 is no longer being read
    if (k + PF_NS - 1 < nst) issue(k + PF_NS - 1);
    // the stage's operand addresses, once per stage: each tile's reads add only its constant offset
    const uint32_t st_lds = ring0 + (uint32_t)((k % PF_NS) * STAGE);
    const uint32_t vad = st_lds + (uint32_t)voff;
#pragma unroll 2
    for (int u = 0; u < PF_TILES; u += 2) {
      if (k * (PF_TILES / 2) + u / 2 >= npairs) break;
      const int pair = next;
      next = pf_next_pair(next, npairs);
      if (nrows <= 0) continue;
      if ((pair & 7) != cur_v) {   // a new class: fold the last one into the row state
        fold();
        fresh = true;
        cur_v = pair & 7;
      }
      if (2 * pair >= ntiles_w) continue;   // wholly above every query of the wave
      typedef __attribute__((address_space(3))) const bf16x8_t LdsK;
      typedef __attribute__((address_space(3))) const short4_t LdsV;
      auto value = [&](int mt) {
        // (an address that the compiler cannot split pairs the two tiles' reads, into the operand's registers)
        uint32_t at = vad + (uint32_t)(u * TB + mt * 16 * 32);
        asm("" : "+v"(at));
        return pair_value(*(LdsV*)(uintptr_t)at, *(LdsV*)(uintptr_t)(at + TB));
      };
      float4_t sc[2][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        bf16x8_t kf[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kf[ks] = *(LdsK*)(uintptr_t)(st_lds + (uint32_t)(koff ^ (ks * kx)) + (uint32_t)((u + h) * TB));
        tile_scores<D, true>(kf, qf, sc[h]);
        __builtin_amdgcn_sched_barrier(0);   // (one tile's keys in registers)
      }
      const int key0 = kbeg + 32 * pair;
      const bool ok[2] = {mapped(key0), 2 * pair + 1 < ntiles && mapped(key0 + 16)};
      pair_step<D, true>(sc, value, key0, ok, fresh, qmax, rpos, rmin, scale, acc, m_run, l_run);
      fresh = false;
    }
  }
  if (nrows <= 0) return;
  fold();
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int r = 16 * nt + l16;
    if (r >= nrows) continue;
#pragma unroll
    for (int mt = 0; mt < MT; mt += 4)
      attn_emit<D, 4>(P, b, s, kbeg, hkv, row0 + r, rpos[nt], mt, Ms[nt], Ls[nt],
                      {O[mt][nt], O[mt + 1][nt], O[mt + 2][nt], O[mt + 3][nt]});
  }
}

// ------------------------------------------------------------------------------------------------
// generic kernel (any dtype, head_dim <= 256, any strides and block size)
// ------------------------------------------------------------------------------------------------
template <int DT>
__global__ void __launch_bounds__(64) attn_generic_kernel(AttnParams P) {
  typedef Elem<DT> E;
  typedef typename E::T T_;
  __shared__ float qs[256];
  __shared__ float ps[64];
  const int lane = threadIdx.x;
  const int s = blockIdx.y;
  const int64_t R = blockIdx.x;  // (b, t, h)
  const int h = (int)(R % P.H);
  const int bt = (int)(R / P.H);
  const int b = bt / P.T, t = bt - b * P.T;
  const int pos = P.pos[bt];
  const int kbeg = s * P.split;
  if (pos < kbeg) return;
  const int kend = min(kbeg + P.split, pos + 1);
  const int D = P.kv.head_dim, BS = P.kv.block_size;
  const int hkv = h / P.G;
  const T_* qrow = reinterpret_cast<const T_*>(P.q) + q_offset(P, b, t) + (int64_t)h * P.q_sh;
  for (int d = lane; d < D; d += 64) qs[d] = E::load(qrow, d);
  __syncthreads();
  const T_* kp = reinterpret_cast<const T_*>(P.kv.k);
  const T_* vp = reinterpret_cast<const T_*>(P.kv.v);
  const int32_t* trow = P.table + (int64_t)b * P.table_stride;

  float m_run = -INFINITY, l_run = 0.f;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int j0 = kbeg; j0 < kend; j0 += 64) {
    const int j = j0 + lane;
    float sv = -INFINITY;
    if (j < kend) {
      const int bi = j / BS;
      const int64_t blk = (bi < P.max_blocks) ? trow[bi] : -1;
      if (blk >= 0 && blk < P.kv.num_blocks) {
        const T_* kr = kp + blk * P.kv.k_block + hkv * P.kv.k_head + (int64_t)(j - bi * BS) * P.kv.k_slot;
        float dot = 0.f;
        for (int d = 0; d < D; ++d) dot = fmaf(qs[d], E::load(kr, key_dim_off(P.kv, d)), dot);
        sv = dot * P.scale_log2;
      }
    }
    const float m_new = fmaxf(m_run, wave_max(sv));
    const float alpha = (m_new == -INFINITY) ? 1.f : exp2f(m_run - m_new);
    const float p = (sv == -INFINITY) ? 0.f : exp2f(sv - m_new);
    l_run = l_run * alpha + wave_sum(p);
    m_run = m_new;
    __syncthreads();
    ps[lane] = p;
    __syncthreads();
    const int nj = min(64, kend - j0);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int d = lane + 64 * c;
      if (d >= D) break;
      float a = acc[c] * alpha;
      for (int jj = 0; jj < nj; ++jj) {
        const float pj = ps[jj];
        if (pj == 0.f) continue;  // masked, invalid-block or underflowed key: adds an exact zero
        const int jk = j0 + jj;
        const int bi = jk / BS;
        const int64_t blk = trow[bi];
        const T_* vr = vp + blk * P.kv.v_block + hkv * P.kv.v_head + (int64_t)(jk - bi * BS) * P.kv.v_slot;
        a = fmaf(pj, E::load(vr, (int64_t)d * P.kv.v_dim), a);
      }
      acc[c] = a;
    }
  }
  float* pa = P.ws_acc + (R * P.nsplit + s) * D;
  for (int c = 0; c < 4; ++c) {
    const int d = lane + 64 * c;
    if (d < D) pa[d] = acc[c];
  }
  if (lane == 0) {
    float* pm = P.ws_ml + (R * P.nsplit + s) * 2;
    pm[0] = m_run;
    pm[1] = l_run;
  }
}

// ------------------------------------------------------------------------------------------------
// float32 kernel: one wave per (batch row, KV head, 16 query rows, chunk of GENERIC_SPLIT keys)
// ------------------------------------------------------------------------------------------------
// The bf16 kernels' transposed products on v_mfma_f32_16x16x4_f32, nothing rounded below float32: 16-key
// tiles, lane group g holding dims 16s + 4g .. +3 of a key (one 16-byte load), so four instructions add 16 dims;
// S^T leaves lane (l16, g) with row l16's scores of keys 4g .. 4g+3, which are the keys it reads 16 bytes of
// per dim of the dim-major values. Dims past head_dim are zeros. A tile's keys and values are loaded while
// the one before is multiplied. A query's result depends on its own position only: a row's tiles run in
// order, a tile above its position leaves its state as it is, chunks are merged by attn_combine.
//
// Latency-bound at the sizes float32 models have (a few waves of a few tiles each). The scalar kernel below
// walked 64 keys per step with a lane per key and then a lane per dim. One row of a token at position 100 (8/4
// heads of 32 dims): 30 -> 12 us; four rows of 160 tokens: 83 -> 18 us.
constexpr int F32_ROWS = 16;

template <int S>   // 16-dim groups: head_dim <= 16 S
__global__ void __launch_bounds__(64) attn_f32_kernel(AttnParams P) {
  const int lane = threadIdx.x, l16 = lane & 15, g = lane >> 4;
  const int nkv = P.kv.n_kv_heads, D = P.kv.head_dim, BS = P.kv.block_size;
  const int qtiles = (P.T * P.G + F32_ROWS - 1) / F32_ROWS;
  const int hkv = (int)(blockIdx.x % nkv);
  const int bz = (int)(blockIdx.x / nkv);
  const int b = bz / qtiles, row0 = (bz - b * qtiles) * F32_ROWS;
  const int s = blockIdx.y;
  const int kbeg = s * P.split;
  const int qmax = rows_qmax(P, b, row0, F32_ROWS);
  if (qmax < kbeg && s > 0) return;
  const int kend = min(kbeg + P.split, qmax + 1);
  const int r = row0 + l16;
  const bool in = r < P.T * P.G;
  const int t = in ? r / P.G : 0, h = hkv * P.G + (in ? r - t * P.G : 0);
  const bool exists = in && token_exists(P, b, t);
  const int pos = in ? P.pos[(int64_t)b * P.T + t] : -1;

  int rmin = in ? pos : 0x7fffffff;   // the smallest position of the 16 rows
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) rmin = min(rmin, __shfl_xor(rmin, o, 64));

  const float4_t zero = float4_t{0.f, 0.f, 0.f, 0.f};
  const float* qr = reinterpret_cast<const float*>(P.q) + (exists ? q_offset(P, b, t) + (int64_t)h * P.q_sh : 0);
  float4_t qf[S];
#pragma unroll
  for (int i = 0; i < S; ++i) qf[i] = exists && 16 * i + 4 * g < D ? *reinterpret_cast<const float4_t*>(qr + 16 * i + 4 * g) : zero;

  const float* kp = reinterpret_cast<const float*>(P.kv.k) + (int64_t)hkv * P.kv.k_head;
  const float* vp = reinterpret_cast<const float*>(P.kv.v) + (int64_t)hkv * P.kv.v_head;
  const int32_t* trow = P.table + (int64_t)b * P.table_stride;
  const int shift = (BS & (BS - 1)) == 0 ? 31 - __clz(BS) : -1;
  auto block_index = [&](int j) { return shift >= 0 ? j >> shift : j / BS; };
  // block of key j, -1 when past the chunk's keys or unmapped
  auto block_of = [&](int j) {
    const int bi = block_index(j);
    const int v = j < kend && bi < P.max_blocks ? trow[bi] : -1;
    return v >= 0 && v < P.kv.num_blocks ? v : -1;
  };
  // A tile: lane (l16, g) holds dims 16i + 4g .. of key j0 + l16, and keys j0 + 4g .. of dim 16i + l16 (block_size
  // % 4 == 0: the four share a block); `ok` has a bit per key of its four that may be used
  struct Tile {
    float4_t k[S], v[S];
    int ok;
  };
  auto load = [&](Tile& x, int j0) {
    const int jk = j0 + l16, bk = block_of(jk), jv = j0 + 4 * g, bv = block_of(jv);
    const float* kr = kp + (bk < 0 ? 0 : bk * P.kv.k_block + (int64_t)(jk - block_index(jk) * BS) * P.kv.k_slot);
    const float* vr = vp + (bv < 0 ? 0 : bv * P.kv.v_block + (int64_t)(jv - block_index(jv) * BS));
    x.ok = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (bv >= 0 && jv + e < kend) x.ok |= 1 << e;
#pragma unroll
    for (int i = 0; i < S; ++i) {
      x.k[i] = bk >= 0 && 16 * i + 4 * g < D ? *reinterpret_cast<const float4_t*>(kr + key_dim_off(P.kv, 16 * i + 4 * g)) : zero;
      x.v[i] = bv >= 0 && 16 * i + l16 < D ? *reinterpret_cast<const float4_t*>(vr + (16 * i + l16) * P.kv.v_dim) : zero;
    }
  };

  float4_t acc[S];
#pragma unroll
  for (int i = 0; i < S; ++i) acc[i] = zero;
  float m_run = -INFINITY, l_run = 0.f;
  auto consume = [&](const Tile& x, int j0) {
    float4_t sc = zero;
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[i][e], qf[i][e], sc, 0, 0, 0);
    float sv[4], tmax = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sv[e] = (x.ok >> e & 1) && j0 + 4 * g + e <= pos ? sc[e] * P.scale_log2 : -INFINITY;
      tmax = fmaxf(tmax, sv[e]);
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m_run, tmax);
    const float alpha = m_new == -INFINITY ? 1.f : exp2f(m_run - m_new);
    float p[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = sv[e] == -INFINITY ? 0.f : exp2f(sv[e] - m_new);
    l_run = l_run * alpha + ((p[0] + p[1]) + (p[2] + p[3]));   // this lane group's keys
    m_run = m_new;
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][e] *= alpha;
    // A key that a row may not see has weight 0 there, which an infinite or NaN value would turn into NaN:
    // in a tile that some row sees only in part, such values take the products key by key.
    float4_t v[S];
    float bad = 0.f;
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {   // (a value never written may be anything)
        v[i][e] = x.ok >> e & 1 ? x.v[i][e] : 0.f;
        bad = fmaf(v[i][e], 0.f, bad);
      }
    if (j0 + 15 > rmin && __any(bad != 0.f)) {
      for (int j = 0; j < 16; ++j) {
        const int src = (j >> 2) * 16;   // the lane group that holds key j's weights and values
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (e != (j & 3)) continue;
          const float pj = __shfl(p[e], src + l16, 64);
#pragma unroll
          for (int i = 0; i < S; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              const float vj = __shfl(v[i][e], src + 4 * g + c, 64);   // dim 16i + 4g + c
              if (pj != 0.f) acc[i][c] = fmaf(pj, vj, acc[i][c]);
            }
        }
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[i][e], p[e], acc[i], 0, 0, 0);
  };

  Tile a, c;
  if (kbeg < kend) load(a, kbeg);
  for (int j0 = kbeg; j0 < kend; j0 += 32) {
    if (j0 + 16 < kend) load(c, j0 + 16);
    consume(a, j0);
    if (j0 + 32 < kend) load(a, j0 + 32);
    if (j0 + 16 < kend) consume(c, j0 + 16);
  }
  // (g0 + g1) + (g2 + g3) in every lane
  float l = l_run + __shfl_xor(l_run, 16, 64);
  l = l + __shfl_xor(l, 32, 64);

  // acc[i]: lane (l16, g) has row l16's dims 16i + 4g .. +3
  if (!in) return;
  if (P.nsplit == 1) {   // one chunk: the same division as attn_combine's (a padding query, pos < 0, gives zeros)
    if (!exists) return;
    float* orow = reinterpret_cast<float*>(P.out) + o_offset(P, b, t, P.o_sb, P.o_st) + (int64_t)h * P.o_sh;
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (16 * i + 4 * g + e < D) orow[16 * i + 4 * g + e] = l > 0.f ? acc[i][e] / l : 0.f;
    return;
  }
  if (pos < kbeg) return;   // attn_combine reads the chunks that hold keys a query sees
  const int64_t R = row_index(P, b, t, h);
#pragma unroll
  for (int i = 0; i < S; ++i)
    if (16 * i + 4 * g < D) *reinterpret_cast<float4_t*>(P.ws_acc + (R * P.nsplit + s) * D + 16 * i + 4 * g) = acc[i];
  if (g == 0) {
    float* pm = P.ws_ml + (R * P.nsplit + s) * 2;
    pm[0] = m_run;
    pm[1] = l;
  }
}

// Whole 16-byte pieces of queries, keys and values, head_dim <= 128, four consecutive keys in one block.
bool f32_eligible(const fs_kv_layout& kv, const void* q, int64_t q_sb, int64_t q_st, int64_t q_sh) {
  if (kv.dtype != FS_F32 || kv.head_dim % 4 || kv.head_dim > 128 || kv.block_size % 4) return false;
  if (kv.k_dim != 1 || kv.v_slot != 1) return false;
  if ((kv.k_block | kv.k_head | kv.k_slot | kv.k_group | kv.v_block | kv.v_head | kv.v_dim | q_sb | q_st | q_sh) & 3) return false;
  return ((reinterpret_cast<uintptr_t>(kv.k) | reinterpret_cast<uintptr_t>(kv.v) | reinterpret_cast<uintptr_t>(q)) & 15) == 0;
}

// ------------------------------------------------------------------------------------------------
// combine: out[b,t,h,:] = sum_s 2^(m_s - M) acc_s / sum_s 2^(m_s - M) l_s, chunks in increasing order
// ------------------------------------------------------------------------------------------------
constexpr int COMBINE_ROWS = 4;   // rows (waves) per combine workgroup

template <int DT>
__global__ void __launch_bounds__(64 * COMBINE_ROWS) attn_combine_kernel(AttnParams P, void* out, int64_t o_sb,
                                                                         int64_t o_st, int64_t o_sh) {
  typedef Elem<DT> E;
  typedef typename E::T T_;
  const int lane = threadIdx.x & 63;
  const int64_t R = (int64_t)blockIdx.x * COMBINE_ROWS + (threadIdx.x >> 6);
  if (R >= (int64_t)P.B * P.T * P.H) return;
  const int h = (int)(R % P.H);
  const int bt = (int)(R / P.H);
  const int b = bt / P.T, t = bt - b * P.T;
  const int pos = P.pos[bt];
  if (P.direct && (pos < P.split || P.nsplit == 1)) return;   // written by its chunk's workgroup
  if (!token_exists(P, b, t)) return;
  const int D = P.kv.head_dim;
  T_* orow = reinterpret_cast<T_*>(out) + o_offset(P, b, t, o_sb, o_st) + (int64_t)h * o_sh;
  if (pos < 0) {
    for (int d = lane; d < D; d += 64) E::store(orow, d, 0.f);
    return;
  }
  const int ns = min(pos / P.split + 1, P.nsplit);  // keys past the table were never visible
  const float* ml = P.ws_ml + R * P.nsplit * 2;
  const float* pa = P.ws_acc + R * P.nsplit * D;
  float M = -INFINITY;
  for (int s = lane; s < ns; s += 64) M = fmaxf(M, ml[2 * s]);
  M = wave_max(M);
  // Chunk s's weight and weighted sum live in lane s % 64; the partial rows are loaded eight chunks
  // at a time and summed in increasing chunk order.
  float L = 0.f;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < ns; s0 += 64) {
    float w = 0.f, lw = 0.f;
    if (s0 + lane < ns) {
      const float ms = ml[2 * (s0 + lane)];
      w = (ms == -INFINITY) ? 0.f : exp2f(ms - M);
      lw = w * ml[2 * (s0 + lane) + 1];
    }
    const int n = min(64, ns - s0);
    for (int j = 0; j < n; j += 8) {
      float v[8][4];
#pragma unroll
      for (int jj = 0; jj < 8; ++jj)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int d = lane + 64 * c;
          v[jj][c] = (j + jj < n && d < D) ? pa[(int64_t)(s0 + j + jj) * D + d] : 0.f;
        }
#pragma unroll
      for (int jj = 0; jj < 8; ++jj) {
        if (j + jj < n) {
          const float wj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), j + jj));
          L += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lw), j + jj));
#pragma unroll
          for (int c = 0; c < 4; ++c) acc[c] += wj * v[jj][c];
        }
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int d = lane + 64 * c;
    if (d < D) E::store(orow, d, L > 0.f ? acc[c] / L : 0.f);
  }
}

bool mfma_eligible(const fs_kv_layout& kv, const void* q, int64_t q_sb, int64_t q_st, int64_t q_sh) {
  if (kv.dtype != FS_BF16) return false;
  if (kv.head_dim != 64 && kv.head_dim != 128) return false;
  if (kv.block_size % 16 != 0) return false;  // a 16-key tile never straddles two blocks
  if (kv.k_dim != 1 || kv.v_slot != 1 || kv.v_dim != kv.block_size) return false;
  const bool slot_major = kv.k_group == 0 && kv.k_slot == kv.head_dim;
  const bool grouped = kv.k_group == 8 * (int64_t)kv.block_size && kv.k_slot == 8;
  if (!slot_major && !grouped) return false;
  if (kv.k_block % 8 || kv.k_head % 8 || kv.v_block % 8 || kv.v_head % 8) return false;
  if ((reinterpret_cast<uintptr_t>(kv.k) | reinterpret_cast<uintptr_t>(kv.v) | reinterpret_cast<uintptr_t>(q)) & 15)
    return false;
  if (q_sb % 8 || q_st % 8 || q_sh % 8) return false;
  return true;
}

// Keys per chunk. The generic kernel uses 512. The MFMA path uses FS_ATTN_SPLIT (default 16384 =
// MAX_SPLIT; a multiple of 64 in [256, MAX_SPLIT]), read once: it must stay fixed for the life of the
// process, since the chunk boundaries decide the rounding of every output. A large chunk keeps batched
// rows of up to 16K keys in one workgroup per KV head (no partials, no combine); few rows of much
// longer contexts spread over more workgroups with a smaller one.
constexpr int GENERIC_SPLIT = 512;

int attn_split() {
  static const int split = [] {
    const char* e = getenv("FS_ATTN_SPLIT");
    int v = e ? atoi(e) : MAX_SPLIT;
    if (v < 256 || v > MAX_SPLIT || v % 64) v = MAX_SPLIT;
    return v;
  }();
  return split;
}

int64_t nsplit_for(int32_t max_blocks, int32_t block_size, int split) {
  const int64_t S = (int64_t)max_blocks * block_size;
  return (S + split - 1) / split;
}

// Upper bound of the plan's length: every (row, query tile, chunk), at the smallest chunk size.
int64_t max_items(int32_t B, int32_t T, int32_t n_heads, int32_t max_blocks, int32_t block_size, int split) {
  const int64_t qtiles = ((int64_t)T * n_heads + QTILE - 1) / QTILE;   // n_heads bounds the group size
  return (int64_t)B * qtiles * nsplit_for(max_blocks, block_size, split);
}

int min_split() { return attn_split() < GENERIC_SPLIT ? attn_split() : GENERIC_SPLIT; }

// Bytes of the split units' published partials for calls of at most `units` units (KV heads never
// outnumber query heads, so items x n_heads bounds the units).
int64_t split_bytes(int64_t units, int32_t head_dim) {
  return (units < SPLIT_UNITS_MAX ? units : (int64_t)SPLIT_UNITS_MAX) * SPLIT_SLOTS * split_slot_floats(head_dim) *
         (int64_t)sizeof(float);
}

// Workgroups per unit of a call of at most `units` units whose tables hold `keys` keys; two: its tiles have a
// second half of query rows (twice the partials to exchange). Measured (us: one, two and four workgroups a
// unit; 32/8 heads, 128 dims unless said): 24 units of 8000-30000 keys, T = 1: 159 / 95 / 63; 8 of 1000: 14.6 /
// 12.0 / 13.9; 32 of 500-2000: 23.3 / 17.4 / 16.3; 64 of 512-4096: 61 / 38 / 29; 128 of them: 46.7 / 39.8 / 41.6;
// 128 of 128-1280 keys, 64 dims: 15.2 / 12.6 / 13.4. With two halves (T = 5): 64 of 512-4096: 64 / 43 / 38; 128 of
// them: 49.6 / 44.9 / 50.8; 16 of 2000-6000: 58 / 39 / 40; 128 of 1000-3000 keys, 64 dims: 21.2 / 22.1 / 24.5; 8 of
// 500, 64 dims: 10.3 / 11.1 / 13.7. 256 units of 512-4096 keys in two: 61 -> 69.
int split_parts(int64_t units, int64_t keys, bool two) {
  if (units > SPLIT_UNITS_MAX || keys < (two ? 3072 : 768)) return 1;
  return units <= SPLIT_UNITS_MAX / 2 && keys >= (two ? 4096 : 2048) ? 4 : 2;
}

}  // namespace

extern "C" int32_t fs_paged_attention_split(void) { return attn_split(); }

extern "C" int64_t fs_paged_attention_workspace_size(int32_t B, int32_t T, int32_t n_heads, int32_t head_dim,
                                                     int32_t max_blocks, int32_t block_size) {
  if (B <= 0 || T <= 0 || n_heads <= 0 || head_dim <= 0 || max_blocks <= 0 || block_size <= 0) return 0;
  const int64_t rows = (int64_t)B * T * n_heads;
  const int64_t ns = nsplit_for(max_blocks, block_size, min_split());
  const int64_t items = max_items(B, T, n_heads, max_blocks, block_size, min_split());
  const int64_t list = (items * (int64_t)sizeof(AttnItem) + 255) / 256 * 256;
  const int64_t partials = (rows * ns * (head_dim + 2) * (int64_t)sizeof(float) + 255) / 256 * 256;
  return WS_HEADER + list + partials + split_bytes(items * n_heads, head_dim) + 256;
}

namespace {
// What the work plan of a call depends on besides the contents of its positions: a call that asks to
// reuse the plan already in its workspace skips the plan kernel only when all of these match the call
// that wrote it (on this host thread); the caller vouches that the positions hold the same values.
struct PlanKey {
  const void* ws = nullptr;
  const int32_t* pos = nullptr;
  const int32_t* row_start = nullptr;
  hipStream_t stream = nullptr;
  int32_t B = 0, T = 0, G = 0, split = 0, nsplit = 0, zgroup = 0;
  bool direct = false;
  bool operator==(const PlanKey& o) const {
    return ws == o.ws && pos == o.pos && row_start == o.row_start && stream == o.stream && B == o.B && T == o.T &&
           G == o.G && split == o.split && nsplit == o.nsplit && direct == o.direct && zgroup == o.zgroup;
  }
};
thread_local PlanKey last_plan;

int paged_attention(const void* q, int64_t q_sb, int64_t q_st, int64_t q_sh, const fs_kv_layout* kv,
                    const int32_t* block_tables, int64_t table_stride, int32_t max_blocks, const int32_t* positions,
                    const int32_t* row_start, int32_t B, int32_t T, int32_t n_heads, float scale, void* out,
                    int64_t o_sb, int64_t o_st, int64_t o_sh, void* workspace, int64_t workspace_bytes,
                    void* stream, bool reuse_plan) {
  FS_CHECK_ARG(kv != nullptr && kv->k && kv->v, "paged_attention: null pool");
  FS_CHECK_ARG(q && block_tables && positions && out && workspace, "paged_attention: null pointer");
  FS_CHECK_ARG(B > 0 && T > 0, "paged_attention: B %d T %d", B, T);
  FS_CHECK_ARG(kv->n_kv_heads > 0 && n_heads > 0 && n_heads % kv->n_kv_heads == 0,
               "paged_attention: n_heads %d, n_kv_heads %d", n_heads, kv->n_kv_heads);
  FS_CHECK_ARG(kv->head_dim > 0 && kv->head_dim <= 256, "paged_attention: head_dim %d (max 256)", kv->head_dim);
  FS_CHECK_ARG(kv->block_size > 0 && max_blocks > 0 && table_stride >= max_blocks,
               "paged_attention: block_size %d max_blocks %d", kv->block_size, max_blocks);
  FS_CHECK_ARG(kv->num_blocks > 0, "paged_attention: num_blocks");
  FS_CHECK_ARG(kv->dtype == FS_F32 || kv->dtype == FS_BF16 || kv->dtype == FS_F16, "paged_attention: dtype %d",
               kv->dtype);
  FS_CHECK_ARG(kv->k_group == 0 || (kv->k_group > 0 && kv->k_dim == 1 && kv->head_dim % 8 == 0),
               "paged_attention: grouped keys need k_group > 0, k_dim == 1 and head_dim %% 8 == 0");
  const int64_t need = fs_paged_attention_workspace_size(B, T, n_heads, kv->head_dim, max_blocks, kv->block_size);
  FS_CHECK_ARG(workspace_bytes >= need, "paged_attention: workspace %lld < %lld bytes", (long long)workspace_bytes,
               (long long)need);
  FS_CHECK_ARG((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, "paged_attention: workspace not 256-aligned");

  AttnParams P;
  P.q = q;
  P.q_sb = q_sb;
  P.q_st = q_st;
  P.q_sh = q_sh;
  P.kv = *kv;
  P.table = block_tables;
  P.table_stride = table_stride;
  P.max_blocks = max_blocks;
  P.pos = positions;
  P.B = B;
  P.T = T;
  P.H = n_heads;
  P.G = n_heads / kv->n_kv_heads;
  P.scale_log2 = scale * LOG2E;
  const bool mfma = mfma_eligible(*kv, q, q_sb, q_st, q_sh);
  P.split = mfma ? attn_split() : GENERIC_SPLIT;
  P.nsplit = (int32_t)nsplit_for(max_blocks, kv->block_size, P.split);
  const int64_t rows = (int64_t)B * T * n_heads;
  char* ws = reinterpret_cast<char*>(workspace);
  const int64_t items = max_items(B, T, n_heads, max_blocks, kv->block_size, min_split());
  const int64_t list = (items * (int64_t)sizeof(AttnItem) + 255) / 256 * 256;
  const int64_t ns_ws = nsplit_for(max_blocks, kv->block_size, min_split());   // >= P.nsplit
  const int64_t partials = (rows * ns_ws * (kv->head_dim + 2) * (int64_t)sizeof(float) + 255) / 256 * 256;
  P.n_items = reinterpret_cast<int32_t*>(ws);
  P.split_cnt = reinterpret_cast<unsigned*>(ws + WS_COUNTERS);
  P.items = reinterpret_cast<AttnItem*>(ws + WS_HEADER);
  P.ws_acc = reinterpret_cast<float*>(ws + WS_HEADER + list);
  P.ws_ml = P.ws_acc + rows * P.nsplit * kv->head_dim;
  P.split_ws = reinterpret_cast<float*>(ws + WS_HEADER + list + partials);
  // direct outputs are stored 4 bf16 at a time
  P.direct = mfma && (reinterpret_cast<uintptr_t>(out) & 7) == 0 && o_sb % 4 == 0 && o_st % 4 == 0 && o_sh % 4 == 0;
  P.out = out;
  P.o_sb = o_sb;
  P.o_st = o_st;
  P.o_sh = o_sh;
  P.row_start = row_start;
  const int64_t qtiles = ((int64_t)T * P.G + QTILE - 1) / QTILE;
  // many query tiles per row (a prompt): groups of PF_WAVES tiles share their key/value reads
  const bool prefill = mfma && qtiles >= PF_MIN_QTILES;
  P.zgroup = prefill ? PF_WAVES : 1;

  hipStream_t st = fs::as_stream(stream);
  if (mfma) {
    const bool bs16 = kv->block_size == 16;
    // one workgroup per (plan item, KV head); items past the plan's length exit at once
    const int64_t units = (int64_t)B * ((qtiles + P.zgroup - 1) / P.zgroup) * P.nsplit * kv->n_kv_heads;
    FS_CHECK_ARG(units < 0x7fffffff, "paged_attention: %lld work units", (long long)units);
    PlanKey key;
    key.ws = workspace;
    key.pos = positions;
    key.row_start = row_start;
    key.stream = st;
    key.B = B;
    key.T = T;
    key.G = P.G;
    key.split = P.split;
    key.nsplit = P.nsplit;
    key.direct = P.direct;
    key.zgroup = P.zgroup;
    if (!(reuse_plan && last_plan == key)) {
      if (prefill) attn_plan_kernel<PLAN_THREADS_PREFILL><<<1, PLAN_THREADS_PREFILL, 0, st>>>(P);
      else attn_plan_kernel<PLAN_THREADS><<<1, PLAN_THREADS, 0, st>>>(P);
    }
    last_plan = key;
    const unsigned grid = (unsigned)units;
    if (prefill) {
      const unsigned threads = 64 * PF_WAVES;
      if (kv->head_dim == 128) {
        if (bs16) attn_prefill_kernel<128, 16><<<grid, threads, 0, st>>>(P);
        else attn_prefill_kernel<128, 0><<<grid, threads, 0, st>>>(P);
      } else {
        if (bs16) attn_prefill_kernel<64, 16><<<grid, threads, 0, st>>>(P);
        else attn_prefill_kernel<64, 0><<<grid, threads, 0, st>>>(P);
      }
    } else {
      // few, possibly long units: several workgroups each, to keep more CUs reading
      const bool two = (int64_t)T * P.G > 16;   // else no tile has a second half of query rows
      const int parts = split_parts(units, (int64_t)max_blocks * kv->block_size, two);
      const unsigned pgrid = grid * (unsigned)parts, pthreads = 64 * UNIT_WAVES / (unsigned)parts;
#define FS_ATTN_LAUNCH(D_, BS_, TWO_)                                                     \
  do {                                                                                    \
    if (parts == 4) attn_unit_part_kernel<D_, BS_, TWO_, 4><<<pgrid, pthreads, 0, st>>>(P); \
    else if (parts == 2) attn_unit_part_kernel<D_, BS_, TWO_, 2><<<pgrid, pthreads, 0, st>>>(P); \
    else attn_unit_kernel<D_, BS_, TWO_><<<grid, 64 * UNIT_WAVES, 0, st>>>(P);                   \
  } while (0)
#define FS_ATTN_LAUNCH_D(D_)                                                              \
  do {                                                                                    \
    if (bs16 && two) FS_ATTN_LAUNCH(D_, 16, true);                                        \
    else if (bs16) FS_ATTN_LAUNCH(D_, 16, false);                                         \
    else if (two) FS_ATTN_LAUNCH(D_, 0, true);                                            \
    else FS_ATTN_LAUNCH(D_, 0, false);                                                    \
  } while (0)
      if (kv->head_dim == 128) FS_ATTN_LAUNCH_D(128);
      else FS_ATTN_LAUNCH_D(64);
#undef FS_ATTN_LAUNCH_D
#undef FS_ATTN_LAUNCH
    }
  } else {
    last_plan = PlanKey{};   // no plan on this path
    dim3 grid((unsigned)rows, (unsigned)P.nsplit);
    if (f32_eligible(*kv, q, q_sb, q_st, q_sh)) {
      const int64_t tiles = (int64_t)B * (((int64_t)T * P.G + F32_ROWS - 1) / F32_ROWS) * kv->n_kv_heads;
      FS_CHECK_ARG(tiles < 0x7fffffff, "paged_attention: %lld work units", (long long)tiles);
      const dim3 fgrid((unsigned)tiles, (unsigned)P.nsplit);
      if (kv->head_dim <= 16) attn_f32_kernel<1><<<fgrid, 64, 0, st>>>(P);
      else if (kv->head_dim <= 32) attn_f32_kernel<2><<<fgrid, 64, 0, st>>>(P);
      else if (kv->head_dim <= 64) attn_f32_kernel<4><<<fgrid, 64, 0, st>>>(P);
      else attn_f32_kernel<8><<<fgrid, 64, 0, st>>>(P);
      if (int e = fs::launch_status("paged_attention")) return e;
      if (P.nsplit == 1) return 0;   // every output is written
    } else switch (kv->dtype) {
      case FS_F32: attn_generic_kernel<FS_F32><<<grid, 64, 0, st>>>(P); break;
      case FS_BF16: attn_generic_kernel<FS_BF16><<<grid, 64, 0, st>>>(P); break;
      default: attn_generic_kernel<FS_F16><<<grid, 64, 0, st>>>(P); break;
    }
  }
  if (int e = fs::launch_status("paged_attention")) return e;
  if (P.direct && P.nsplit == 1) return 0;   // every query sees one chunk: all outputs are written
  dim3 cgrid((unsigned)((rows + COMBINE_ROWS - 1) / COMBINE_ROWS));
  switch (kv->dtype) {
    case FS_F32: attn_combine_kernel<FS_F32><<<cgrid, 64 * COMBINE_ROWS, 0, st>>>(P, out, o_sb, o_st, o_sh); break;
    case FS_BF16: attn_combine_kernel<FS_BF16><<<cgrid, 64 * COMBINE_ROWS, 0, st>>>(P, out, o_sb, o_st, o_sh); break;
    default: attn_combine_kernel<FS_F16><<<cgrid, 64 * COMBINE_ROWS, 0, st>>>(P, out, o_sb, o_st, o_sh); break;
  }
  return fs::launch_status("paged_attention_combine");
}
}  // namespace

extern "C" int fs_paged_attention(const void* q, int64_t q_sb, int64_t q_st, int64_t q_sh, const fs_kv_layout* kv,
                                  const int32_t* block_tables, int64_t table_stride, int32_t max_blocks,
                                  const int32_t* positions, int32_t B, int32_t T, int32_t n_heads, float scale,
                                  void* out, int64_t o_sb, int64_t o_st, int64_t o_sh, void* workspace,
                                  int64_t workspace_bytes, void* stream) {
  return paged_attention(q, q_sb, q_st, q_sh, kv, block_tables, table_stride, max_blocks, positions, nullptr, B, T,
                         n_heads, scale, out, o_sb, o_st, o_sh, workspace, workspace_bytes, stream, false);
}

extern "C" int fs_paged_attention_reuse_plan(const void* q, int64_t q_sb, int64_t q_st, int64_t q_sh,
                                             const fs_kv_layout* kv, const int32_t* block_tables,
                                             int64_t table_stride, int32_t max_blocks, const int32_t* positions,
                                             int32_t B, int32_t T, int32_t n_heads, float scale, void* out,
                                             int64_t o_sb, int64_t o_st, int64_t o_sh, void* workspace,
                                             int64_t workspace_bytes, void* stream) {
  return paged_attention(q, q_sb, q_st, q_sh, kv, block_tables, table_stride, max_blocks, positions, nullptr, B, T,
                         n_heads, scale, out, o_sb, o_st, o_sh, workspace, workspace_bytes, stream, true);
}

extern "C" int fs_paged_attention_varlen(const void* q, int64_t q_st, int64_t q_sh, const fs_kv_layout* kv,
                                         const int32_t* block_tables, int64_t table_stride, int32_t max_blocks,
                                         const int32_t* positions, const int32_t* cu_seqlens, int32_t S,
                                         int32_t T, int32_t n_heads, float scale, void* out, int64_t o_st,
                                         int64_t o_sh, void* workspace, int64_t workspace_bytes, void* stream) {
  FS_CHECK_ARG(cu_seqlens, "paged_attention_varlen: null cu_seqlens");
  return paged_attention(q, 0, q_st, q_sh, kv, block_tables, table_stride, max_blocks, positions, cu_seqlens, S, T,
                         n_heads, scale, out, 0, o_st, o_sh, workspace, workspace_bytes, stream, false);
}

extern "C" int fs_paged_attention_varlen_reuse_plan(const void* q, int64_t q_st, int64_t q_sh,
                                                    const fs_kv_layout* kv, const int32_t* block_tables,
                                                    int64_t table_stride, int32_t max_blocks,
                                                    const int32_t* positions, const int32_t* cu_seqlens, int32_t S,
                                                    int32_t T, int32_t n_heads, float scale, void* out,
                                                    int64_t o_st, int64_t o_sh, void* workspace,
                                                    int64_t workspace_bytes, void* stream) {
  FS_CHECK_ARG(cu_seqlens, "paged_attention_varlen: null cu_seqlens");
  return paged_attention(q, 0, q_st, q_sh, kv, block_tables, table_stride, max_blocks, positions, cu_seqlens, S, T,
                         n_heads, scale, out, 0, o_st, o_sh, workspace, workspace_bytes, stream, true);
}
