// Block-sparse causal attention over per-token page plans.
//
// Contract: infllmv2_attn_varlen_func(..., topk_idx=)
// (third_party/infllmv2/paper1.patch:1993-2100; called from
// leanselect/models/minicpm.py:3216-3244): for query row t and KV group g the
// keys are those of the valid ids in topk_idx[g, t, :] (each page once) with
// j <= t + len_k - len_q when causal; all H/G heads of the group share the plan.
//
// Design (one workgroup per 8, 12 or 24 query rows of one KV group and 16-head tile):
//   * the plan rows are turned into an ascending, duplicate-free page list
//     through an LDS table of row masks (ids past the causal frontier are dropped);
//   * S^T = K . Q^T on v_mfma_f32_16x16x32: keys are MFMA rows, the 16 heads of
//     the group are columns, so each lane owns one head and the online-softmax
//     row statistics need only two cross-lane steps;
//   * K rows are permuted inside each 32-key chunk so that lane group q ends up
//     with the 8 contiguous keys base+8q..base+8q+7; P^T then feeds the second
//     MFMA (O^T = V^T . P^T) straight from registers as its B operand and V^T
//     is read as 16-byte rows of a transposed, page-aligned copy of V built by
//     ls_kv_stage_kernel (zero-filled past each sequence end);
//   * float32 softmax in base 2; P . V runs on the fp16 MFMA (P in [0, 1]
//     keeps 10 mantissa bits instead of bf16's 7; V is staged to fp16 with an
//     exact per-page power-of-two scale that moves onto P), output rounded once.
#include "ls_common.h"

#include <mutex>
#include <type_traits>

// Work-item and workgroup ids straight from the hardware: this file is built
// without IEEE NaN quieting, and the device library's id helpers (built with
// it) would then stay out-of-line calls.
#define LS_TID ((int)__builtin_amdgcn_workitem_id_x())
#define LS_BID_X ((int)__builtin_amdgcn_workgroup_id_x())
#define LS_BID_Y ((int)__builtin_amdgcn_workgroup_id_y())
#define LS_BID_Z ((int)__builtin_amdgcn_workgroup_id_z())

#define LS_ATTN_MAX_PAGES 8192
#define LS_ATTN_MAX_TAKE 128
#define LS_ATTN_RING_TIMEOUT 1  // status bit: a ring wait expired (outputs invalid)

// pg_off[b] = sum_{b' < b} ceil(len_k(b') / 64): page-aligned start of each
// sequence in the transposed V copy (in pages); tile_off[b] = sum_{b' < b}
// ceil(len_q(b') / tile): first row tile of each sequence; tok[i] = i for
// i < n_tok (the ready tokens the tile kernel's copies deliver); *status = 0
// (the tile kernel ORs in LS_ATTN_RING_TIMEOUT when a ring wait expires).
__global__ void ls_attn_plan_kernel(const int32_t* __restrict__ cu_q,
                                    const int32_t* __restrict__ cu_k, int batch, int tile,
                                    int32_t* __restrict__ pg_off, int32_t* __restrict__ tile_off,
                                    int32_t* __restrict__ tok, int n_tok,
                                    int32_t* __restrict__ status) {
  if (LS_BID_X != 0) return;
  for (int i = LS_TID; i < n_tok; i += 64) tok[i] = i;
  if (LS_TID != 0) return;
  *status = 0;
  int32_t acc = 0, acc_t = 0;
  pg_off[0] = 0;
  tile_off[0] = 0;
  for (int b = 0; b < batch; ++b) {
    const int len = cu_k[b + 1] - cu_k[b];
    acc += len > 0 ? (len + 63) / 64 : 0;
    pg_off[b + 1] = acc;
    const int lq = cu_q[b + 1] - cu_q[b];
    acc_t += lq > 0 ? (lq + tile - 1) / tile : 0;
    tile_off[b + 1] = acc_t;
  }
}

// Writes 0 to a caller's status word (a kernel rather than a memset, so that
// the call stays safe to capture in a graph).
__global__ void ls_attn_status_clear_kernel(int32_t* __restrict__ status) {
  if (LS_BID_X == 0 && LS_TID == 0) *status = 0;
}

// ---------------------------------------------------------------------------
// Tile kernel: one workgroup = 8, 12 or 24 consecutive query rows of one sequence
// and one KV group for 16 of its query heads (8 waves of up to TPW rows, two waves
// per SIMD; the launcher picks TPW).  The rows' page plans are OR-ed into a union page list;
// each union page of staged K and V^T is streamed once into a 4-stage LDS ring
// with direct global->LDS loads, and every row that selected the page runs its
// MFMAs on it.  Rows that did not select a page skip it (no masked-out work).
// A wave keeps its rows' O^T accumulators (TPW x 8 x 4 floats per lane) and
// Q^T fragments in registers.  Larger tiles share each page copy among more
// rows; three rows of O and Q are what the register file holds at two waves per
// SIMD (254 to 256 registers; the chunk's K and V^T fragments are read once for all
// rows).
// ---------------------------------------------------------------------------
#ifndef LS_ATT_WAVES
#define LS_ATT_WAVES 8                       // waves per workgroup
#endif
#define LS_ATT_THREADS (64 * LS_ATT_WAVES)
#define LS_ATT_STAGES 4
#define LS_ATT_KBYTES (64 * 256)             // K page: 64 rows x 256 B
#define LS_ATT_STAGE_BYTES (2 * LS_ATT_KBYTES)  // + V^T page: 128 rows x 128 B
#ifndef LS_ATT_SHARE_STRIDED
#define LS_ATT_SHARE_STRIDED 25              // plan ids per union page (x10) for the strided order
#endif
#ifndef LS_ATT_SPIN_SLEEP
#define LS_ATT_SPIN_SLEEP 1                  // s_sleep units between a waiting wave's polls
#endif
#define LS_ATT_UNION_CAP 4096                // union pages of a tile (ready tokens in the workspace)

// Tile geometry for at most TPW rows per wave: rows per tile, each wave's rows,
// the most ids per row it accepts (so that its union fits LS_ATT_UNION_CAP) and
// the union bound.  Tiles have 8, 12 or 24 rows: with TPW = 2 the first half of the
// waves has two rows and the other half one, three on every SIMD (waves w and w + 4
// share one).
//
// A row's pages are visited in the order that the plans of the 24 rows around it
// give (rows 24 i .. 24 i + 23 of the sequence, the group of rows, which holds
// whole tiles of each height).  So a row's sums, and with them its output, are bit
// for bit the same whichever height the launcher takes: they don't depend on what
// else is packed into the call.  (Tiles of 16 rows would straddle two groups, with
// both groups' orders to form and pages copied for each: 197 us for 4096 rows,
// where 24-row tiles take 205.)
#define LS_ATT_GROUP 24
template <int TPW>
struct LsAttTile {
  static constexpr int kTile = TPW == 2 ? 12 : LS_ATT_WAVES * TPW;
  static constexpr int kMaxTake =
      LS_ATTN_MAX_TAKE < LS_ATT_UNION_CAP / kTile ? LS_ATTN_MAX_TAKE : LS_ATT_UNION_CAP / kTile;
  static constexpr int kMaxUnion = kTile * kMaxTake;
  __host__ __device__ static constexpr int rows(int w) {
    return TPW == 2 && w >= LS_ATT_WAVES / 2 ? 1 : TPW;
  }
  __host__ __device__ static constexpr int row0(int w) {
    return TPW == 2 && w >= LS_ATT_WAVES / 2 ? w + LS_ATT_WAVES / 2 : w * TPW;
  }
  static_assert(LS_ATT_WAVES == 8 && row0(LS_ATT_WAVES - 1) + rows(LS_ATT_WAVES - 1) == kTile,
                "the waves' rows make up the tile");
  static_assert(kTile <= LS_ATT_GROUP && LS_ATT_GROUP % kTile == 0 && LS_ATT_GROUP <= 32,
                "a group holds whole tiles, and its row masks are 32-bit");
  static_assert(kMaxUnion <= LS_ATT_UNION_CAP, "one ready token per union page");
};

typedef _Float16 ls_half2 __attribute__((ext_vector_type(2)));
typedef float ls_float2 __attribute__((ext_vector_type(2)));

// LDS row of key j (0..63) of a page: inside each 32-key chunk, MFMA row r of
// key block nb holds key 8*(r/4) + 4*nb + r%4, so storing that key at row
// 16*nb + r makes the 16 rows an MFMA reads consecutive, while lane group q
// still ends up with the keys 8q..8q+7 of the chunk.
__device__ __forceinline__ int ls_att_key_of_row(int row) {
  const int c = row >> 5, rr = row & 31, nb = rr >> 4, r = rr & 15;
  return 32 * c + 8 * (r >> 2) + 4 * nb + (r & 3);
}

// Page-major staging of K and V in the ring's own byte order: block
// kv[g][pg_off[b] + p] (LS_ATT_STAGE_BYTES) holds page p of sequence b, group
// g, exactly as a ring stage holds it, so a page copy is one contiguous
// 32 KB transfer:
//  - bytes [0, 16K): K, 64 rows of 256 B; row R holds key ls_att_key_of_row(R)
//    of the page, its 16-byte chunk C (dims 8C..8C+7) at position C ^ (R & 15);
//  - bytes [16K, 32K): V^T, 128 rows of 128 B; row d holds fp16(v[key][d] * 2^-e)
//    of the page's 64 keys, chunk C (keys 8C..8C+7) at position C ^ ((d >> 1) & 7).
// Keys past the sequence end are zero (their scores are always masked).
// vexp[g * n_pages + pg_off[b] + p] = e: the smallest e >= 0 (at most 15) that
// keeps the page's scaled V within +-32768, so it is finite in fp16 (e = 0 for
// ordinary activations; bf16 values are then exact in fp16 down to 2^-14).
// One workgroup stages one page of one group (V^T goes through LDS).
template <int DT>
__global__ __launch_bounds__(256) void ls_kv_stage_kernel(
    const uint16_t* __restrict__ k, int64_t k_rs, const uint16_t* __restrict__ v, int64_t v_rs,
    const int32_t* __restrict__ cu_k, const int32_t* __restrict__ pg_off, int batch,
    int64_t n_pages, uint8_t* __restrict__ kv, int32_t* __restrict__ vexp) {
  constexpr int D = 128, PITCH = D + 2, CH = D / 8;
  __shared__ uint16_t tile[64 * PITCH];
  __shared__ float wave_max[4];
  const int64_t tile_id = LS_BID_X;
  if (tile_id >= pg_off[batch]) return;
  const int g = LS_BID_Y;
  const int b = ls_find_segment(pg_off, batch, tile_id);
  const int p = (int)(tile_id - pg_off[b]);
  const int lk = cu_k[b + 1] - cu_k[b];
  const int64_t krow0 = (int64_t)cu_k[b] + 64LL * p;
  uint8_t* blk = kv + ((int64_t)g * n_pages + pg_off[b] + p) * LS_ATT_STAGE_BYTES;
  // K: output chunk o = 16 R + position.
  for (int o = LS_TID; o < 64 * CH; o += 256) {
    const int R = o >> 4, C = (o & 15) ^ (R & 15);
    const int key = ls_att_key_of_row(R);
    ls_u32x4 val = {0u, 0u, 0u, 0u};
    if (64 * p + key < lk) val = ls_load16(k + (krow0 + key) * k_rs + (int64_t)g * D + 8 * C);
    *reinterpret_cast<ls_u32x4*>(blk + 16 * o) = val;
  }
  // V through LDS, then V^T rows.
  float mx = 0.f;
  for (int c = LS_TID; c < 64 * CH; c += 256) {
    const int key = c / CH, d0 = (c % CH) * 8;
    ls_u32x4 val = {0u, 0u, 0u, 0u};
    if (64 * p + key < lk) val = ls_load16(v + (krow0 + key) * v_rs + (int64_t)g * D + d0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint16_t lo = (uint16_t)(val[i] & 0xffffu), hi = (uint16_t)(val[i] >> 16);
      mx = fmaxf(mx, fmaxf(fabsf(LsElem<DT>::to_f(lo)), fabsf(LsElem<DT>::to_f(hi))));
      tile[key * PITCH + d0 + 2 * i] = lo;
      tile[key * PITCH + d0 + 2 * i + 1] = hi;
    }
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, LS_WAVE));
  if ((LS_TID & 63) == 0) wave_max[LS_TID >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
  int e = 0;
  while (e < 15 && mx * __builtin_ldexpf(1.f, -e) > 32768.f) ++e;
  const float scale = __builtin_ldexpf(1.f, -e);
  if (LS_TID == 0) vexp[(int64_t)g * n_pages + pg_off[b] + p] = e;
  uint8_t* vblk = blk + LS_ATT_KBYTES;
  for (int c = LS_TID; c < D * 8; c += 256) {
    const int d = c / 8, k0 = (c % 8) * 8;
    ls_u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = ls_pack2(ls_f32_to_f16(LsElem<DT>::to_f(tile[(k0 + 2 * i) * PITCH + d]) * scale),
                      ls_f32_to_f16(LsElem<DT>::to_f(tile[(k0 + 2 * i + 1) * PITCH + d]) * scale));
    *reinterpret_cast<ls_u32x4*>(vblk + d * 128 + 16 * ((c % 8) ^ ((d >> 1) & 7))) = o;
  }
}




// Two float32 -> one packed fp16 pair (round to nearest even).
__device__ __forceinline__ uint32_t ls_pack_f16x2(float a, float b) {
  const ls_half2 h = __builtin_convertvector((ls_float2){a, b}, ls_half2);
  return __builtin_bit_cast(uint32_t, h);
}

// acc + lo(x) + hi(x) for a packed fp16 pair, in float32.
__device__ __forceinline__ float ls_sum_f16x2(uint32_t x, float acc) {
  const ls_half2 one = {(_Float16)1.0f, (_Float16)1.0f};
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(ls_half2, x), one, acc, false);
}


// What bounds it.  At two waves per SIMD the chunk math is a latency chain, not
// an issue limit: a probe of the same instruction mix (16 MFMAs, 8 exponentials,
// 24 other vector instructions) takes 150 ns per row-chunk with two waves, the
// kernel took 245.  So the loop keeps a wave's waits off that chain: V^T is read
// from LDS before the first row's Q K (and once for all rows), the second chunk's
// K behind the first's softmax, the visit list and the ready word ahead of their
// use, and the rare branches (causal frontier, rescale) out of line.  This kernel
// alone, one box, before -> now: 13.67 -> 12.16 ms (one 128K sequence, 64 pages),
// 3.99 -> 3.33 ms (32K, 96 pages, few shared), 3.28 -> 2.77 ms (32K with BIAS), 275
// -> 186 us (4096 rows), 82 -> 38 us (1337 rows, 8-row tiles).
// BIAS adds a per-key score bias (the NOSA eviction score, pre-scaled to base
// 2): weight_j = 2^(scale_log2 * q.k_j + cb_j).  cb[g][64 pg_off[b] + j] is
// staged like V^T and copied with each page (256 B per stage).
template <int DT, bool BIAS, int TPW>
__global__ __launch_bounds__(LS_ATT_THREADS, LS_ATT_THREADS / 256) void ls_attn_tile_kernel(
    const uint16_t* __restrict__ qg, int64_t q_rs, const uint8_t* __restrict__ kv, int64_t lpad,
    const int32_t* __restrict__ vexp, const float* __restrict__ cb,
    const int32_t* __restrict__ tok, int64_t n_pages_ws,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ cu_k,
    const int32_t* __restrict__ pg_off, const int32_t* __restrict__ tile_off, int batch,
    int64_t total_q, int G, int gs, const int32_t* __restrict__ topk_idx, int take,
    float scale_log2, int causal, uint16_t* __restrict__ out, float* __restrict__ lse,
    int run, int span, int per_xcd, int32_t* __restrict__ status, int spin_limit) {
  constexpr int D = 128;
  constexpr int TILE = LsAttTile<TPW>::kTile;
  constexpr int MAX_UNION = LsAttTile<TPW>::kMaxUnion;
  constexpr int MAX_VISITS = TPW * LsAttTile<TPW>::kMaxTake;  // pages of one wave
  constexpr int GROUP = LS_ATT_GROUP, GROUP_RPW = GROUP / LS_ATT_WAVES;
  constexpr int MAX_ORDER = GROUP * LsAttTile<TPW>::kMaxTake;  // pages of a group
  constexpr uint32_t TILE_MASK = (1u << TILE) - 1u;
  // The setup tables (rows per page, the group's pages in visit order) are only
  // needed before streaming starts and share their LDS with the ring.
  __shared__ __align__(16) uint8_t s_ring[LS_ATT_STAGES * LS_ATT_STAGE_BYTES];
  uint32_t* s_rows = reinterpret_cast<uint32_t*>(s_ring);  // [page]: mask of the group rows on it
  uint32_t* s_omask = s_rows + LS_ATTN_MAX_PAGES;          // [place in the order]: the same mask
  uint16_t* s_opage = reinterpret_cast<uint16_t*>(s_omask + MAX_ORDER);  // and the page
  // The tile's own pages, the union, in that order.
  __shared__ uint16_t s_upage[MAX_UNION];
  __shared__ uint8_t s_uneed[MAX_UNION];  // waves with a row on the page
  // The pages of each wave in the order it visits them: page | its rows on it
  // << 13 | union index << 16.
  __shared__ uint32_t s_wlist[LS_ATT_WAVES][MAX_VISITS];
  __shared__ int s_wsum[LS_ATT_WAVES];
  // Ring protocol: s_next = next union page to be claimed for copying;
  // s_rdy[st][0] = union index + 1 of the page whose copy into stage st has
  // landed, s_rdy[st][1] = that page's V exponent (read together); s_done[st] =
  // (union index << 8) | number of its waves done with it, for the page in stage
  // st (tagged, so a stale count never matches).
  __shared__ uint32_t s_next, s_done[LS_ATT_STAGES];
  __shared__ __align__(8) uint32_t s_rdy[LS_ATT_STAGES][2];
  __shared__ __align__(16) float s_bias[BIAS ? LS_ATT_STAGES * 64 : 4];
  static_assert(LS_ATTN_MAX_PAGES * 4 + MAX_ORDER * 6 <= LS_ATT_STAGES * LS_ATT_STAGE_BYTES,
                "the setup tables must fit in the ring");
  static_assert(GROUP % LS_ATT_WAVES == 0, "each wave takes part in the setup alike");
  static_assert(LS_ATTN_MAX_PAGES <= 1 << 13 && TPW <= 3 && MAX_UNION <= 1 << 16,
                "fields of a visit entry");

  const int tid = LS_TID;
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  // This wave's rows of the tile: n_mine from row w0 on.
  const int w0 = LsAttTile<TPW>::row0(w), n_mine = LsAttTile<TPW>::rows(w);
  const uint32_t rows_mask = (1u << n_mine) - 1u;

  // XCD-aware tile order.  The grid is 8 * per_xcd workgroups by the KV groups,
  // numbered as they are started, x first; consecutive workgroups land on different
  // XCDs (workgroup i runs on XCD i % 8).  Each XCD takes runs of `run` consecutive
  // tiles, so the tiles in flight on one XCD are neighbours that share pages in
  // its L2, and turns to the next KV group every `span` tiles (a multiple of
  // run).  The runs are dealt over the XCDs there and back (0..7, then 7..0), and
  // from the end of the sequence first, so every XCD gets an even share of late
  // (large-union) and early (small-union) rows, the largest tiles start first and
  // small ones fill the tail.  per_xcd is a multiple of span, so this is a
  // permutation of the workgroups.
  const int xcd = LS_BID_X % 8;
  const uint32_t xi = (uint32_t)LS_BID_Y * (uint32_t)per_xcd + (uint32_t)(LS_BID_X / 8);
  const uint32_t turn = xi / (uint32_t)span;
  const int g = (int)(turn % (uint32_t)G);
  const int at = (int)(turn / (uint32_t)G * (uint32_t)span + xi % (uint32_t)span);
  const int deal = at / run;
  const int64_t tile = 8LL * per_xcd - 1 -
                       ((int64_t)(8 * deal + ((deal & 1) ? 7 - xcd : xcd)) * run + at % run);
  if (tile >= tile_off[batch]) return;
  const int head = LS_BID_Z * 16 + r;
  const bool head_ok = head < gs;

  const int b = ls_find_segment(tile_off, batch, tile);
  const int64_t t0 = (int64_t)cu_q[b] + TILE * (tile - tile_off[b]);
  const int n_rows = (int)min((int64_t)TILE, (int64_t)cu_q[b + 1] - t0);
  const int lq = cu_q[b + 1] - cu_q[b];
  const int lk = cu_k[b + 1] - cu_k[b];
  const int64_t vbase = 64LL * pg_off[b];
  const int64_t tr0 = t0 - cu_q[b];
  // The tile's group: rows gr0 .. gr0 + n_grp - 1 of the sequence, the tile's from `off` on.
  const int64_t gr0 = tr0 / GROUP * GROUP;
  const int off = (int)(tr0 - gr0);
  const int n_grp = (int)min((int64_t)GROUP, (int64_t)lq - gr0);
  // Keys visible to row i of the group: j <= jmax(i) (the last row sees the most).
  auto row_jmax = [&](int i) -> int64_t {
    int64_t jm = lk - 1;
    if (causal) jm = min(jm, gr0 + i + (int64_t)(lk - lq));
    return jm;
  };
  const int64_t group_jmax = row_jmax(n_grp - 1);
  const int last_page =
      group_jmax >= 0 ? (int)min(group_jmax / 64, (int64_t)LS_ATTN_MAX_PAGES - 1) : -1;

  // ---- per-row state: Q^T fragments (B operand), softmax stats, O^T ----
  // (the Q loads are issued first; they land while the page list is built)
  ls_u32x4 qf[TPW][4];
  // m_run: running maximum in base-2 units (score * scale_log2).  The score above
  // which a key would exceed it by more than 2^8 is formed from it for each chunk:
  // the maximum formed from that score instead would be rounded once more, and so
  // would the lse.
  float m_run[TPW], l_run[TPW];
  int jmax_r[TPW];
  ls_f32x4 o[TPW][8];
#pragma unroll
  for (int j = 0; j < TPW; ++j) {
    const int row = w0 + j;
    const int64_t t = t0 + min(row, n_rows - 1);
    const uint16_t* qrow = qg + t * q_rs + ((int64_t)g * gs + (head_ok ? head : 0)) * D + 8 * q;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      qf[j][ks] = ls_load16(qrow + 32 * ks);
      if (!head_ok) qf[j][ks] = ls_u32x4{0u, 0u, 0u, 0u};
    }
    l_run[j] = 0.f;
    m_run[j] = -INFINITY;
    // Wave-uniform, so each chunk's row mask below is scalar work.
    jmax_r[j] = __builtin_amdgcn_readfirstlane(j < n_mine && row < n_rows ? (int)row_jmax(off + row) : -1);
#pragma unroll
    for (int db = 0; db < 8; ++db) o[j][db] = ls_f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // ---- the group's pages: rows per page, then their order, then the tile's among them ----
  // Every step works on 64 pages or ids per wave at a time: the tile's setup
  // is exposed (one workgroup fills a CU's LDS), so it must not loop serially
  // over a word's bits or a thread's pages.
  for (int i = tid; i <= last_page; i += LS_ATT_THREADS) s_rows[i] = 0u;
  if (tid < LS_ATT_STAGES) {
    s_rdy[tid][0] = 0u;
    s_done[tid] = 0u;
  }
  if (tid == 0) s_next = LS_ATT_STAGES;  // pages 0..3 are copied at the start
  __syncthreads();
  if (last_page >= 0) {
    const int32_t* ids = topk_idx + ((int64_t)g * total_q + cu_q[b] + gr0) * take;
#pragma unroll
    for (int j = 0; j < GROUP_RPW; ++j) {
      const int row = w * GROUP_RPW + j;
      const int jm = __builtin_amdgcn_readfirstlane((int)row_jmax(row));
      const int pmax = jm >= 0 ? min(jm / 64, last_page) : -1;
      if (row < n_grp)
        for (int i = lane; i < take; i += 64) {
          const int p = ids[(int64_t)row * take + i];
          if (p >= 0 && p <= pmax) atomicOr(&s_rows[p], 1u << row);
        }
    }
  }
  __syncthreads();
  // Wave w counts, then places, the pages [w, w + 1) * seg64 of 64-page segments.
  const int n_seg = (last_page + 64) / 64, seg_per = (n_seg + LS_ATT_WAVES - 1) / LS_ATT_WAVES;
  const int seg0 = w * seg_per, seg1 = min(n_seg, seg0 + seg_per);
  int wave_pages = 0;
  for (int sg = seg0; sg < seg1; ++sg) {
    const int p = 64 * sg + lane;
    wave_pages += __popcll(__ballot(p <= last_page && s_rows[p] != 0u));
  }
  if (lane == 0) s_wsum[w] = wave_pages;
  __syncthreads();
  int pos0 = 0, n_order = 0;
#pragma unroll
  for (int i = 0; i < LS_ATT_WAVES; ++i) {
    const int c = s_wsum[i];
    pos0 += i < w ? c : 0;
    n_order += c;
  }
  pos0 = __builtin_amdgcn_readfirstlane(pos0);
  n_order = __builtin_amdgcn_readfirstlane(n_order);
  const int32_t* vexp_seq = vexp + (int64_t)g * n_pages_ws + pg_off[b];
  // Wave-uniform floats are kept in scalar registers: with three rows of O and Q,
  // the chunk's K and V^T fragments and a row's scores no vector register is spare.
  auto uniform_f = [](float x) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(x)));
  };
  const float inv_scale_log2 = uniform_f(1.f / scale_log2);
  // Page order.  Where the group's rows share many pages (at least
  // LS_ATT_SHARE_STRIDED / 10 plan ids per page) the pages are visited in
  // a strided order (ascending page i goes to place i * stride mod n_order, a
  // bijection for stride coprime to n_order): neighbouring pages tend to be
  // selected by the same rows, and spreading them out evens the work of the
  // waves over any window of pages.  Where they share few, ascending order:
  // the tiles running side by side on an XCD then reach a shared page at
  // nearly the same time, while it is still in that XCD's L2, and the waves'
  // work is even anyway.  The stride is the first odd number from 7 on that is
  // coprime to n_order: 7, else 9, 11, 13 (15 shares the 3 that ruled 9 out),
  // else 17 (a length that 3, 7, 11 and 13 divide is 3003 pages).
  static_assert(MAX_ORDER < 2 * 3003, "17 is coprime to a length that rules out the others");
  int stride = 1;
  if (n_order > 1 && 10 * n_grp * take >= LS_ATT_SHARE_STRIDED * n_order)
    stride = n_order % 7 ? 7 : n_order % 3 ? 9 : n_order % 11 ? 11 : n_order % 13 ? 13 : 17;
  for (int sg = seg0; sg < seg1; ++sg) {
    const int page = 64 * sg + lane;
    const uint32_t rows = page <= last_page ? s_rows[page] : 0u;
    const uint64_t mk = __ballot(rows != 0u);
    const int pos = (int)__builtin_amdgcn_mbcnt_hi(
        (uint32_t)(mk >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mk, (uint32_t)pos0));
    if (rows != 0u) {
      const int dst = (int)(((uint32_t)pos * (uint32_t)stride) % (uint32_t)n_order);
      s_omask[dst] = rows;
      s_opage[dst] = (uint16_t)page;
    }
    pos0 += __popcll(mk);
  }
  __syncthreads();
  // The tile's pages of the order are its union; every wave finds their places
  // there (the waves take turns to write them down) and its own pages among them.
  int n_union = 0, n_visits = 0;
  for (int u0 = 0; u0 < n_order; u0 += 64) {
    const int u = u0 + lane;
    const uint32_t rows = u < n_order ? (s_omask[u] >> off) & TILE_MASK : 0u;
    const uint32_t mine = (rows >> w0) & rows_mask;
    const uint64_t tk = __ballot(rows != 0u), mk = __ballot(mine != 0u);
    const int ui = (int)__builtin_amdgcn_mbcnt_hi(
        (uint32_t)(tk >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)tk, (uint32_t)n_union));
    const int pos = (int)__builtin_amdgcn_mbcnt_hi(
        (uint32_t)(mk >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mk, (uint32_t)n_visits));
    const int page = u < n_order ? (int)s_opage[u] : 0;
    if (mine != 0u) s_wlist[w][pos] = (uint32_t)page | mine << 13 | (uint32_t)ui << 16;
    if ((u0 / 64) % LS_ATT_WAVES == w && rows != 0u) {
      int n_waves = 0;
#pragma unroll
      for (int i = 0; i < LS_ATT_WAVES; ++i)
        n_waves += ((rows >> LsAttTile<TPW>::row0(i)) & ((1u << LsAttTile<TPW>::rows(i)) - 1u)) != 0u;
      s_upage[ui] = (uint16_t)page;
      s_uneed[ui] = (uint8_t)n_waves;
    }
    n_union += __popcll(tk);
    n_visits += __popcll(mk);
  }
  __syncthreads();  // the lists are complete and the tables are dead, so the
                    // ring may be written
  LS_WAIT_VMCNT(0);

  // ---- staging ----
  // One wave copies a whole union page into its stage: the page's staged
  // block (K rows with chunk C of row R at position C ^ (R & 15), V^T rows
  // with chunk C of row d at C ^ ((d >> 1) & 7), so the sixteen lanes of an
  // MFMA operand read hit sixteen distinct bank groups) is copied byte for
  // byte, 1 KB per load (lane l -> byte 16 l).
  //
  // Waves are not kept in lockstep, and a wave visits only the pages its rows
  // selected, waiting only for the page it is about to read.  Union page u
  // goes to stage u % 4.  The copies of pages 0..3 are issued at the start.
  // A waiting wave claims the next unclaimed page (at most three ahead of the
  // page it waits for) once every wave with rows on the stage's previous page
  // is done with it, issues its copy and goes back to waiting without
  // waiting for the copy: the copy's final load brings the page's token
  // (union index + 1) from global memory into s_rdy[stage][0], and a wave's
  // loads land in issue order, so the token lands after the page's K, V^T and
  // bias.  Computing waves never copy (the last wave on a page is often the
  // slowest one).  A page's copy depends only on earlier pages being
  // finished, so every wait ends.
  const uint8_t* kvgrp = kv + ((int64_t)g * n_pages_ws + pg_off[b]) * LS_ATT_STAGE_BYTES;
  const float* cgrp = BIAS ? cb + (int64_t)g * lpad + vbase : nullptr;
  const uint32_t ring_off = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(ls_lds_void*)s_ring);
  auto issue_page = [&](int ui_copy) {
    const int page = __builtin_amdgcn_readfirstlane((int)s_upage[ui_copy]);
    const uint32_t kb = ring_off + (ui_copy % LS_ATT_STAGES) * LS_ATT_STAGE_BYTES;
    // The staged page is the stage's byte image: 32 contiguous 1 KB copies.
    const uint8_t* src = kvgrp + (int64_t)page * LS_ATT_STAGE_BYTES;
#pragma unroll
    for (int i = 0; i < LS_ATT_STAGE_BYTES / 1024; ++i)
      ls_dma16(src + 1024 * i, 16u * (uint32_t)lane, kb + i * 1024);
    // The page's 64 biases (lanes 0..15, 16 bytes each).
    if constexpr (BIAS)
      if (lane < 16)
        ls_dma16(cgrp + 64LL * page, 16u * (uint32_t)lane,
                 (uint32_t)(uintptr_t)(ls_lds_void*)s_bias + (ui_copy % LS_ATT_STAGES) * 256u);
    // The page's V exponent, then last the ready token ui_copy + 1 (lane 0 only).
    if (lane == 0) {
      ls_dma4(vexp_seq + page, 0u,
              (uint32_t)(uintptr_t)(ls_lds_void*)&s_rdy[ui_copy % LS_ATT_STAGES][1]);
      ls_dma4(tok + ui_copy + 1, 0u,
              (uint32_t)(uintptr_t)(ls_lds_void*)&s_rdy[ui_copy % LS_ATT_STAGES][0]);
    }
  };
  // Hands stage u % 4 to page u (its waves count from zero) and copies it.
  auto issue_copy = [&](int u) {
    if (lane == 0)
      __hip_atomic_store(&s_done[u % LS_ATT_STAGES], (uint32_t)u << 8, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_WORKGROUP);
    LS_WAIT_LGKMCNT0();  // the count is reset before the token can land
    issue_page(u);
  };
  // A waiting wave at page ui claims and copies page s_next when its stage is free.
  auto try_claim = [&](int ui) {
    const int nx = __builtin_amdgcn_readfirstlane(
        (int)__hip_atomic_load(&s_next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
    if (nx >= n_union || nx > ui + LS_ATT_STAGES - 1) return false;
    const int prev = nx - LS_ATT_STAGES;  // >= 0: pages 0..3 are copied at the start
    const uint32_t want = ((uint32_t)prev << 8) | (uint32_t)s_uneed[prev];
    if ((uint32_t)__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(
            &s_done[nx % LS_ATT_STAGES], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP)) != want)
      return false;  // a wave may still read the stage's previous page
    int won = 0;
    if (lane == 0) {
      uint32_t expect = (uint32_t)nx;
      won = __hip_atomic_compare_exchange_strong(&s_next, &expect, (uint32_t)nx + 1u,
                                                 __ATOMIC_ACQ_REL, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (!__builtin_amdgcn_readfirstlane(won)) return false;
    issue_copy(nx);
    return true;
  };
  if (w < LS_ATT_STAGES && w < n_union) issue_copy(w);
  // The ready token (low word) and V exponent (high word) of union page ui's
  // stage, read in one access: the exponent lands before the token, so a
  // read that sees the token sees the page's exponent.
  auto stage_word = [&](int ui) -> uint64_t {
    return __hip_atomic_load(reinterpret_cast<uint64_t*>(&s_rdy[ui % LS_ATT_STAGES][0]),
                             __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto is_ready = [&](int ui, uint64_t word) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)word) == (uint32_t)ui + 1u;
  };

  // K fragments of the chunk computed next.  The page's second chunk is read
  // while the last row of the first still has its softmax and P V ahead of it:
  // the fragments are dead once that row's Q K is issued, so this costs no
  // register.  (Reading the next page's first chunk the same way, when it has
  // already landed, measured 1-3% slower on every plan set.)
  ls_u32x4 kf0[4], kf1[4];
  auto load_k = [&](int ui, int c) {
    const uint8_t* kb = s_ring + (ui % LS_ATT_STAGES) * LS_ATT_STAGE_BYTES;
    const int R0 = 32 * c + r, R1 = 32 * c + 16 + r;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int C = 4 * ks + q;
      kf0[ks] = *reinterpret_cast<const ls_u32x4*>(kb + R0 * 256 + ((C ^ (R0 & 15)) << 4));
      kf1[ks] = *reinterpret_cast<const ls_u32x4*>(kb + R1 * 256 + ((C ^ (R1 & 15)) << 4));
    }
  };

  // Chunk c (32 keys from key `base`) of the page in stage ui, for the rows in `need`.
  auto chunk = [&](int ui, int c, int base, uint32_t need, int v_e, uint64_t ve_mask,
                   float p_unscale) {
    // V^T row 16 db + r (so (row >> 1) & 7 == (r >> 1) & 7), logical chunk 4c + q;
    // read once for all rows, in flight during the first row's Q K and softmax.
    const uint8_t* vrow = s_ring + (ui % LS_ATT_STAGES) * LS_ATT_STAGE_BYTES + LS_ATT_KBYTES +
                          r * 128 + (((4 * c + q) ^ ((r >> 1) & 7)) << 4);
    ls_u32x4 vf[8];
#pragma unroll
    for (int db = 0; db < 8; ++db) vf[db] = *reinterpret_cast<const ls_u32x4*>(vrow + db * 2048);
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      if (!((need >> j) & 1u)) continue;
      // S^T: lane (r, q) gets head r's raw scores of keys base + 8q + 0..7.
      ls_f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        s0 = LsElem<DT>::mfma(kf0[ks], qf[j][ks], s0);
        s1 = LsElem<DT>::mfma(kf1[ks], qf[j][ks], s1);
      }
      if (c == 0 && (need >> (j + 1)) == 0u) load_k(ui, 1);
      float sv[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
      if (__builtin_expect(base + 31 > jmax_r[j], 0)) {  // the chunk crosses this row's causal frontier
        // This lane's last visible key offset, formed here so that the eight
        // key indices are not kept for every chunk (the empty asm keeps the
        // compiler from rewriting the compares back into them).
        int lim = jmax_r[j] - base - 8 * q;
        asm("" : "+v"(lim));
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (i > lim) sv[i] = -INFINITY;
      }
      // With a bias the scores are taken to base-2 units here (the maxima and
      // the threshold below are then in those units).
      if constexpr (BIAS) {
        const float* bp = s_bias + (ui % LS_ATT_STAGES) * 64 + 32 * c + 8 * q;
        const ls_f32x4 cbv0 = *reinterpret_cast<const ls_f32x4*>(bp);
        const ls_f32x4 cbv1 = *reinterpret_cast<const ls_f32x4*>(bp + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sv[i] = fmaf(sv[i], scale_log2, cbv0[i]);
          sv[4 + i] = fmaf(sv[4 + i], scale_log2, cbv1[i]);
        }
      }
      // Plain maxima: the compiler inserts the wait states an MFMA result
      // needs before a VALU read (it cannot for inline asm), and this file is
      // built without IEEE NaN quieting, so they fuse into v_max3 (grouped
      // here as three v_max3 and one v_max).
      const float lmax = fmaxf(fmaxf(fmaxf(sv[6], sv[7]), fmaxf(fmaxf(sv[0], sv[1]), sv[2])),
                               fmaxf(fmaxf(sv[3], sv[4]), sv[5]));
      // Rescale only when some head's max grows by more than 2^8 (or when the
      // page's V scale leaves too little fp16 headroom for P up to 2^8).
      const float thr = BIAS ? m_run[j] + 8.f : (m_run[j] + 8.f) * inv_scale_log2;
      if (__builtin_expect((__ballot(lmax > thr) | ve_mask) != 0ull, 0)) {
        float cm = lmax;
        cm = fmaxf(cm, ls_shfl_xor(cm, 16));
        cm = fmaxf(cm, ls_shfl_xor(cm, 32));
        const float m_new = fmaxf(m_run[j], BIAS ? cm : cm * scale_log2);
        const float alpha = __builtin_amdgcn_exp2f(m_run[j] - m_new);
        m_run[j] = m_new;
        l_run[j] *= alpha;
#pragma unroll
        for (int db = 0; db < 8; ++db) o[j][db] *= alpha;
      }
      // P' = P * 2^e (the page's V scale moved onto P, exact): one exp each;
      // the row sum adds the fp16 P' that the MFMA uses, scaled back by 2^-e.
      const float bias = (float)v_e - m_run[j];
      ls_u32x4 pf;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (BIAS)
          pf[i] = ls_pack_f16x2(__builtin_amdgcn_exp2f(sv[2 * i] + bias),
                                __builtin_amdgcn_exp2f(sv[2 * i + 1] + bias));
        else
          pf[i] = ls_pack_f16x2(__builtin_amdgcn_exp2f(fmaf(sv[2 * i], scale_log2, bias)),
                                __builtin_amdgcn_exp2f(fmaf(sv[2 * i + 1], scale_log2, bias)));
      }
      const float lsum = ls_sum_f16x2(pf[3], ls_sum_f16x2(pf[2], ls_sum_f16x2(pf[1], ls_sum_f16x2(pf[0], 0.f))));
      l_run[j] = fmaf(lsum, p_unscale, l_run[j]);
#pragma unroll
      for (int db = 0; db < 8; ++db) o[j][db] = LsElem<LS_F16>::mfma(vf[db], pf, o[j][db]);
    }
  };

  // A visit's list entry is read two visits ahead and its stage word during the
  // visit before, so that neither read is waited for where the page is ready: a
  // page stays in its stage until this wave is done with it, so a word that showed
  // its token once stays valid, and LDS accesses of a wave are in order, so the
  // page's data is read after it.
  auto entry = [&](int k) -> uint32_t { return k < n_visits ? s_wlist[w][k] : 0u; };
  auto uniform = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
  auto stage_peek = [&](int ui) -> uint64_t {
    return __hip_atomic_load(reinterpret_cast<uint64_t*>(&s_rdy[ui % LS_ATT_STAGES][0]),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  uint32_t e_cur = uniform(entry(0));
  uint32_t e_next = entry(1);
  uint64_t sw = stage_peek((int)(e_cur >> 16));
  int spins = spin_limit;  // bound of this wave's next wait (in polls)
  for (int k = 0; k < n_visits; ++k) {
    const int ui = (int)(e_cur >> 16);
    if (!is_ready(ui, sw)) {
      // Bounded wait (the protocol cannot deadlock; the bound only guarantees
      // that a wave always finishes).  A wave whose wait expires reports it
      // in the status word and goes on without waiting again (its outputs are
      // void), so a broken ring costs one bound per wave, not one per page;
      // the host turns the status into an error, and the epilogue below
      // writes NaN rows once it is set.
      bool landed = false;
      for (int spin = 0; spin < spins; ++spin) {
        if (!try_claim(ui)) __builtin_amdgcn_s_sleep(LS_ATT_SPIN_SLEEP);
        sw = stage_word(ui);
        if (is_ready(ui, sw)) {
          landed = true;
          break;
        }
      }
      if (!landed) {
        spins = 0;
        if (lane == 0)
          __hip_atomic_fetch_or(status, LS_ATTN_RING_TIMEOUT, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int v_e = __builtin_amdgcn_readfirstlane((int)(uint32_t)(sw >> 32));
    const uint32_t e = e_cur;
    e_cur = uniform(e_next);
    e_next = entry(k + 2);
    const int page = (int)(e & 0x1fffu);
    const uint32_t sel = (e >> 13) & ((1u << TPW) - 1u);
    const float p_unscale = uniform_f(__builtin_ldexpf(1.f, -v_e));
    const uint64_t ve_mask = v_e > 7 ? ~0ull : 0ull;
    load_k(ui, 0);
    // Every row of the entry sees the page's first chunk.
    chunk(ui, 0, 64 * page, sel, v_e, ve_mask, p_unscale);
    uint32_t need = 0;
#pragma unroll
    for (int j = 0; j < TPW; ++j)
      need |= (uint32_t)(((sel >> j) & 1u) && 64 * page + 32 <= jmax_r[j]) << j;
    sw = stage_peek((int)(e_cur >> 16));
    if (need) chunk(ui, 1, 64 * page + 32, need, v_e, ve_mask, p_unscale);
    // Done with the stage (the release orders this wave's reads of it first).
    if (lane == 0)
      __hip_atomic_fetch_add(&s_done[ui % LS_ATT_STAGES], 1u, __ATOMIC_RELEASE,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  LS_WAIT_VMCNT(0);  // no copy of this wave may land after the workgroup ends

  // ---- epilogue ----
  // A wait that expired (this wave's, or any earlier one seen here) makes the
  // rows NaN, so the failure also shows where the host cannot read the status
  // word (a replayed graph).  Read once per wave, after the loop.
  const bool expired = (__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(
                            status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) &
                        LS_ATTN_RING_TIMEOUT) != 0;
#pragma unroll
  for (int j = 0; j < TPW; ++j) {
    const int row = w0 + j;
    float l_tot = l_run[j] + ls_shfl_xor(l_run[j], 16);
    l_tot += ls_shfl_xor(l_tot, 32);
    if (j >= n_mine || row >= n_rows || !head_ok) continue;
    const int64_t t = t0 + row;
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    uint16_t* orow = out + (t * G * gs + (int64_t)g * gs + head) * D + 4 * q;
    if (expired) {  // quiet-NaN bit patterns (this file assumes no NaN arithmetic)
      const uint32_t nan2 = DT == LS_BF16 ? 0x7fc07fc0u : 0x7e007e00u;
#pragma unroll
      for (int db = 0; db < 8; ++db) *reinterpret_cast<uint2*>(orow + 16 * db) = make_uint2(nan2, nan2);
      if (lse && q == 0) lse[((int64_t)g * gs + head) * total_q + t] = __uint_as_float(0x7fc00000u);
      continue;
    }
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      const uint32_t lo = ls_pack2(LsElem<DT>::from_f(o[j][db][0] * inv), LsElem<DT>::from_f(o[j][db][1] * inv));
      const uint32_t hi = ls_pack2(LsElem<DT>::from_f(o[j][db][2] * inv), LsElem<DT>::from_f(o[j][db][3] * inv));
      *reinterpret_cast<uint2*>(orow + 16 * db) = make_uint2(lo, hi);
    }
    if (lse && q == 0)
      lse[((int64_t)g * gs + head) * total_q + t] =
          l_tot > 0.f ? m_run[j] * 0.69314718055994531f + __logf(l_tot) : INFINITY;
  }
}

// NOSA key biases: cb[g][64 pg_off[b] + j] = log2(e) * cis[cu_k[b] + j][g] for
// j < len_k(b), 0 past each sequence end (those keys are never visible).  One
// workgroup per 64-key page of one group.
template <int CT>
__global__ __launch_bounds__(64) void ls_bias_kernel(const typename LsElem<CT>::T* __restrict__ cis,
                                                     int64_t cis_rs, const int32_t* __restrict__ cu_k,
                                                     const int32_t* __restrict__ pg_off, int batch,
                                                     int64_t lpad, float* __restrict__ cb) {
  const int64_t tile_id = LS_BID_X;
  if (tile_id >= pg_off[batch]) return;
  const int g = LS_BID_Y;
  const int b = ls_find_segment(pg_off, batch, tile_id);
  const int p = (int)(tile_id - pg_off[b]);
  const int lk = cu_k[b + 1] - cu_k[b];
  const int j = 64 * p + LS_TID;
  float v = 0.f;
  if (j < lk) v = LsElem<CT>::to_f(cis[((int64_t)cu_k[b] + j) * cis_rs + g]) * 1.4426950408889634f;
  cb[(int64_t)g * lpad + 64LL * (pg_off[b] + p) + LS_TID] = v;
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
namespace {
constexpr int kDefaultSpinLimit = 1 << 22;
int g_spin_limit = kDefaultSpinLimit;  // bound of one ring wait (in polls)

struct AttnWs {
  size_t status, kv, pg, tiles, vexp, cb, tok, total;
  int64_t lpad, n_pages;
};
AttnWs attn_ws(int64_t total_k, int batch, int G, bool bias) {
  AttnWs L;
  L.n_pages = (total_k + 63) / 64 + batch;
  L.lpad = L.n_pages * 64;
  size_t off = 0;
  L.status = off; off += 256;  // the call's status word comes first
  L.kv = off; off += ls_align256((size_t)G * L.n_pages * LS_ATT_STAGE_BYTES);
  L.pg = off; off += ls_align256((size_t)(batch + 1) * 4);
  L.tiles = off; off += ls_align256((size_t)(batch + 1) * 4);
  L.vexp = off; off += ls_align256((size_t)G * L.n_pages * 4);
  L.cb = off; off += bias ? ls_align256((size_t)G * L.lpad * 4) : 0;
  L.tok = off; off += ls_align256((size_t)(LS_ATT_UNION_CAP + 1) * 4);
  L.total = off;
  return L;
}

// How a call's rows are cut into tiles and dealt to the XCDs: rows per wave of a
// tile, consecutive tiles per XCD run, tiles of one KV group an XCD takes before
// it turns to the next group, and tiles of one group per XCD.
struct AttnTiling {
  int tpw, run, span, per_xcd;
};

int attn_tile_rows(int tpw) {
  return tpw == 1 ? LsAttTile<1>::kTile : tpw == 2 ? LsAttTile<2>::kTile : LsAttTile<3>::kTile;
}

// One workgroup fills a CU's LDS, so a call runs in rounds of 256 tiles.  24-row
// tiles share each page copy among the most rows, but a call of few rows then
// leaves CUs idle and waits for its largest tile: while a smaller tile gives at
// most two rounds it is the faster one (the attention call of one sequence, us,
// tiles of 8 / 12 / 24 rows: 600 rows 43 / 47 / 53, 2048 83 / 88 / 113, 2300 102 /
// 95 / 122, 3072 146 / 129 / 153, 3400 174 / 164 / 172, 4096 217 / 217 / 205).
// Sequences of up to 256 keys have few pages, so a round takes about as long at
// every height (it is mostly the tile's setup) and one round of larger tiles beats
// two of smaller ones (100 sequences of 20 rows 56 / 55 / 50, 40 of 64 rows 55 / 54
// / 44, 20 of 40 rows, one round, 35 / 36 / 41).  Runs of 4 tiles even the XCDs'
// loads where runs of 16 leave some idle (8K rows 411 against 463 us) and cost
// nothing at 128K (12.06 against 12.08 ms).  An XCD that alternates between the KV
// groups run by run starts every group's large tiles early, which a call of up to
// four rounds needs (three sequences of 4500 rows in all 106 against 134 us);
// longer calls keep to one group at a time, whose pages then have the XCD's L2 to
// themselves (128K 12.06 against 12.42 ms, four sequences of 24K rows in all 1.20
// against 1.25).
AttnTiling attn_tiling(int64_t total_q, int batch, int G, int head_tiles, int max_seqlen_k) {
  constexpr int64_t kCus = 256;
  // At most this many tiles of one group: each sequence's last tile may be partial.
  auto tiles = [&](int tpw) {
    const int rows = attn_tile_rows(tpw);
    return (total_q + (int64_t)batch * (rows - 1)) / rows;
  };
  const int64_t per_tile = (int64_t)G * head_tiles;
  const int64_t most = (max_seqlen_k <= 256 ? 1 : 2) * kCus;
  AttnTiling t;
  t.tpw = tiles(1) * per_tile <= most ? 1 : tiles(2) * per_tile <= most ? 2 : 3;
  t.run = 4;
  t.per_xcd = (int)(t.run * ((tiles(t.tpw) + 8 * t.run - 1) / (8 * t.run)));
  t.span = tiles(t.tpw) * per_tile <= 4 * kCus ? t.run : t.per_xcd;
  return t;
}

template <int DT, bool BIAS, int TPW>
void launch_tile(dim3 grid, hipStream_t s, const void* q, int64_t q_rs, const uint8_t* kv,
                 const AttnWs& L, const int32_t* vexp, const float* cb,
                 const int32_t* tok,
                 const int32_t* cu_q, const int32_t* cu_k, const int32_t* pg,
                 const int32_t* tiles, int batch, int64_t total_q, int G, int gs,
                 const int32_t* topk_idx, int take, float scale_log2, int causal, void* out,
                 float* lse, const AttnTiling& tl, int32_t* status) {
  hipLaunchKernelGGL((ls_attn_tile_kernel<DT, BIAS, TPW>), grid, dim3(LS_ATT_THREADS), 0, s,
                     (const uint16_t*)q, q_rs, kv, L.lpad, vexp, cb, tok,
                     L.n_pages, cu_q, cu_k, pg, tiles, batch, total_q, G, gs, topk_idx, take,
                     scale_log2, causal, (uint16_t*)out, lse, tl.run, tl.span, tl.per_xcd, status,
                     g_spin_limit);
}

// Shared body of the plain and the NOSA (cis != nullptr) entry points.
int attn_run(const char* who, const void* q, int64_t q_row_stride, const void* k,
             int64_t k_row_stride, const void* v, int64_t v_row_stride, const void* cis,
             int64_t cis_row_stride, int32_t cis_dtype, const int32_t* cu_seqlens_q,
             const int32_t* cu_seqlens_k, int32_t batch, int64_t total_q, int64_t total_k,
             int32_t max_seqlen_k, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
             int32_t dtype, const int32_t* topk_idx, int32_t take, int32_t block_size,
             float softmax_scale, int32_t causal, void* out, float* lse, void* workspace,
             size_t workspace_bytes, void* stream, int32_t* status_out = nullptr) {
  const bool bias = cis != nullptr;
  LS_REQUIRE(dtype == LS_BF16 || dtype == LS_F16, LS_ERR_UNSUPPORTED,
             "%s: only bf16 and fp16 are supported (dtype %d)", who, dtype);
  LS_REQUIRE(head_dim == 128, LS_ERR_UNSUPPORTED, "%s: head_dim must be 128 (got %d)", who,
             head_dim);
  LS_REQUIRE(block_size == 64, LS_ERR_UNSUPPORTED, "%s: block_size must be 64 (got %d)", who,
             block_size);
  LS_REQUIRE(num_heads > 0 && num_kv_heads > 0 && num_heads % num_kv_heads == 0, LS_ERR_INVALID,
             "%s: num_heads must be a positive multiple of num_kv_heads", who);
  LS_REQUIRE(batch >= 0 && total_q >= 0 && total_k >= 0 && take >= 0, LS_ERR_INVALID,
             "%s: bad sizes", who);
  LS_REQUIRE(take <= LS_ATTN_MAX_TAKE, LS_ERR_UNSUPPORTED, "%s: at most %d ids per row (got %d)",
             who, LS_ATTN_MAX_TAKE, take);
  LS_REQUIRE((int64_t)max_seqlen_k <= 64LL * LS_ATTN_MAX_PAGES, LS_ERR_UNSUPPORTED,
             "%s: max_seqlen_k above %d", who, 64 * LS_ATTN_MAX_PAGES);
  LS_REQUIRE(!bias || cis_dtype == LS_F32 || cis_dtype == LS_BF16 || cis_dtype == LS_F16,
             LS_ERR_INVALID, "%s: unknown CIS dtype %d", who, cis_dtype);
  if (total_q == 0 || batch == 0) return LS_OK;
  LS_REQUIRE(q && k && v && out && cu_seqlens_q && cu_seqlens_k && (take == 0 || topk_idx),
             LS_ERR_INVALID, "%s: null pointer", who);
  LS_REQUIRE(ls_aligned16(q) && ls_aligned16(k) && ls_aligned16(v) && ls_aligned16(out) &&
                 q_row_stride % 8 == 0 && k_row_stride % 8 == 0 && v_row_stride % 8 == 0,
             LS_ERR_UNSUPPORTED,
             "%s: tensors must be 16-byte aligned with row strides %% 8 == 0", who);
  const AttnWs L = attn_ws(total_k, batch, num_kv_heads, bias);
  LS_REQUIRE(workspace && workspace_bytes >= L.total, LS_ERR_WORKSPACE,
             "%s: workspace needs %zu bytes", who, L.total);
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)workspace;
  uint8_t* kv = (uint8_t*)(ws + L.kv);
  int32_t* pg = (int32_t*)(ws + L.pg);
  int32_t* vexp = (int32_t*)(ws + L.vexp);
  int32_t* tiles = (int32_t*)(ws + L.tiles);
  float* cb = bias ? (float*)(ws + L.cb) : nullptr;
  int32_t* tok = (int32_t*)(ws + L.tok);
  int32_t* status = status_out ? status_out : (int32_t*)(ws + L.status);
  const int gs = num_heads / num_kv_heads;
  const AttnTiling tl =
      attn_tiling(total_q, batch, num_kv_heads, (gs + 15) / 16, max_seqlen_k);
  const int tile_rows = attn_tile_rows(tl.tpw);
  hipLaunchKernelGGL(ls_attn_plan_kernel, dim3(1), dim3(64), 0, s, cu_seqlens_q, cu_seqlens_k,
                     batch, tile_rows, pg, tiles, tok, LS_ATT_UNION_CAP + 1, status);
  int rc = ls_check_launch("ls_attn_plan_kernel");
  if (rc) return rc;
  if (total_k > 0) {
    const dim3 vgrid((unsigned)((total_k + 63) / 64 + batch), num_kv_heads);
    if (dtype == LS_BF16)
      hipLaunchKernelGGL(ls_kv_stage_kernel<LS_BF16>, vgrid, dim3(256), 0, s, (const uint16_t*)k,
                         k_row_stride, (const uint16_t*)v, v_row_stride, cu_seqlens_k, pg, batch,
                         L.n_pages, kv, vexp);
    else
      hipLaunchKernelGGL(ls_kv_stage_kernel<LS_F16>, vgrid, dim3(256), 0, s, (const uint16_t*)k,
                         k_row_stride, (const uint16_t*)v, v_row_stride, cu_seqlens_k, pg, batch,
                         L.n_pages, kv, vexp);
    if ((rc = ls_check_launch("ls_kv_stage_kernel"))) return rc;
    if (bias) {
      if (cis_dtype == LS_BF16)
        hipLaunchKernelGGL(ls_bias_kernel<LS_BF16>, vgrid, dim3(64), 0, s, (const uint16_t*)cis,
                           cis_row_stride, cu_seqlens_k, pg, batch, L.lpad, cb);
      else if (cis_dtype == LS_F16)
        hipLaunchKernelGGL(ls_bias_kernel<LS_F16>, vgrid, dim3(64), 0, s, (const uint16_t*)cis,
                           cis_row_stride, cu_seqlens_k, pg, batch, L.lpad, cb);
      else
        hipLaunchKernelGGL(ls_bias_kernel<LS_F32>, vgrid, dim3(64), 0, s, (const float*)cis,
                           cis_row_stride, cu_seqlens_k, pg, batch, L.lpad, cb);
      if ((rc = ls_check_launch("ls_bias_kernel"))) return rc;
    }
  }
  const float scale = softmax_scale > 0.f ? softmax_scale : 1.0f / sqrtf((float)head_dim);
  const float scale_log2 = scale * 1.4426950408889634f;
  const dim3 grid((unsigned)(8 * tl.per_xcd), num_kv_heads, (gs + 15) / 16);
#define LS_TILE_ARGS                                                                              \
  grid, s, q, q_row_stride, kv, L, vexp, cb, tok, cu_seqlens_q, cu_seqlens_k, pg,              \
      tiles, batch, total_q, num_kv_heads, gs, topk_idx, take, scale_log2, causal, out, lse, \
      tl, status
  auto launch = [&](auto tpw) {
    constexpr int kTpw = decltype(tpw)::value;
    static_assert(LsAttTile<kTpw>::kMaxTake >= LS_ATTN_MAX_TAKE, "every accepted plan fits a tile");
    if (dtype == LS_BF16) {
      if (bias) launch_tile<LS_BF16, true, kTpw>(LS_TILE_ARGS);
      else launch_tile<LS_BF16, false, kTpw>(LS_TILE_ARGS);
    } else {
      if (bias) launch_tile<LS_F16, true, kTpw>(LS_TILE_ARGS);
      else launch_tile<LS_F16, false, kTpw>(LS_TILE_ARGS);
    }
  };
  if (tl.tpw == 1) launch(std::integral_constant<int, 1>());
  else if (tl.tpw == 2) launch(std::integral_constant<int, 2>());
  else launch(std::integral_constant<int, 3>());
#undef LS_TILE_ARGS
  return ls_check_launch("ls_attn_tile_kernel");
}
}  // namespace

extern "C" int32_t ls_attn_set_spin_limit(int32_t spins) {
  const int32_t prev = g_spin_limit;
  g_spin_limit = spins < 0 ? kDefaultSpinLimit : spins;
  return prev;
}

extern "C" int32_t ls_attn_tile_rows(int64_t total_q, int32_t batch, int32_t num_heads,
                                     int32_t num_kv_heads, int32_t max_seqlen_k) {
  if (total_q < 0 || batch < 0 || num_kv_heads <= 0 || num_heads <= 0 ||
      num_heads % num_kv_heads != 0)
    return 0;
  const int head_tiles = (num_heads / num_kv_heads + 15) / 16;
  return attn_tile_rows(attn_tiling(total_q, batch, num_kv_heads, head_tiles, max_seqlen_k).tpw);
}

extern "C" size_t ls_sparse_attn_workspace_size(int64_t total_k, int32_t batch,
                                                int32_t num_kv_heads, int32_t head_dim,
                                                int32_t max_seqlen_k, int32_t dtype) {
  (void)max_seqlen_k;
  (void)head_dim;
  (void)dtype;
  return attn_ws(total_k, batch, num_kv_heads, false).total;
}

extern "C" size_t ls_nosa_attn_workspace_size(int64_t total_k, int32_t batch,
                                              int32_t num_kv_heads, int32_t head_dim,
                                              int32_t max_seqlen_k, int32_t dtype) {
  (void)max_seqlen_k;
  (void)head_dim;
  (void)dtype;
  return attn_ws(total_k, batch, num_kv_heads, true).total;
}

extern "C" int ls_sparse_attn_varlen(const void* q, int64_t q_row_stride, const void* k,
                                     int64_t k_row_stride, const void* v, int64_t v_row_stride,
                                     const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                     int32_t batch, int64_t total_q, int64_t total_k,
                                     int32_t max_seqlen_q, int32_t max_seqlen_k,
                                     int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                                     int32_t dtype, const int32_t* topk_idx, int32_t take,
                                     int32_t block_size, float softmax_scale, int32_t causal,
                                     void* out, float* lse, void* workspace,
                                     size_t workspace_bytes, void* stream) {
  (void)max_seqlen_q;
  return attn_run("ls_sparse_attn_varlen", q, q_row_stride, k, k_row_stride, v, v_row_stride,
                  nullptr, 0, 0, cu_seqlens_q, cu_seqlens_k, batch, total_q, total_k,
                  max_seqlen_k, num_heads, num_kv_heads, head_dim, dtype, topk_idx, take,
                  block_size, softmax_scale, causal, out, lse, workspace, workspace_bytes,
                  stream);
}

extern "C" int ls_nosa_attn_varlen(const void* q, int64_t q_row_stride, const void* k,
                                   int64_t k_row_stride, const void* v, int64_t v_row_stride,
                                   const void* cis, int64_t cis_row_stride, int32_t cis_dtype,
                                   const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                   int32_t batch, int64_t total_q, int64_t total_k,
                                   int32_t max_seqlen_q, int32_t max_seqlen_k, int32_t num_heads,
                                   int32_t num_kv_heads, int32_t head_dim, int32_t dtype,
                                   const int32_t* topk_idx, int32_t take, int32_t block_size,
                                   float softmax_scale, void* out, float* lse, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  (void)max_seqlen_q;
  LS_REQUIRE(total_k == 0 || cis, LS_ERR_INVALID, "ls_nosa_attn_varlen: null CIS scores");
  static const uint16_t kNoKeys = 0;  // any non-null pointer: no key reads it
  return attn_run("ls_nosa_attn_varlen", q, q_row_stride, k, k_row_stride, v, v_row_stride,
                  cis ? cis : &kNoKeys, cis_row_stride, cis_dtype, cu_seqlens_q, cu_seqlens_k,
                  batch, total_q, total_k, max_seqlen_k, num_heads, num_kv_heads, head_dim,
                  dtype, topk_idx, take, block_size, softmax_scale, 1, out, lse, workspace,
                  workspace_bytes, stream);
}

// ---------------------------------------------------------------------------
// Allocation-free variant of ls_sparse_attn_varlen: the workspace is a static
// device array of the library instead of a caller buffer.  In host code
// `scratch` only names the symbol; its device address (one per GPU) comes
// from hipGetSymbolAddress, taken once per device with that device current.
// ---------------------------------------------------------------------------
#define LS_MAX_DEVICES 64  // LS_NOALLOC_SCRATCH_BYTES comes from the public header

static __device__ __align__(256) uint8_t scratch[LS_NOALLOC_SCRATCH_BYTES];

namespace {
std::mutex g_scratch_mu;
void* g_scratch_ptr[LS_MAX_DEVICES] = {};

// Device address of `scratch` on the device that owns `stream`.
int scratch_for_stream(hipStream_t stream, void** ptr) {
  int dev = -1;
  hipError_t e = stream ? hipStreamGetDevice(stream, &dev) : hipGetDevice(&dev);
  if (e != hipSuccess)
    return ls_fail(LS_ERR_HIP, "ls_sparse_attn_varlen_noalloc: no device for the stream: %s",
                   hipGetErrorString(e));
  LS_REQUIRE(dev >= 0 && dev < LS_MAX_DEVICES, LS_ERR_UNSUPPORTED,
             "ls_sparse_attn_varlen_noalloc: device %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    int cur = -1;
    if ((e = hipGetDevice(&cur)) != hipSuccess)
      return ls_fail(LS_ERR_HIP, "ls_sparse_attn_varlen_noalloc: %s", hipGetErrorString(e));
    if (cur != dev && (e = hipSetDevice(dev)) != hipSuccess)
      return ls_fail(LS_ERR_HIP, "ls_sparse_attn_varlen_noalloc: %s", hipGetErrorString(e));
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != dev) (void)hipSetDevice(cur);
    if (e != hipSuccess || !p)
      return ls_fail(LS_ERR_HIP, "ls_sparse_attn_varlen_noalloc: scratch address on device %d: %s",
                     dev, hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return LS_OK;
}
}  // namespace

extern "C" int ls_sparse_attn_varlen_noalloc(
    const void* q, int64_t q_row_stride, const void* k, int64_t k_row_stride, const void* v,
    int64_t v_row_stride, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int32_t batch,
    int64_t total_q, int64_t total_k, int32_t max_seqlen_q, int32_t max_seqlen_k,
    int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t dtype,
    const int32_t* topk_idx, int32_t take, int32_t block_size, float softmax_scale,
    int32_t causal, void* out, float* lse, int32_t* status, void* stream) {
  (void)max_seqlen_q;
  // The size check comes first and touches no device.
  LS_REQUIRE(batch >= 0 && total_k >= 0 && num_kv_heads > 0, LS_ERR_INVALID,
             "ls_sparse_attn_varlen_noalloc: bad sizes");
  const size_t need = attn_ws(total_k, batch, num_kv_heads, false).total;
  LS_REQUIRE(need <= LS_NOALLOC_SCRATCH_BYTES, LS_ERR_UNSUPPORTED,
             "ls_sparse_attn_varlen_noalloc: %lld keys in %d sequences of %d KV heads need "
             "%zu bytes of scratch, above the static %u (use ls_sparse_attn_varlen with a "
             "workspace)",
             (long long)total_k, batch, num_kv_heads, need, LS_NOALLOC_SCRATCH_BYTES);
  if (total_q == 0 || batch == 0) {
    // Nothing to attend; the caller's status word still gets this call's value.
    if (!status) return LS_OK;
    hipLaunchKernelGGL(ls_attn_status_clear_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream,
                       status);
    return ls_check_launch("ls_attn_status_clear_kernel");
  }
  void* ws = nullptr;
  const int rc = scratch_for_stream((hipStream_t)stream, &ws);
  if (rc) return rc;
  return attn_run("ls_sparse_attn_varlen_noalloc", q, q_row_stride, k, k_row_stride, v,
                  v_row_stride, nullptr, 0, 0, cu_seqlens_q, cu_seqlens_k, batch, total_q,
                  total_k, max_seqlen_k, num_heads, num_kv_heads, head_dim, dtype, topk_idx,
                  take, block_size, softmax_scale, causal, out, lse, ws,
                  LS_NOALLOC_SCRATCH_BYTES, stream, status);
}
