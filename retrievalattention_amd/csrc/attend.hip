// Weighted flash decoding for the wave index (gfx950).
//
// One kernel serves every attention call of the decode step.  A workgroup (8 waves) takes
// one split of one group's rows; a wave owns a contiguous run of rows of one kind and walks it in batches
// of 64 rows = 4 chunks of 16.  For a batch it first fetches one row descriptor per lane
// (where the row lives); a chunk's loads are requested while the chunk before it is computed:
//   * key/value rows: scores = scale * q·k on bf16 MFMA 16x16x32 with the
//     query heads as the A rows and 16 key rows as the B columns, so each lane ends up with
//     the scores of one key row for four heads;
//   * estimation rows: the score of a cluster is the logit already computed
//     by the scoring kernel, the "value" row is the cluster's value sum and the softmax
//     denominator is weighted by the cluster size.
// P·V runs on the matrix cores too: the chunk's probabilities go to LDS as bf16 [head][row], the 16 x 128
// value tile row-major, and eight MFMA 16x16x16 (B operands read with LDS transpose loads) add the chunk
// to fp32 accumulators that hold, per lane, four heads of one dimension per 16-wide tile.  A group with few
// rows has one workgroup, which writes the output; otherwise every workgroup writes a (max, denominator, numerator)
// partial, and of each share of the heads the wave that finishes last for a group merges the partials (and an optional
// previous result) with the log-sum-exp rule and writes the output, so the whole call is one launch.
//
// Semantics follow the weighted_flash_decoding call sites at
// cache_hub/retroinfer_cache.py:611-617 and :666-674.
#include <math.h>
#include <stdint.h>

#include <mutex>

#include "attend_common.h"
#include "ri_common.h"
#include "step_route.h"

// (what the first loads want stands before the struct: in registers at the start; 32 groups of 4 heads over 8192 clusters 16.5
// -> 16.3 us, 12 groups of 7 heads over 1856 in half 9.34 -> 9.14)
template <int GS_PAD, bool HALF>
__global__ __launch_bounds__(64 * ATT_WAVES, 2) void attend_kernel(ri_ptr4 in, ri_int4 n, ri_int2 len, AttendParams A) {
  AttendParams P = A;
  P.ret_off = ri_global<const int32_t>(in[0]);
  P.ret_start = ri_global<const int32_t>(in[1]);
  P.lenB_ptr = ri_global<const int32_t>(in[2]);
  P.q = ri_global<const uint16_t>(in[3]);
  P.np = n[0];
  P.gs = n[1];
  P.S = n[2];
  P.W_kv = n[3];
  P.lenB_ptr_stride = len[0];
  P.lenA = len[1];
  attend_group<GS_PAD, HALF, KEPT_NONE>(P, blockIdx.x, blockIdx.y, AttendKept{});
}

// ------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------
#define RI_MAX_SPLITS 64
#define RI_MAX_PROBES 4096  // rank tables of a launch: (2 * np + 1) * 4 bytes of LDS (what the selection lays out)
#define RI_MAX_GROUPS 4096  // groups of a launch; words of the counter area at the head of the workspace

// workgroups per group at most: one per compute unit for all groups together (plan_splits)
static int attn_max_splits(int BG) { return min(RI_MAX_SPLITS, max(256 / BG, 1)); }
static constexpr bool counters_fit(int BG) { return BG * ATT_WAVES * attend_counter_pitch(BG) <= RI_MAX_GROUPS; }
static_assert(counters_fit(16) && counters_fit(32) && counters_fit(64) && counters_fit(128), "more than one workgroup per group: up to 128 groups");

static size_t attn_workspace_bytes(int BG, int gs) {
  if (BG <= 0 || BG > RI_MAX_GROUPS || gs <= 0 || gs > 16) return 0;
  const size_t per = (size_t)BG * attn_max_splits(BG) * gs_pad_of(gs);
  return RI_MAX_GROUPS * sizeof(int) + per * (2 + RI_DIM) * sizeof(float);
}

extern "C" size_t ri_flash_decoding_workspace_bytes(int BG, int gs) { return attn_workspace_bytes(BG, gs); }
extern "C" size_t ri_wave_attention_workspace_bytes(int BG, int gs) { return attn_workspace_bytes(BG, gs); }

// Bytes a launch with S splits per group really uses: the counter area, then the
// (max, denominator) pairs and the numerators of BG * S partials.
static size_t attn_scratch_used(int BG, int gp, int S) {
  return RI_MAX_GROUPS * sizeof(int) + (size_t)BG * S * gp * (2 + RI_DIM) * sizeof(float);
}

static void carve_workspace(AttendParams& P, void* workspace, int BG, int gp) {
  P.counters = (int*)workspace;
  P.pitch = attend_counter_pitch(BG);
  P.part_ml = (float*)((char*)workspace + RI_MAX_GROUPS * sizeof(int));
  P.part_acc = P.part_ml + (size_t)BG * P.S * gp * 2;
}

template <bool HALF>
static void launch_attend_t(const AttendParams& P, dim3 grid, int gp, size_t tab_bytes, hipStream_t s) {
  auto* kernel = gp == 4 ? attend_kernel<4, HALF> : gp == 8 ? attend_kernel<8, HALF> : attend_kernel<16, HALF>;
  kernel<<<grid, 64 * ATT_WAVES, tab_bytes, s>>>(ri_pack_ptrs(P.ret_off, P.ret_start, P.lenB_ptr, P.q),
                                                 (ri_int4){P.np, P.gs, P.S, P.W_kv}, (ri_int2){P.lenB_ptr_stride, P.lenA}, P);
}

static int launch_attend(AttendParams& P, int BG, int gs, bool half, hipStream_t s) {
  // Groups vary fastest: workgroups go to the eight chiplets in turn, and with eight splits that vary fastest the chiplets
  // of the last ones have estimation rows only, the others none (32 groups of 16 heads over 4096 clusters 15.2 -> 13.9 us, of
  // 4 over 1024 8.5 -> 8.2, of 8 over 16384 26.6 -> 25.9; elsewhere up to 2 %).
  const dim3 grid(BG, P.S);
  const size_t tab_bytes = P.ret_off ? (size_t)(2 * P.np + 1) * sizeof(int) : 0;
  if (half) launch_attend_t<true>(P, grid, gs_pad_of(gs), tab_bytes, s);
  else launch_attend_t<false>(P, grid, gs_pad_of(gs), tab_bytes, s);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

// Memory traffic of one estimation row: its value-sum row, the 32-byte sector around its cluster size, and
// either one 32-byte sector per query head around its logit or, when the scores are computed in the launch,
// its centroid row.
static int est_row_bytes(int gs, bool scored_here) { return 256 + 32 + (scored_here ? 256 : 32 * gs); }

// Split plan of a launch: workgroups per group, and the waves of a group that take key/value rows, shared with the
// estimation rows in proportion to the memory traffic of a row, es_row_bytes against the 512 bytes of a K and a V row.
//  * One workgroup of eight waves per compute unit: 64 groups of 8 heads over 16384 clusters 54.7 us, two per unit or
//    three of four waves 55.3 .. 60 us; 11 groups, 29000 rows: 38.0 against 41.9 .. 45.  256 / BG rounds down, which
//    leaves units without work between 86 and 255 groups (4 heads over 8192 clusters: 100 groups 33.8 us, 128: 42.0, 160:
//    58.6, 200: 67.0, 256: 88.8), and is still ahead of the two or more workgroups of four waves per group that it
//    replaced (42.4, 46.7, 78.7, 86.8, 101.8 us).
//  * A compute unit reads about 25 KB per microsecond, so more workgroups stream a group's rows faster, but the waves
//    that come last read the partials of all of them at that same rate: the sum of both is least near
//    sqrt(bytes of the group / bytes of a partial), flat towards fewer (12 groups of 7 heads in half, 3488 rows: 12 workgroups
//    9.9 us, 15 and 16 8.9, 21 9.3; 8 of 8, 4000: 12 9.8, 16 8.8, 21 9.3).
//  * A wave requests eight splits at a time, whether there are as many or not (combine_share), so one or two past a multiple of eight
//    cost as much as eight: 9 -> 8 workgroups 7.2 -> 6.8 us (16 groups of 4 heads, 623 rows), 17 -> 16 9.3 -> 8.9 (12 of 7, 3488), 26 -> 24
//    9.2 -> 8.8 (4 of 4, 4350), 34 -> 32 12.2 -> 11.8 (2 of 8, 15100), 20 -> 16 13.8 -> 12.8 (4 of 12, 8000); layers of captured
//    steps, 16 groups of 4 heads, 1024 clusters 18.4 -> 17.9, 8 of 8, 8192 28.6 -> 28.2, 4 of 4, 8192 24.7 -> 24.3.  It loses where a wave
//    gets a second chunk of rows by it: 20 -> 16 7.8 -> 8.3 (8 of 4, 2500), a layer of 1 of 8, 8192 24.6 -> 25.4, 12 of 7 24.2 -> 24.5.
//    More than a fifth is not worth giving up, nor any of them once a wave has more than four chunks.
//  * A few rows (less of them the more heads share their arithmetic) stay with one workgroup, which hands no partial to
//    another: one, two and three workgroups, 8 groups of 4 heads, 331 rows 6.7, 7.5, 6.6 us; of 8 heads, 200 rows 5.9, 7.0, 7.1, 331
//    7.1, 8.1, 7.1.
static void plan_splits(AttendParams& P, int64_t kv_rows, int64_t es_rows, int es_row_bytes, int BG, int gs,
                        int max_splits = RI_MAX_SPLITS, bool several = false) {
  const int64_t rows = kv_rows + es_rows, wk = kv_rows * 512, we = es_rows * es_row_bytes;
  int64_t per_group = attn_max_splits(BG);
  per_group = min(per_group, (int64_t)sqrt((double)(wk + we) / (double)(gs * 800)));
  per_group = min(per_group, (rows + 8 * ATT_WAVES - 1) / (8 * ATT_WAVES));   // half a chunk per wave at least
  per_group = min(per_group, (int64_t)max_splits);
  if (per_group > 8 && per_group % 8 * 5 <= per_group && rows <= 64 * ATT_WAVES * per_group) per_group -= per_group % 8;
  if ((!several && attend_alone(rows, gs, BG)) || per_group < 1) per_group = 1;
  const auto with_keys = [&](int64_t waves) {
    return (int)(es_rows > 0 ? min(max((wk * waves + (wk + we) / 2) / (wk + we), (int64_t)1), waves - 1) : waves);
  };
  P.S = (int)per_group;
  P.W_kv = with_keys(per_group * ATT_WAVES);
  P.W_one = with_keys(ATT_WAVES);
  const auto inverse = [](int64_t waves) { return ATT_INVERSE(max(waves, (int64_t)1)); };
  P.inv_kv = inverse(P.W_kv);
  P.inv_es = inverse(per_group * ATT_WAVES - P.W_kv);
  P.inv_kv_one = inverse(P.W_one);
  P.inv_es_one = inverse(ATT_WAVES - P.W_one);
}

static int flash_decoding_impl(const void* q, const void* k, const void* v, const void* weight,
                               const int32_t* cache_seqlens, const void* prev_out, const float* prev_lse, void* out,
                               float* lse_out, int BG, int gs, int S, int64_t kv_stride, float scale, void* workspace,
                               size_t workspace_bytes, bool half, ri_stream_t stream) {
  if (!q || !k || !v || !out || !workspace) return RI_ERR_ARG;
  if (ri_any_misaligned16(q, k, v, weight, prev_out, out, workspace)) return RI_ERR_ARG;
  if (BG <= 0 || BG > RI_MAX_GROUPS || gs <= 0 || gs > 16 || S < 0 || kv_stride < S) return RI_ERR_ARG;
  if ((prev_out == nullptr) != (prev_lse == nullptr)) return RI_ERR_ARG;
  if (workspace_bytes < attn_workspace_bytes(BG, gs)) return RI_ERR_WORKSPACE;
  const int gp = gs_pad_of(gs);
  AttendParams P = {};
  P.q = (const uint16_t*)q;
  P.kA = P.kB = (const uint16_t*)k;
  P.vA = P.vB = (const uint16_t*)v;
  P.strideA = P.strideB = kv_stride;
  P.lenA = 0;
  P.lenB_ptr = cache_seqlens;
  P.lenB_ptr_stride = 1;
  P.lenB_const = S;
  P.weightB = (const uint16_t*)weight;
  P.weight_stride = S;
  plan_splits(P, S, 0, 0, BG, gs);
  P.gs = gs;
  P.scale = scale;
  P.prev_out = (const uint16_t*)prev_out;
  P.prev_lse = prev_lse;
  P.out = (uint16_t*)out;
  P.lse_out = lse_out;
  carve_workspace(P, workspace, BG, gp);
  return launch_attend(P, BG, gs, half, (hipStream_t)stream);
}

extern "C" int ri_weighted_flash_decoding(const void* q, const void* k, const void* v, const void* weight,
                                          const int32_t* cache_seqlens, const void* prev_out,
                                          const float* prev_lse, void* out, float* lse_out, int BG, int gs,
                                          int S, int64_t kv_stride, float scale, void* workspace,
                                          size_t workspace_bytes, ri_stream_t stream) {
  return flash_decoding_impl(q, k, v, weight, cache_seqlens, prev_out, prev_lse, out, lse_out, BG, gs, S, kv_stride,
                             scale, workspace, workspace_bytes, false, stream);
}

extern "C" int ri_weighted_flash_decoding_f16(const void* q, const void* k, const void* v, const void* weight,
                                              const int32_t* cache_seqlens, const void* prev_out,
                                              const float* prev_lse, void* out, float* lse_out, int BG, int gs,
                                              int S, int64_t kv_stride, float scale, void* workspace,
                                              size_t workspace_bytes, ri_stream_t stream) {
  return flash_decoding_impl(q, k, v, weight, cache_seqlens, prev_out, prev_lse, out, lse_out, BG, gs, S, kv_stride,
                             scale, workspace, workspace_bytes, true, stream);
}

int ri_prepare_wave_attention(AttendParams* out_params, const void* q, const void* steady_k, const void* steady_v,
                              int64_t steady_stride, int static_len, const int32_t* static_len_dev, const void* store_k,
                              const void* store_v, int64_t store_stride, const int32_t* row_src, int row_src_stride,
                              const int32_t* ret_tok_off, const int32_t* ret_start, int np, const int32_t* meta,
                              const int32_t* est_ids, const float* logits, const void* est_centroids, const void* value_sum,
                              const void* cluster_size_bf16, void* out, int32_t* valid_lengths, int BG, int gs, int nc,
                              int es, float scale, void* scratch, size_t scratch_bytes, int plan) {
  if (!q || !steady_k || !steady_v || !store_k || !store_v || !meta || !out || !scratch) return RI_ERR_ARG;
  if (ri_any_misaligned16(q, steady_k, steady_v, store_k, store_v, value_sum, est_centroids, out, scratch))
    return RI_ERR_ARG;
  if (!row_src && (!ret_tok_off || !ret_start || np <= 0 || np > RI_MAX_PROBES)) return RI_ERR_ARG;
  if ((row_src && row_src_stride <= 0) || store_stride < 0) return RI_ERR_ARG;
  if (BG <= 0 || BG > RI_MAX_GROUPS || gs <= 0 || gs > 16 || static_len < 0 || static_len > steady_stride ||
      es < 0 || nc <= 0)
    return RI_ERR_ARG;
  if (es > 0 && (!est_ids || (!logits == !est_centroids) || !value_sum || !cluster_size_bf16)) return RI_ERR_ARG;
  const int gp = gs_pad_of(gs);
  AttendParams P = {};
  P.q = (const uint16_t*)q;
  P.kA = (const uint16_t*)steady_k;
  P.vA = (const uint16_t*)steady_v;
  P.strideA = steady_stride;
  P.lenA = static_len;
  P.lenA_ptr = static_len_dev;
  // (a store without rows: its table has only entries that are skipped, and the row read for them is the query's)
  P.kB = (const uint16_t*)(store_stride > 0 ? store_k : q);
  P.vB = (const uint16_t*)(store_stride > 0 ? store_v : q);
  P.strideB = store_stride;
  P.row_src = row_src;
  P.rs_stride = row_src_stride;
  P.src_hi = INT32_MAX;   // (an entry below 0 is padding in every window)
  if (!row_src) {
    P.ret_off = ret_tok_off;
    P.ret_start = ret_start;
    P.np = np;
  }
  P.lenB_ptr = meta + 1;
  P.lenB_ptr_stride = 4;
  P.est_ids = est_ids;
  P.logits = logits;
  P.est_cent = (const uint16_t*)est_centroids;
  P.value_sum = (const uint16_t*)value_sum;
  P.csize = (const uint16_t*)cluster_size_bf16;
  P.nc = nc;
  P.es = es;
  P.gs = gs;
  P.scale = scale;
  P.out = (uint16_t*)out;
  P.valid_lengths = valid_lengths;
  // the retrieved-token count is only known on the device: size the split for the row table
  // capacity scaled by the usual fill (a quarter) or for 16 tokens per rank, the estimation zone by
  // its exact size
  plan_splits(P, static_len + (row_src ? row_src_stride / 4 : np * 16), es,
              est_row_bytes(gs, est_centroids != nullptr), BG, gs, plan == ATT_ONE ? 1 : RI_MAX_SPLITS, plan == ATT_SEVERAL);
  if (scratch_bytes < attn_scratch_used(BG, gp, P.S)) return RI_ERR_WORKSPACE;
  carve_workspace(P, scratch, BG, gp);
  *out_params = P;
  return RI_OK;
}

// Shared body of ri_wave_attention and ri_wave_attention_static.  `scratch` holds the arrival
// counters and the split partials; with scratch_bytes == 0 the caller vouches for its size through
// scratch_limit (the static array) and the counters are cleared by a fill kernel first.
__global__ void attend_clear_counters_kernel(int* counters, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) counters[i] = 0;
}

static int wave_attention_impl(const void* q, const void* steady_k, const void* steady_v, int64_t steady_stride,
                               int static_len, const int32_t* static_len_dev, const void* store_k,
                               const void* store_v, int64_t store_stride, const int32_t* row_src,
                               int row_src_stride, const int32_t* ret_tok_off, const int32_t* ret_start, int np,
                               const int32_t* meta, const int32_t* est_ids, const float* logits,
                               const void* est_centroids, const void* value_sum, const void* cluster_size_bf16,
                               void* out, int32_t* valid_lengths, int BG, int gs, int nc, int es, float scale,
                               void* scratch, size_t scratch_bytes, bool clear_counters, bool half, hipStream_t stream,
                               int src_lo = INT32_MIN, int src_hi = INT32_MAX, const void* prev_out = nullptr,
                               const float* prev_lse = nullptr, float* lse_out = nullptr) {
  if ((prev_out == nullptr) != (prev_lse == nullptr) || ri_misaligned16(prev_out)) return RI_ERR_ARG;
  AttendParams P;
  const int rc = ri_prepare_wave_attention(&P, q, steady_k, steady_v, steady_stride, static_len, static_len_dev, store_k,
                                           store_v, store_stride, row_src, row_src_stride, ret_tok_off, ret_start, np, meta,
                                           est_ids, logits, est_centroids, value_sum, cluster_size_bf16, out, valid_lengths,
                                           BG, gs, nc, es, scale, scratch, scratch_bytes, ATT_PLAN);
  if (rc) return rc;
  P.src_lo = max(src_lo, 0);
  P.src_hi = src_hi;
  P.prev_out = (const uint16_t*)prev_out;
  P.prev_lse = prev_lse;
  P.lse_out = lse_out;
  if (clear_counters) {
    attend_clear_counters_kernel<<<RI_MAX_GROUPS / 256, 256, 0, stream>>>(P.counters, RI_MAX_GROUPS);
    RI_HIP_CHECK_LAUNCH();
  }
  return launch_attend(P, BG, gs, half, stream);
}

// Clears the arrival counters at the head of an attention workspace with a small kernel on `stream` (no
// memset: the call can be captured).  Every attention launch leaves its counters at zero, so this is only
// needed after a launch that did not run to its end (a fault, a device reset): its groups' counters may be
// left non-zero, and later launches on that workspace would then never see a last arrival and write nothing.
extern "C" int ri_attention_workspace_reset(void* workspace, size_t workspace_bytes, ri_stream_t stream) {
  if (!workspace || ri_misaligned16(workspace)) return RI_ERR_ARG;
  if (workspace_bytes < RI_MAX_GROUPS * sizeof(int)) return RI_ERR_WORKSPACE;
  attend_clear_counters_kernel<<<(RI_MAX_GROUPS + 255) / 256, 256, 0, (hipStream_t)stream>>>((int*)workspace,
                                                                                             RI_MAX_GROUPS);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

static int ri_wave_attention_any(const void* q, const void* steady_k, const void* steady_v,
                                 int64_t steady_stride, int static_len, const int32_t* static_len_dev,
                                 const void* store_k,
                                 const void* store_v, int64_t store_stride, const int32_t* row_src,
                                 int row_src_stride, const int32_t* ret_tok_off, const int32_t* ret_start, int np,
                                 const int32_t* meta, const int32_t* est_ids,
                                 const float* logits, const void* est_centroids, const void* value_sum,
                                 const void* cluster_size_bf16, void* out, int32_t* valid_lengths, int BG, int gs,
                                 int nc, int es, float scale, void* workspace, size_t workspace_bytes,
                                 ri_stream_t stream, bool half) {
  if (workspace && workspace_bytes < attn_workspace_bytes(BG, gs)) return RI_ERR_WORKSPACE;
  return wave_attention_impl(q, steady_k, steady_v, steady_stride, static_len, static_len_dev, store_k, store_v,
                             store_stride, row_src, row_src_stride, ret_tok_off, ret_start, np, meta, est_ids, logits,
                             est_centroids, value_sum, cluster_size_bf16, out, valid_lengths, BG, gs, nc, es, scale,
                             workspace, workspace_bytes, false, half, (hipStream_t)stream);
}

extern "C" int ri_wave_attention(const void* q, const void* steady_k, const void* steady_v,
                                 int64_t steady_stride, int static_len, const int32_t* static_len_dev,
                                 const void* store_k,
                                 const void* store_v, int64_t store_stride, const int32_t* row_src,
                                 int row_src_stride, const int32_t* ret_tok_off, const int32_t* ret_start, int np,
                                 const int32_t* meta, const int32_t* est_ids,
                                 const float* logits, const void* est_centroids, const void* value_sum,
                                 const void* cluster_size_bf16, void* out, int32_t* valid_lengths, int BG, int gs,
                                 int nc, int es, float scale, void* workspace, size_t workspace_bytes,
                                 ri_stream_t stream) {
  return ri_wave_attention_any(q, steady_k, steady_v, steady_stride, static_len, static_len_dev, store_k, store_v, store_stride, row_src, row_src_stride, ret_tok_off, ret_start, np, meta, est_ids, logits, est_centroids, value_sum, cluster_size_bf16, out, valid_lengths, BG, gs, nc, es, scale, workspace, workspace_bytes, stream, false);
}

extern "C" int ri_wave_attention_f16(const void* q, const void* steady_k, const void* steady_v,
                                 int64_t steady_stride, int static_len, const int32_t* static_len_dev,
                                 const void* store_k,
                                 const void* store_v, int64_t store_stride, const int32_t* row_src,
                                 int row_src_stride, const int32_t* ret_tok_off, const int32_t* ret_start, int np,
                                 const int32_t* meta, const int32_t* est_ids,
                                 const float* logits, const void* est_centroids, const void* value_sum,
                                 const void* cluster_size_bf16, void* out, int32_t* valid_lengths, int BG, int gs,
                                 int nc, int es, float scale, void* workspace, size_t workspace_bytes,
                                 ri_stream_t stream) {
  return ri_wave_attention_any(q, steady_k, steady_v, steady_stride, static_len, static_len_dev, store_k, store_v, store_stride, row_src, row_src_stride, ret_tok_off, ret_start, np, meta, est_ids, logits, est_centroids, value_sum, cluster_size_bf16, out, valid_lengths, BG, gs, nc, es, scale, workspace, workspace_bytes, stream, true);
}

// Part of a wave attention: the steady zone and estimation zone as asked for, and of the rows of the row
// table only those whose source row lies in [src_row_lo, src_row_hi); an earlier part's result comes in
// as (prev_out, prev_lse) and this part's log-sum-exp goes out, so that two launches over disjoint row
// windows give the attention over all rows.  Used with a host-resident store: the rows already in the
// block cache are attended while the missed blocks are still being staged, and the staged rows follow.
static int ri_wave_attention_part_any(const void* q, const void* steady_k, const void* steady_v,
                                      int64_t steady_stride, int static_len, const int32_t* static_len_dev,
                                      const void* store_k, const void* store_v, int64_t store_stride,
                                      const int32_t* row_src, int row_src_stride, int src_row_lo, int src_row_hi,
                                      const int32_t* meta, const int32_t* est_ids, const float* logits,
                                      const void* value_sum, const void* cluster_size_bf16, const void* prev_out,
                                      const float* prev_lse, void* out, float* lse_out, int32_t* valid_lengths,
                                      int BG, int gs, int nc, int es, float scale, void* workspace,
                                      size_t workspace_bytes, ri_stream_t stream, bool half) {
  if (!row_src || src_row_lo > src_row_hi) return RI_ERR_ARG;   // an empty window attends none of the table's rows
  if (workspace && workspace_bytes < attn_workspace_bytes(BG, gs)) return RI_ERR_WORKSPACE;
  // a part that leaves the steady zone out must not pick its length up from the device either
  if (static_len == 0) static_len_dev = nullptr;
  return wave_attention_impl(q, steady_k, steady_v, steady_stride, static_len, static_len_dev, store_k, store_v,
                             store_stride, row_src, row_src_stride, nullptr, nullptr, 0, meta, est_ids, logits, nullptr,
                             value_sum, cluster_size_bf16, out, valid_lengths, BG, gs, nc, es, scale, workspace,
                             workspace_bytes, false, half, (hipStream_t)stream, src_row_lo, src_row_hi, prev_out, prev_lse,
                             lse_out);
}

extern "C" int ri_wave_attention_part(const void* q, const void* steady_k, const void* steady_v,
                                      int64_t steady_stride, int static_len, const int32_t* static_len_dev,
                                      const void* store_k, const void* store_v, int64_t store_stride,
                                      const int32_t* row_src, int row_src_stride, int src_row_lo, int src_row_hi,
                                      const int32_t* meta, const int32_t* est_ids, const float* logits,
                                      const void* value_sum, const void* cluster_size_bf16, const void* prev_out,
                                      const float* prev_lse, void* out, float* lse_out, int32_t* valid_lengths,
                                      int BG, int gs, int nc, int es, float scale, void* workspace,
                                      size_t workspace_bytes, ri_stream_t stream) {
  return ri_wave_attention_part_any(q, steady_k, steady_v, steady_stride, static_len, static_len_dev, store_k, store_v, store_stride, row_src, row_src_stride, src_row_lo, src_row_hi, meta, est_ids, logits, value_sum, cluster_size_bf16, prev_out, prev_lse, out, lse_out, valid_lengths, BG, gs, nc, es, scale, workspace, workspace_bytes, stream, false);
}

extern "C" int ri_wave_attention_part_f16(const void* q, const void* steady_k, const void* steady_v,
                                      int64_t steady_stride, int static_len, const int32_t* static_len_dev,
                                      const void* store_k, const void* store_v, int64_t store_stride,
                                      const int32_t* row_src, int row_src_stride, int src_row_lo, int src_row_hi,
                                      const int32_t* meta, const int32_t* est_ids, const float* logits,
                                      const void* value_sum, const void* cluster_size_bf16, const void* prev_out,
                                      const float* prev_lse, void* out, float* lse_out, int32_t* valid_lengths,
                                      int BG, int gs, int nc, int es, float scale, void* workspace,
                                      size_t workspace_bytes, ri_stream_t stream) {
  return ri_wave_attention_part_any(q, steady_k, steady_v, steady_stride, static_len, static_len_dev, store_k, store_v, store_stride, row_src, row_src_stride, src_row_lo, src_row_hi, meta, est_ids, logits, value_sum, cluster_size_bf16, prev_out, prev_lse, out, lse_out, valid_lengths, BG, gs, nc, es, scale, workspace, workspace_bytes, stream, true);
}

// ------------------------------------------------------------------------------------
// The same attention for callers that cannot allocate (code under stream capture, serving loops,
// harnesses that forbid hipMalloc): arrival counters and split partials live in a static device
// array of RI_STATIC_SCRATCH_BYTES that every GPU holds from the moment the library is loaded.
// Its address is looked up once per device; host code only ever uses that address.
// ------------------------------------------------------------------------------------
#define RI_STATIC_SCRATCH_BYTES (8u << 20)
#define RI_MAX_DEVICES 64
static __device__ __align__(256) unsigned char scratch[RI_STATIC_SCRATCH_BYTES];
static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[RI_MAX_DEVICES] = {};

// device address of this GPU's copy of `scratch` (looked up on the first call on the device)
static int static_scratch_ptr(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) { ri_set_last_hip_error((int)e); return RI_ERR_LAUNCH; }
  if (dev < 0 || dev >= RI_MAX_DEVICES) return RI_ERR_ARG;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) { ri_set_last_hip_error((int)e); return RI_ERR_LAUNCH; }
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return RI_OK;
}

// (also looks the array's address up on the current device, so that a caller who asks for the size before
// capturing a stream has the first-call work behind it: the look-up can load the code object)
extern "C" size_t ri_wave_attention_static_scratch_bytes(void) {
  void* ptr = nullptr;
  (void)static_scratch_ptr(&ptr);
  return RI_STATIC_SCRATCH_BYTES;
}

static int ri_wave_attention_static_any(const void* q, const void* steady_k, const void* steady_v,
                                        int64_t steady_stride, int static_len, const int32_t* static_len_dev,
                                        const void* store_k, const void* store_v, int64_t store_stride,
                                        const int32_t* row_src, int row_src_stride, const int32_t* ret_tok_off,
                                        const int32_t* ret_start, int np, const int32_t* meta,
                                        const int32_t* est_ids, const float* logits, const void* est_centroids,
                                        const void* value_sum, const void* cluster_size_bf16, void* out,
                                        int32_t* valid_lengths, int BG, int gs, int nc, int es, float scale,
                                        ri_stream_t stream, bool half) {
  void* ptr = nullptr;
  const int rc = static_scratch_ptr(&ptr);
  if (rc) return rc;
  // the array keeps what the previous call left: the counters are cleared by a kernel on the caller's
  // stream (a fill kernel, not a memset, so that the call can be captured into a graph)
  return wave_attention_impl(q, steady_k, steady_v, steady_stride, static_len, static_len_dev, store_k, store_v,
                             store_stride, row_src, row_src_stride, ret_tok_off, ret_start, np, meta, est_ids, logits,
                             est_centroids, value_sum, cluster_size_bf16, out, valid_lengths, BG, gs, nc, es, scale, ptr,
                             RI_STATIC_SCRATCH_BYTES, true, half, (hipStream_t)stream);
}

extern "C" int ri_wave_attention_static(const void* q, const void* steady_k, const void* steady_v,
                                        int64_t steady_stride, int static_len, const int32_t* static_len_dev,
                                        const void* store_k, const void* store_v, int64_t store_stride,
                                        const int32_t* row_src, int row_src_stride, const int32_t* ret_tok_off,
                                        const int32_t* ret_start, int np, const int32_t* meta,
                                        const int32_t* est_ids, const float* logits, const void* est_centroids,
                                        const void* value_sum, const void* cluster_size_bf16, void* out,
                                        int32_t* valid_lengths, int BG, int gs, int nc, int es, float scale,
                                        ri_stream_t stream) {
  return ri_wave_attention_static_any(q, steady_k, steady_v, steady_stride, static_len, static_len_dev, store_k, store_v, store_stride, row_src, row_src_stride, ret_tok_off, ret_start, np, meta, est_ids, logits, est_centroids, value_sum, cluster_size_bf16, out, valid_lengths, BG, gs, nc, es, scale, stream, false);
}

extern "C" int ri_wave_attention_static_f16(const void* q, const void* steady_k, const void* steady_v,
                                        int64_t steady_stride, int static_len, const int32_t* static_len_dev,
                                        const void* store_k, const void* store_v, int64_t store_stride,
                                        const int32_t* row_src, int row_src_stride, const int32_t* ret_tok_off,
                                        const int32_t* ret_start, int np, const int32_t* meta,
                                        const int32_t* est_ids, const float* logits, const void* est_centroids,
                                        const void* value_sum, const void* cluster_size_bf16, void* out,
                                        int32_t* valid_lengths, int BG, int gs, int nc, int es, float scale,
                                        ri_stream_t stream) {
  return ri_wave_attention_static_any(q, steady_k, steady_v, steady_stride, static_len, static_len_dev, store_k, store_v, store_stride, row_src, row_src_stride, ret_tok_off, ret_start, np, meta, est_ids, logits, est_centroids, value_sum, cluster_size_bf16, out, valid_lengths, BG, gs, nc, es, scale, stream, true);
}

static int ri_buffer_attention_any(const void* q, const void* buf_k, const void* buf_v, int64_t buf_stride,
                                   const int32_t* cache_seqlens, int max_len, const int32_t* est_ids,
                                   const float* logits, const void* value_sum, const void* cluster_size_bf16,
                                   void* out, int BG, int gs, int nc, int es, float scale, void* workspace,
                                   size_t workspace_bytes, ri_stream_t stream, bool half) {
  if (!q || !buf_k || !buf_v || !cache_seqlens || !out || !workspace) return RI_ERR_ARG;
  if (ri_any_misaligned16(q, buf_k, buf_v, value_sum, out, workspace)) return RI_ERR_ARG;
  if (BG <= 0 || BG > RI_MAX_GROUPS || gs <= 0 || gs > 16 || max_len <= 0 || max_len > buf_stride || es < 0 ||
      nc <= 0)
    return RI_ERR_ARG;
  if (es > 0 && (!est_ids || !logits || !value_sum || !cluster_size_bf16)) return RI_ERR_ARG;
  if (workspace_bytes < attn_workspace_bytes(BG, gs)) return RI_ERR_WORKSPACE;
  const int gp = gs_pad_of(gs);
  AttendParams P = {};
  P.q = (const uint16_t*)q;
  P.kA = P.kB = (const uint16_t*)buf_k;
  P.vA = P.vB = (const uint16_t*)buf_v;
  P.strideA = P.strideB = buf_stride;
  P.lenA = 0;
  P.lenB_ptr = cache_seqlens;
  P.lenB_ptr_stride = 1;
  P.lenB_const = max_len;
  P.est_ids = est_ids;
  P.logits = logits;
  P.value_sum = (const uint16_t*)value_sum;
  P.csize = (const uint16_t*)cluster_size_bf16;
  P.nc = nc;
  P.es = es;
  P.gs = gs;
  P.scale = scale;
  P.out = (uint16_t*)out;
  // the valid lengths are only known on the device: size the split for a quarter of the buffer
  plan_splits(P, max_len / 4 + 64, es, est_row_bytes(gs, false), BG, gs);
  carve_workspace(P, workspace, BG, gp);
  return launch_attend(P, BG, gs, half, (hipStream_t)stream);
}

extern "C" int ri_buffer_attention(const void* q, const void* buf_k, const void* buf_v, int64_t buf_stride,
                                   const int32_t* cache_seqlens, int max_len, const int32_t* est_ids,
                                   const float* logits, const void* value_sum, const void* cluster_size_bf16,
                                   void* out, int BG, int gs, int nc, int es, float scale, void* workspace,
                                   size_t workspace_bytes, ri_stream_t stream) {
  return ri_buffer_attention_any(q, buf_k, buf_v, buf_stride, cache_seqlens, max_len, est_ids, logits, value_sum, cluster_size_bf16, out, BG, gs, nc, es, scale, workspace, workspace_bytes, stream, false);
}

extern "C" int ri_buffer_attention_f16(const void* q, const void* buf_k, const void* buf_v, int64_t buf_stride,
                                   const int32_t* cache_seqlens, int max_len, const int32_t* est_ids,
                                   const float* logits, const void* value_sum, const void* cluster_size_bf16,
                                   void* out, int BG, int gs, int nc, int es, float scale, void* workspace,
                                   size_t workspace_bytes, ri_stream_t stream) {
  return ri_buffer_attention_any(q, buf_k, buf_v, buf_stride, cache_seqlens, max_len, est_ids, logits, value_sum, cluster_size_bf16, out, BG, gs, nc, es, scale, workspace, workspace_bytes, stream, true);
}

