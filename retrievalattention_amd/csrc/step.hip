// The decode step of one layer as two calls with few arguments (gfx950): appending the new token's K/V to the
// steady zone, and scoring + selection + attention over a device-resident cluster store.
//
// A short context's step is bound by what the host spends on it, not by the GPU: through torch's slice copies and one
// wrapper call per stage a layer-step took 46 us of host time, of which the launches are 1 us each.  The addresses and
// sizes of a layer do not change from token to token, so the caller keeps them in one struct and hands over its address.
#include "attend_common.h"
#include "select_body.h"
#include "step_route.h"

// ------------------------------------------------------------------------------------
// append: steady_k/v[g, pos] = key/value[g]; 16 lanes per 256-byte row, grid.y = K, V.
// One launch for both tensors (a slice copy each: 2.4-4.9 us per launch); the row's position is an argument
// or is read from the device, so that a captured call follows the position that the device keeps.
// ------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void append_kernel(const uint4* __restrict__ key, const uint4* __restrict__ value,
                                                     uint4* __restrict__ steady_k, uint4* __restrict__ steady_v,
                                                     int64_t stride, int64_t pos, const int64_t* __restrict__ pos_dev,
                                                     int BG) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int g = i >> 4, piece = i & 15;
  if (g >= BG) return;
  const uint4 v = (blockIdx.y ? value : key)[i];
  if (pos_dev) pos = *pos_dev;
  if (pos < 0 || pos >= stride) return;   // the steady zone is full: nothing is written past its end
  (blockIdx.y ? steady_v : steady_k)[((size_t)g * stride + pos) * 16 + piece] = v;
}

extern "C" int ri_append_kv(const void* key, const void* value, void* steady_k, void* steady_v, int64_t steady_stride,
                            int64_t pos, const int64_t* pos_dev, int BG, ri_stream_t stream) {
  if (!key || !value || !steady_k || !steady_v || BG <= 0 || steady_stride <= 0) return RI_ERR_ARG;
  if (!pos_dev && (pos < 0 || pos >= steady_stride)) return RI_ERR_ARG;
  if (ri_any_misaligned16(key, value, steady_k, steady_v)) return RI_ERR_ARG;
  append_kernel<<<dim3((BG * 16 + 255) / 256, 2), 256, 0, (hipStream_t)stream>>>(
      (const uint4*)key, (const uint4*)value, (uint4*)steady_k, (uint4*)steady_v, steady_stride, pos, pos_dev, BG);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

// ------------------------------------------------------------------------------------
// step: scoring, selection and attention of a group by one workgroup, for short contexts.
// With up to 512 clusters the selection is one workgroup per group that scores for itself, and with few rows the attention
// is, too: as one kernel the second half finds ids, tables and logits in LDS, and a launch is left out, which counts on the
// host as well.  What bounds it is the chain of either half on one compute unit.  8 groups of 4 heads, 512 clusters, 331
// rows: 14.9 -> 13.5 us; 8 heads 16.3 -> 14.7; 128 groups 17.6 -> 15.8.  110060 bytes of LDS (119532 with 8 heads): one
// workgroup per compute unit, hence at most 256 groups; sixteen heads would not fit.  step_route.h says which steps take it.
// ------------------------------------------------------------------------------------
// (what the first loads want stands before the structs: in registers at the start; 64 groups of 8 heads 15.3 -> 15.0 us, 8 of 4
// the same)
template <int GSM, bool HALF>
__global__ __launch_bounds__(64 * ATT_WAVES) void step_kernel(ri_ptr4 in, ri_int4 n, float scale, SelectArgs S0, AttendParams A0) {
  static_assert(64 * ATT_WAVES == STEP_CLUSTERS, "a cluster per thread");
  __shared__ __attribute__((aligned(16))) float sh_logits[STEP_CLUSTERS * GSM];
  static_assert(__alignof__(sh_logits) == 16, "read four heads at a time");
  __shared__ int sh_est[STEP_CLUSTERS], sh_off[STEP_CLUSTERS + 1], sh_start[STEP_CLUSTERS];
  SelectArgs S = S0;
  AttendParams A = A0;
  S.cent = ri_global<const uint16_t>(in[0]);
  S.q = A.q = ri_global<const uint16_t>(in[1]);
  S.mask = ri_global<const uint8_t>(in[2]);
  S.cluster_size = ri_global<const int32_t>(in[3]);
  S.nc = A.nc = n[0];
  S.gs = A.gs = n[1];
  S.np = A.np = n[2];
  S.es = A.es = n[3];
  S.scale = A.scale = scale;
  select_group<STEP_CLUSTERS, 1, GSM, HALF, SEL_SCORE, true>(S, blockIdx.x, SelectKept{sh_logits, sh_est, sh_off, sh_start});
  lds_barrier();
  attend_group<GSM, HALF, true>(A, blockIdx.x, 0, AttendKept{sh_logits, sh_est, sh_off, sh_start});
}

static int step_short(const ri_decode_step_t* s, const void* q, int static_len, void* out, hipStream_t stream) {
  SelectArgs S;
  int rc = ri_prepare_select(&S, q, s->centroids, s->mask, s->cluster_size_i32, s->cluster_start, s->logits, nullptr, nullptr,
                             s->ret_ids, s->est_ids, s->ret_tok_off, s->ret_start, nullptr, 0, s->meta, s->BG, s->gs, s->nc,
                             s->np, s->es, s->page, s->max_pages, s->scale, s->score_workspace, s->score_workspace_bytes);
  if (rc) return rc;
  if (s->attn_workspace && s->attn_workspace_bytes < ri_wave_attention_workspace_bytes(s->BG, s->gs)) return RI_ERR_WORKSPACE;
  AttendParams A;
  rc = ri_prepare_wave_attention(&A, q, s->steady_k, s->steady_v, s->steady_stride, static_len, s->static_len_dev, s->store_k,
                                 s->store_v, s->store_stride, nullptr, 0, s->ret_tok_off, s->ret_start, s->np, s->meta,
                                 s->est_ids, s->es > 0 ? s->logits : nullptr, nullptr, s->value_sum, s->cluster_size, out,
                                 s->valid_lengths, s->BG, s->gs, s->nc, s->es, s->scale, s->attn_workspace,
                                 s->attn_workspace_bytes, true);
  if (rc) return rc;
  auto* kernel = s->gs <= 4 ? (s->half ? step_kernel<4, true> : step_kernel<4, false>)
                            : (s->half ? step_kernel<8, true> : step_kernel<8, false>);
  kernel<<<s->BG, 64 * ATT_WAVES, 0, stream>>>(ri_pack_ptrs(S.cent, S.q, S.mask, S.cluster_size),
                                               (ri_int4){S.nc, S.gs, S.np, S.es}, S.scale, S, A);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_decode_step(const ri_decode_step_t* s, const void* q, int static_len, void* out, ri_stream_t stream) {
  if (!s) return RI_ERR_ARG;
  if (step_is_short(s, static_len)) return step_short(s, q, static_len, out, (hipStream_t)stream);
  auto* select = s->half ? ri_score_select_f16 : ri_score_select;
  auto* attend = s->half ? ri_wave_attention_f16 : ri_wave_attention;
  const int rc = select(q, s->centroids, s->mask, s->cluster_size_i32, s->cluster_start, s->logits, nullptr, nullptr,
                        s->ret_ids, s->est_ids, s->ret_tok_off, s->ret_start, nullptr, 0, s->meta, s->BG, s->gs, s->nc,
                        s->np, s->es, s->page, s->max_pages, s->scale, s->score_workspace, s->score_workspace_bytes,
                        stream);
  if (rc) return rc;
  return attend(q, s->steady_k, s->steady_v, s->steady_stride, static_len, s->static_len_dev, s->store_k, s->store_v,
                s->store_stride, nullptr, 0, s->ret_tok_off, s->ret_start, s->np, s->meta, s->est_ids,
                s->es > 0 ? s->logits : nullptr, nullptr, s->value_sum, s->cluster_size, out, s->valid_lengths, s->BG,
                s->gs, s->nc, s->es, s->scale, s->attn_workspace, s->attn_workspace_bytes, stream);
}

extern "C" int ri_host_step(const ri_decode_step_t* s, const ri_lru_t* lru, const void* q, int static_len, void* out,
                            ri_stream_t stream) {
  if (!s || !lru) return RI_ERR_ARG;
  auto* select = s->half ? ri_score_select_f16 : ri_score_select;
  auto* attend = s->half ? ri_wave_attention_f16 : ri_wave_attention;
  int rc = select(q, s->centroids, s->mask, nullptr, nullptr, s->logits, nullptr, nullptr, s->ret_ids, s->est_ids, nullptr,
                  nullptr, nullptr, 0, nullptr, s->BG, s->gs, s->nc, s->np, s->es, s->page, s->max_pages, s->scale,
                  s->score_workspace, s->score_workspace_bytes, stream);
  if (rc) return rc;
  if ((rc = ri_lru_access(lru, stream))) return rc;
  if ((rc = ri_lru_stage_update(lru, stream))) return rc;
  rc = attend(q, s->steady_k, s->steady_v, s->steady_stride, static_len, s->static_len_dev, s->store_k, s->store_v,
              s->store_stride, lru->row_src, lru->row_src_stride, nullptr, nullptr, 0, s->meta, s->est_ids,
              s->es > 0 ? s->logits : nullptr, nullptr, s->value_sum, s->cluster_size, out, s->valid_lengths, s->BG, s->gs,
              s->nc, s->es, s->scale, s->attn_workspace, s->attn_workspace_bytes, stream);
  if (rc) return rc;
  const size_t stage = (size_t)lru->stage_row0 * RI_DIM * 2;
  return ri_gather_copy_and_scatter((const char*)lru->cache_k + stage, lru->cache_k, (const char*)lru->cache_v + stage,
                                    lru->cache_v, lru->upd_buf, lru->upd_sizes, lru->upd_cache, lru->upd_num, lru->BG,
                                    (int)lru->cache_stride, (int)(lru->cache_stride / lru->block), lru->buffer_size, 0,
                                    stream);
}
