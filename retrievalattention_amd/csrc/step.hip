// The decode step of one layer as two calls with few arguments (gfx950): appending the new token's K/V to the
// steady zone, and scoring + selection + attention over a device-resident cluster store.
//
// A short context's step is bound by what the host spends on it, not by the GPU: through torch's slice copies and one
// wrapper call per stage a layer-step took 46 us of host time, of which the launches are 1 us each.  The addresses and
// sizes of a layer do not change from token to token, so the caller keeps them in one struct and hands over its address.
#include "attend_common.h"
#include "lru_body.h"
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

// The selection's bins and rank arrays lie where the attention's value tiles will.
template <int NT>
__device__ __forceinline__ uint32_t* select_scratch() {
  static_assert(SEL_SCRATCH<NT> * sizeof(uint32_t) <= ATT_WAVES * 16 * ATT_VT_STRIDE * sizeof(uint16_t), "room for them");
  return reinterpret_cast<uint32_t*>(att_tiles());
}

// What a selection with KEEP_TABLES left in LDS goes to memory, by one of the workgroups that made it and when its rows are
// attended.
__device__ __forceinline__ void store_selection(const SelectArgs& S, int g, const SelectKept& K) {
  const int np = S.np, es = S.es, tid = threadIdx.x;
  for (int i = tid; i < np; i += 64 * ATT_WAVES) {
    S.ret_ids[(size_t)g * np + i] = K.ids[i];
    S.ret_start[(size_t)g * np + i] = K.start[i];
  }
  for (int i = tid; i <= np; i += 64 * ATT_WAVES) S.ret_tok_off[(size_t)g * (np + 1) + i] = K.off[i];
  for (int i = tid; i < es; i += 64 * ATT_WAVES) S.est_ids[(size_t)g * es + i] = K.est[i];
  if (tid < 4) S.meta[g * 4 + tid] = K.meta[tid];
}

// ------------------------------------------------------------------------------------
// step: scoring, selection and attention of a group in one launch, for short contexts.
// With up to 512 clusters the selection is one workgroup per group that scores for itself: as one kernel with the attention
// the second half finds ids, tables and logits in LDS, and a launch is left out, which counts on the
// host as well.  What bounds it is the chain of either half on one compute unit.  Captured layers with their appends, in launches of
// their own -> one, us: 8 groups of 4 heads, 512 clusters, 331 rows 18.0 -> 16.3; 8 heads 19.0 -> 17.8; 128 groups of 4 20.7 -> 18.7.
// 103564 bytes of LDS (113036 with 8 heads): one workgroup per compute unit, hence at most 256 groups; more
// heads: launch_score_attend.
// SPLIT: several workgroups per group, which all make the same selection and attend a part of the rows each (see
// select_attend_kernel): with the query and the zone's length requested behind the first loads and the results stored behind
// the attention, the launch takes much the same at any length.  8 groups of 8 heads, 512 clusters, 331 / 521 / 831 / 1331 rows:
// 17.8 / 20.2 / 21.9 / 27.3 us with one workgroup, 17.0 / 17.1 / 17.0 / 18.6 with several (19.0 / 19.2 / 19.0 / 20.3 in launches of their own);
// the retrieval of 10 % of the clusters, launches of their own -> SPLIT, 8 groups of 8 heads 22.1 -> 20.1, 16 of 4 21.3 -> 19.5, 128 of 8
// 35.0 -> 32.4.  step_route.h says which step takes which form.  The rows that the clusters hold, and the zone's in a captured
// step, are known behind the selection only: where they turn out to be few, one workgroup attends them all and hands no partial
// over, and another stores the results (8 groups of 1 head, 256 clusters 15.8 -> 14.8 us, of 4 heads 16.2 -> 15.0, 128 of 8, 512 23.9 ->
// 22.9; 8 of 8, 512 17.1 either way).
// The scoring half is bound by its instructions and waits, not by the centroids' bytes (a quarter of them takes as long): with
// its own statistics and those of the eight waves made without branches, the clusters' masks not looked at in front of the other
// loads, and the results stored behind the attention by one workgroup as by several, captured layers took 16.05 -> 15.5 us (8
// groups of 4 heads, 8192 tokens), 17.3 -> 16.4 (8 of 8), 16.55 -> 15.95 (16 of 4), 17.35 -> 16.7 (32 of 4, 8000).
// ------------------------------------------------------------------------------------
// (what the first loads want stands before the structs: in registers at the start; 64 groups of 8 heads 15.3 -> 15.0 us, 8 of 4
// the same)
template <int GSM, bool HALF, bool SPLIT>
__global__ __launch_bounds__(64 * ATT_WAVES) void step_kernel(ri_ptr4 in, ri_int4 n, float scale, int one_rows,
                                                           SelectArgs S0, AttendParams A0) {
  static_assert(64 * ATT_WAVES == STEP_CLUSTERS, "a cluster per thread");
  __shared__ __attribute__((aligned(16))) float sh_logits[STEP_CLUSTERS * GSM];
  static_assert(__alignof__(sh_logits) == 16, "read four heads at a time");
  __shared__ int sh_est[STEP_CLUSTERS], sh_off[STEP_CLUSTERS + 1], sh_start[STEP_CLUSTERS], sh_ids[STEP_CLUSTERS],
      sh_meta[4];
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
  const SelectKept kept = {sh_logits, sh_est, sh_off, sh_start, sh_ids, sh_meta, select_scratch<STEP_CLUSTERS>(), nullptr};
  AttendKept known = {sh_logits, sh_est, sh_off, sh_start};
  uint4 query;
  select_group<STEP_CLUSTERS, 1, GSM, HALF, SEL_SCORE, KEEP_TABLES>(S, blockIdx.x, kept, [&] {
    query = att_query_piece(A, blockIdx.x);
    known.lenA = att_steady_rows(A);
    att_clear<GSM>();
  });
  att_put_query<GSM>(query, S.gs);
  lds_barrier();
  // (the same in all of the group's workgroups)
  const bool one = SPLIT && __builtin_amdgcn_readfirstlane(known.lenA + sh_off[S.np]) + S.es <= one_rows;
  if (one) {
    A.S = 1;
    A.W_kv = A.W_one;
    A.inv_kv = A.inv_kv_one;
    A.inv_es = A.inv_es_one;
  }
  if (!one || blockIdx.y == 0)
    attend_group<GSM, HALF, SPLIT ? KEPT_LOGITS : KEPT_ALL>(A, blockIdx.x, SPLIT ? blockIdx.y : 0, known);
  if (blockIdx.y == (one && gridDim.y > 1 ? 1 : 0)) {
    store_selection(S, blockIdx.x, kept);
    const int nc = S.nc;
    for (int j = 0; j < S.gs; ++j)
      if ((int)threadIdx.x < nc) S.logits[((size_t)blockIdx.x * S.gs + j) * nc + threadIdx.x] = sh_logits[threadIdx.x * GSM + j];
  }
}

// ------------------------------------------------------------------------------------
// select + attend, behind the scoring: the attention's workgroups of a group each make the group's selection and go on with its
// tables in LDS.  The compute units that repeat it would wait for it otherwise; a launch, and the tables' way through memory, are
// left out.  The query's pieces and the zone's length are requested before the selection looks at anything (behind its own first
// loads: in front of them, with a wait for the struct's words and a load per head's partials under a condition, steps took 17.6
// instead of 17.15 us in the first of the shapes below, 44.5 / 43.6 in the second, 22.5 / 21.7 for 12 of 7 heads, 1856 in half,
// 127.5 / 126.0 in the fourth), and one of the workgroups stores its
// results when its rows are attended (a load's wait covers the stores in front of it): without both 19.0, 47.5 and 26.2 us in
// the first, second and third of these steps (captured, 4 layers a graph; in launches of their own -> joined): 16 groups of 4
// heads, 1024 clusters 20.4 -> 18.0; 32 of 4, 8192 48.0 -> 45.1; 12 of 7, 1920 half 24.8 -> 22.6; 64 of 8, 16384 130.8 -> 128.1; 8 of
// 4, 2048 21.7 -> 19.6; 1 of 4, 8192 25.2 -> 23.0; 8 of 8, 4096 27.6 -> 23.8; 32 of 16, 4096 38.9 -> 36.2; 4 of 12, 8192 32.4 ->
// 30.2; 16 of 1, 1920 22.2 -> 19.7; 320 of 8, 1280 72.6 -> 67.4; 512 of 4, 1024 74.4 -> 70.5.
// What bounds it is the selection's chain (see select_body.h), then what bounds the attention.
// NT: threads that select; the attention is eight waves' always, and the others leave before it (a barrier counts the waves
// there are).  512 up to 8192 clusters (512 / 1024 threads: 16 groups of 4 heads, 1024 17.9 / 19.6, 8 of 4, 2048 19.4 / 20.7, 12 of 7, 1920 22.0
// / 23.8, 32 of 8, 4096 31.1 / 31.6, 32 of 4, 8192 44.0 / 44.3, 8 of 4 25.8 / 25.9), 1024 past them, where it makes no difference any
// more (64 of 8, 16384 127.9 / 128.2, 8 of 4 33.4 / 33.2), and for more than 512 probes, which 512 threads do not hold (in launches of
// their own -> joined: 32 of 4, 8192 clusters, 819 probes 85.5 -> 81.9; 12 of 7, 5632, 563 42.2 -> 39.2; 64 of 8, 8192, 819 150.8 ->
// 146.9).
// ------------------------------------------------------------------------------------
template <int NT, int E, int GSM, bool HALF, int SRC>
__global__ __launch_bounds__(NT, NT / 256) void select_attend_kernel(ri_ptr4 in, ri_int4 n, ri_int2 m, SelectArgs S0,
                                                                          AttendParams A0) {
  extern __shared__ __attribute__((aligned(16))) int sh_kept[];
  SelectArgs S = S0;
  AttendParams A = A0;
  if (SRC == SEL_KEYS) {
    S.keys = ri_global<uint16_t>(in[0]);
  } else if (SRC == SEL_SCORE) {
    S.cent = ri_global<const uint16_t>(in[0]);
    S.q = A.q = ri_global<const uint16_t>(in[1]);
    S.cluster_size = ri_global<const int32_t>(in[2]);
  } else {
    S.logits = ri_global<float>(in[0]);
    S.tile_max = ri_global<float>(in[1]);
    S.tile_sum = ri_global<float>(in[2]);
  }
  S.mask = ri_global<const uint8_t>(in[3]);
  S.nc = A.nc = n[0];
  S.gs = A.gs = n[1];
  S.np = A.np = n[2];
  S.es = A.es = n[3];
  S.ntiles = m[0] & 0xffff;
  A.S = m[0] >> 16;
  A.W_kv = m[1];
  const int np = S.np, g = blockIdx.x;
  int *const meta = sh_kept, *const off = meta + 4, *const start = off + np + 1, *const ids = start + np, *const est = ids + np;
  static_assert(SRC != SEL_SCORE || SEL_AREA<NT, GSM> <= (size_t)ATT_WAVES * GSM * RI_DIM * sizeof(float), "room in the numerators");
  static_assert(SRC != SEL_SCORE || GSM == 16, "step_kernel's otherwise");
  const SelectKept kept = {nullptr, est, off, start, ids, meta, select_scratch<NT>(),
                           SRC == SEL_SCORE ? reinterpret_cast<uint4*>(att_numerators<GSM>()) : nullptr};
  AttendKept known = {nullptr, est, off, start};
  uint4 query;
  select_group<NT, E, GSM, HALF, SRC, KEEP_TABLES>(S, g, kept, [&] {
    query = att_query_piece(A, g);
    known.lenA = att_steady_rows(A);
    att_clear<GSM>();
  });
  att_put_query<GSM>(query, S.gs);
  if (SRC == SEL_SCORE) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the logits, which other waves read back)
  lds_barrier();
  if (NT > 64 * ATT_WAVES && threadIdx.x >= 64 * ATT_WAVES) return;
  attend_group<GSM, HALF, KEPT_TABLES>(A, g, blockIdx.y, known);
  if (blockIdx.y == 0) store_selection(S, g, kept);
}

template <int NT, int E, int SRC>
static void launch_select_attend(const SelectArgs& S, const AttendParams& A, int BG, bool half, hipStream_t stream) {
  const void* a = SRC == SEL_KEYS ? (const void*)S.keys : (const void*)S.logits;
  // (sixteen heads: up to 512 threads, and no logits past 2048 clusters; more than 8192 clusters in so few: sixteen heads)
  constexpr int LEAST = NT == 512 && E == 32 ? 16 : 4, MOST = NT == 512 && !(SRC == SEL_LOGITS && E == 8) ? 16 : 8;
  constexpr int G4 = LEAST > 4 ? LEAST : 4, G8 = LEAST > 8 ? LEAST : 8, G16 = MOST;
  auto* kernel = S.gs <= 4   ? (half ? select_attend_kernel<NT, E, G4, true, SRC> : select_attend_kernel<NT, E, G4, false, SRC>)
                 : S.gs <= 8 ? (half ? select_attend_kernel<NT, E, G8, true, SRC> : select_attend_kernel<NT, E, G8, false, SRC>)
                             : (half ? select_attend_kernel<NT, E, G16, true, SRC> : select_attend_kernel<NT, E, G16, false, SRC>);
  const size_t lds = (size_t)(4 + 3 * S.np + 1 + S.es) * sizeof(int);
  kernel<<<dim3(BG, A.S), NT, lds, stream>>>(ri_pack_ptrs(a, S.tile_max, S.tile_sum, S.mask),
                                                         (ri_int4){S.nc, S.gs, S.np, S.es}, (ri_int2){S.ntiles | A.S << 16, A.W_kv}, S,
                                                         A);
}

// More than eight heads over few clusters: scoring, selection and attention in one launch too, but the logits go to memory, from
// which the attention's waves read them back (every workgroup of a group writes the same ones), and the selection's rows and
// probabilities lie where the numerators will: LDS holds no more. What bounds it is the same chain as step_kernel's. Captured layers with their
// appends, us, selection and attention in launches of their own / as it is: 8 groups of 16 heads, 480 clusters 19.15 / 17.25; of 12, 256 16.8 / 15.1;
// 1 of 12, 192 15.7 / 14.3; 32 of 16, 512 20.0 / 17.9; 2 of 16, 160 16.6 / 15.2; 128 of 12, 384 19.9 / 17.8; 16 of 12, 448 17.65 / 15.7.
static void launch_score_attend(const SelectArgs& S, const AttendParams& A, int BG, bool half, hipStream_t stream) {
  auto* kernel = half ? select_attend_kernel<512, 1, 16, true, SEL_SCORE> : select_attend_kernel<512, 1, 16, false, SEL_SCORE>;
  const size_t lds = (size_t)(4 + 3 * S.np + 1 + S.es) * sizeof(int);
  kernel<<<dim3(BG, A.S), 512, lds, stream>>>(ri_pack_ptrs(S.cent, S.q, S.cluster_size, S.mask), (ri_int4){S.nc, S.gs, S.np, S.es},
                                              (ri_int2){S.ntiles | A.S << 16, A.W_kv}, S, A);
}

template <bool SPLIT>
static void launch_step(const SelectArgs& S, const AttendParams& A, int BG, bool half, hipStream_t stream) {
  auto* kernel = S.gs <= 4 ? (half ? step_kernel<4, true, SPLIT> : step_kernel<4, false, SPLIT>)
                           : (half ? step_kernel<8, true, SPLIT> : step_kernel<8, false, SPLIT>);
  kernel<<<dim3(BG, A.S), 64 * ATT_WAVES, 0, stream>>>(ri_pack_ptrs(S.cent, S.q, S.mask, S.cluster_size),
                                                       (ri_int4){S.nc, S.gs, S.np, S.es}, S.scale, step_alone_rows(BG), S,
                                                       A);
}

// The step in one launch (nc <= STEP_CLUSTERS), or in scoring, perhaps the scores' sums, and one more.
static int step_joined(const ri_decode_step_t* s, const void* q, int static_len, bool one, void* out, hipStream_t stream) {
  SelectArgs S;
  int rc = ri_prepare_select(&S, q, s->centroids, s->mask, s->cluster_size_i32, s->cluster_start, s->logits, nullptr, nullptr,
                             s->ret_ids, s->est_ids, s->ret_tok_off, s->ret_start, nullptr, 0, s->meta, s->BG, s->gs, s->nc,
                             s->np, s->es, s->page, s->max_pages, s->scale, s->score_workspace, s->score_workspace_bytes);
  if (rc) return rc;
  if (s->attn_workspace && s->attn_workspace_bytes < ri_wave_attention_workspace_bytes(s->BG, s->gs)) return RI_ERR_WORKSPACE;
  const bool wide = step_is_wide(s);
  AttendParams A;
  rc = ri_prepare_wave_attention(&A, q, s->steady_k, s->steady_v, s->steady_stride, static_len, s->static_len_dev, s->store_k,
                                 s->store_v, s->store_stride, nullptr, 0, s->ret_tok_off, s->ret_start, s->np, s->meta,
                                 s->est_ids, s->es > 0 ? s->logits : nullptr, nullptr, s->value_sum, s->cluster_size, out,
                                 s->valid_lengths, s->BG, s->gs, s->nc, s->es, s->scale, s->attn_workspace,
                                 s->attn_workspace_bytes, one ? ATT_ONE : S.nc <= STEP_CLUSTERS && S.gs <= 8 ? ATT_SEVERAL : ATT_PLAN);
  if (rc) return rc;
  if (S.nc <= STEP_CLUSTERS) {
    if (S.gs > 8) launch_score_attend(S, A, s->BG, s->half, stream);
    else if (one) launch_step<false>(S, A, s->BG, s->half, stream);
    else launch_step<true>(S, A, s->BG, s->half, stream);
    RI_HIP_CHECK_LAUNCH();
    return RI_OK;
  }
  const bool keys = step_sums_apart(S.gs, s->BG, S.nc);
  rc = ri_launch_select_inputs(S, s->BG, s->half, keys, stream);
  if (rc) return rc;
  if (wide) {
    if (keys) {
      if (S.nc <= 8192) launch_select_attend<1024, 8, SEL_KEYS>(S, A, s->BG, s->half, stream);
      else launch_select_attend<1024, 16, SEL_KEYS>(S, A, s->BG, s->half, stream);
    } else launch_select_attend<1024, 4, SEL_LOGITS>(S, A, s->BG, s->half, stream);
  } else if (keys) {
    if (S.nc <= 4096) launch_select_attend<512, 8, SEL_KEYS>(S, A, s->BG, s->half, stream);
    else if (S.nc <= 8192) launch_select_attend<512, 16, SEL_KEYS>(S, A, s->BG, s->half, stream);
    else launch_select_attend<512, 32, SEL_KEYS>(S, A, s->BG, s->half, stream);
  } else if (S.nc <= 1024) launch_select_attend<512, 2, SEL_LOGITS>(S, A, s->BG, s->half, stream);
  else if (S.nc <= 2048) launch_select_attend<512, 4, SEL_LOGITS>(S, A, s->BG, s->half, stream);
  else launch_select_attend<512, 8, SEL_LOGITS>(S, A, s->BG, s->half, stream);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_decode_step(const ri_decode_step_t* s, const void* q, int static_len, void* out, ri_stream_t stream) {
  if (!s) return RI_ERR_ARG;
  if (step_is_joined(s)) return step_joined(s, q, static_len, step_is_one(s, static_len), out, (hipStream_t)stream);
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
  SelectArgs S;
  int rc = ri_prepare_select(&S, q, s->centroids, s->mask, nullptr, nullptr, s->logits, nullptr, nullptr, s->ret_ids,
                             s->est_ids, nullptr, nullptr, nullptr, 0, nullptr, s->BG, s->gs, s->nc, s->np, s->es, s->page,
                             s->max_pages, s->scale, s->score_workspace, s->score_workspace_bytes);
  if (rc) return rc;
  bool taken = false;
  if (ri_lru_check(*lru) == RI_OK) rc = ri_launch_select_access(S, *lru, s->BG, s->half, &taken, (hipStream_t)stream);
  if (rc) return rc;
  if (!taken) {
    rc = select(q, s->centroids, s->mask, nullptr, nullptr, s->logits, nullptr, nullptr, s->ret_ids, s->est_ids, nullptr,
                nullptr, nullptr, 0, nullptr, s->BG, s->gs, s->nc, s->np, s->es, s->page, s->max_pages, s->scale,
                s->score_workspace, s->score_workspace_bytes, stream);
    if (rc) return rc;
    if ((rc = ri_lru_access(lru, stream))) return rc;
  }
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
