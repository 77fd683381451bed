// Device-side block cache manager for a host-resident cluster store (gfx950).
//
// Does on the GPU, without a host round trip, what the reference does on CPU
// worker threads between the top-k search and the gather:
//   BufferManager::batch_access  (library/retroinfer/retroinfer_kernels/src/wave_buffer_cpu.cpp:190-257)
//     walk the retrieved clusters in rank order, stop when their blocks no longer fit the
//     execution buffer, emit the hit list (cache block ids) and the miss list (host rows);
//   BufferManager::batch_update  (wave_buffer_cpu.cpp:102-188)
//     touch the hits, admit the longest prefix of the misses that fits the cache, evict
//     least-recently-used clusters until enough blocks are free, hand out block ids, emit the
//     admission list for the scatter kernel.
// The lists have the layout the copy kernels of gather.hip read.
//
// Recency is kept per resident cluster as a pair: the number of the last step that touched it and its order
// inside that step.  That reproduces the reference's list (wave_buffer_cpu.cpp:106-114: the hits are moved to
// the front in reverse rank order; :170-176: then the admitted misses are pushed in rank order): inside a
// step the admitted misses are the most recent, later-ranked ones first, then the hits, earlier-ranked ones
// first.  Eviction takes whole clusters from the least recent end until the request is covered, hits of the
// current step included (:140-142; their blocks have been listed for this step's attention, which runs
// before the admission copy overwrites them).  The victims are found without sorting: a radix selection over
// the step ages (8-bit digits) gives the boundary step, and inside that step the clusters are ranked by
// their order through an LDS table indexed by it.
//
// A group's workgroup is one serial chain of scans and dependent loads.  Everything the attention waits for (hits,
// misses, row table) is its first half; the second (eviction, admission) only has to be done before the admission copy.
// So the two are also launched apart, the second beside the copy of the missed rows from the host, which is bound by the
// link and leaves the compute units idle (32 groups, 3840 clusters, 10 MB of misses: access and update in one launch in
// front of the copy 27.8 + 200 us, access alone 7 and both others together 187, all with a copy that took as long by itself).
#include "lru_body.h"
#include "select_body.h"

#define LRU_COPIERS 64      // workgroups that copy missed rows

template <int R, int PHASE>
__global__ __launch_bounds__(LRU_THREADS) void lru_kernel(ri_lru_t P) {
  lru_group<R, PHASE>(P, blockIdx.x);
}

// grid groups + LRU_COPIERS: the first workgroups, one per group, update the cache's books; the others copy the missed rows of all
// groups from the host store into the staging rows, with one wave each where the items have eight rows on average, and with up to
// eight where they have fewer (the rest of a workgroup's threads leave).  The items, of at most `block` rows, are numbered through
// all groups and dealt out to the waves in turn: eight rows at a time, 16 lanes per row,
// with both halves requested before either is stored.  What is in flight is what counts: the link wants about 256 KB of it and
// carries less the more there is (32 groups, 2830 blocks of up to 8 rows, 10.2 MB, GB/s by waves: 48 55.5, 64 55.7, 128 52.1,
// 256 55.1, 512 54.3, 2048 49.6; a workgroup of sixteen waves to every eight items of a group, as many as there may be, 53.1;
// plain reads of as much in a row 55.9).  Hence the waves for short items, each of which keeps less in flight: 2880 items of 32
// groups, us with one wave to a workgroup / as many as taken here: one row 74.3 / 33.6, two rows 76.3 / 58.8, three 85.1 / 84.7, four
// 109.4 / 109.6 (one; two are 110.3 - 112.9), eight 211.1 / 211.6; 46294 rows of all lengths 420.6 / 421.2.
template <int R>
__global__ __launch_bounds__(LRU_THREADS) void lru_stage_kernel(ri_lru_t P) {
  if ((int)blockIdx.x < P.BG) {
    lru_group<R, LRU_UPDATE>(P, blockIdx.x);
    return;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), vec = lane >> 4, piece = lane & 15;
  if (wave >= 8) return;
  const auto copy = [&](int g, int j) {
    const size_t at = (size_t)g * P.buffer_size + j;
    const int rows = P.miss_sizes[at];
    const size_t src = (size_t)g * P.host_stride + P.miss_ids[at];
    const size_t dst = (size_t)g * P.cache_stride + P.stage_row0 + P.miss_cumsum[at];
    for (int r0 = 0; r0 < rows; r0 += 8) {   // (rows that there are not are not read: they would cross the link)
      const int r = r0 + vec, r2 = r + 4;
      uint4 k, v, k2, v2;
      if (r < rows) {
        k = reinterpret_cast<const uint4*>(P.host_k)[(src + r) * 16 + piece];
        v = reinterpret_cast<const uint4*>(P.host_v)[(src + r) * 16 + piece];
      }
      if (r2 < rows) {
        k2 = reinterpret_cast<const uint4*>(P.host_k)[(src + r2) * 16 + piece];
        v2 = reinterpret_cast<const uint4*>(P.host_v)[(src + r2) * 16 + piece];
      }
      if (r < rows) {
        reinterpret_cast<uint4*>(P.cache_k)[(dst + r) * 16 + piece] = k;
        reinterpret_cast<uint4*>(P.cache_v)[(dst + r) * 16 + piece] = v;
      }
      if (r2 < rows) {
        reinterpret_cast<uint4*>(P.cache_k)[(dst + r2) * 16 + piece] = k2;
        reinterpret_cast<uint4*>(P.cache_v)[(dst + r2) * 16 + piece] = v2;
      }
    }
  };
  int item = blockIdx.x - P.BG, step = 0, first = 0;   // the item's number; that of the window's first
  for (int g0 = 0; g0 < P.BG; g0 += 64) {
    const int g = g0 + lane, own = g < P.BG ? P.miss_num[g] : 0;
    const int upto = (int)ri_wave_incl_scan((uint32_t)own), last = first + __builtin_amdgcn_readlane(upto, 63);
    const auto next = [&]() {
      const int in = __popcll(__ballot(upto <= item - first));   // the item's group in the window
      copy(g0 + in, item - first - __builtin_amdgcn_readlane(upto - own, in));
    };
    if (g0 == 0) {
      // How many waves, by the first window's rows, while the first wave's first item is on its way: that is its own in any case.
      int rows = 0;
      if (own > 0) {
        const size_t end = (size_t)g * P.buffer_size + own - 1;
        rows = P.miss_cumsum[end] + P.miss_sizes[end];
      }
      const bool begun = wave == 0 && item < last;
      if (begun) next();
      rows = __builtin_amdgcn_readlane((int)ri_wave_incl_scan((uint32_t)rows), 63);
      const int waves = rows < 4 * last ? min((8 * last + rows - 1) / max(rows, 1), 8) : 1;
      if (wave >= waves) return;
      step = LRU_COPIERS * waves;
      item += begun ? step : LRU_COPIERS * wave;
    }
    for (; item < last; item += step) next();
    first = last;
  }
}

int ri_lru_check(const ri_lru_t& P) {
  // (a cache without blocks has an empty free list: its pointer may be null)
  if (!P.ret_ids || !P.sizes || !P.starts || !P.blk_off || !P.stamp || !P.order || !P.blk_ids ||
      (!P.free_list && P.capacity > 0) || !P.free_count || !P.epoch || !P.hit_ids || !P.hit_sizes || !P.hit_cumsum ||
      !P.hit_num || !P.miss_ids || !P.miss_sizes || !P.miss_cumsum || !P.miss_num || !P.upd_buf || !P.upd_sizes ||
      !P.upd_cache || !P.upd_num)
    return RI_ERR_ARG;
  if (P.BG <= 0 || P.np <= 0 || P.np > 4 * LRU_THREADS || P.ncl <= 0 || P.ncl > 64 * LRU_THREADS || P.buffer_size <= 0 ||
      P.capacity < 0 || P.block <= 0)
    return RI_ERR_ARG;
  if (P.meta_stride < P.ncl || P.blk_off_stride < P.ncl + 1 || P.stamp_stride < P.ncl || P.blk_ids_stride <= 0)
    return RI_ERR_ARG;
  if (P.row_src && (!P.meta || P.row_src_stride < P.buffer_size * P.block || P.stage_row0 < P.capacity * P.block))
    return RI_ERR_ARG;
  return RI_OK;
}

extern "C" int ri_lru_access_update(const int32_t* ret_ids, const int32_t* sizes, const int32_t* starts,
                                    int meta_stride, const int32_t* blk_off, int blk_off_stride, int32_t* stamp,
                                    int32_t* order, int stamp_stride, int32_t* blk_ids, int blk_ids_stride, int32_t* free_list,
                                    int32_t* free_count, int32_t* epoch, int32_t* hit_ids, int32_t* hit_sizes,
                                    int32_t* hit_cumsum, int32_t* hit_num, int32_t* miss_ids, int32_t* miss_sizes,
                                    int32_t* miss_cumsum, int32_t* miss_num, int32_t* upd_buf, int32_t* upd_sizes,
                                    int32_t* upd_cache, int32_t* upd_num, int32_t* row_src, int row_src_stride,
                                    int stage_row0, int32_t* meta, int BG, int np, int ncl, int buffer_size,
                                    int capacity, int block, ri_stream_t stream) {
  const ri_lru_t P = {ret_ids, sizes, starts, blk_off, stamp, order, blk_ids, free_list, free_count, epoch,
                      hit_ids, hit_sizes, hit_cumsum, hit_num, miss_ids, miss_sizes, miss_cumsum, miss_num,
                      upd_buf, upd_sizes, upd_cache, upd_num, row_src, meta, nullptr, nullptr, nullptr, nullptr, 0, 0,
                      row_src_stride, stage_row0, np, ncl, meta_stride, blk_off_stride, stamp_stride, blk_ids_stride,
                      buffer_size, capacity, block, BG};
  const int rc = ri_lru_check(P);
  if (rc) return rc;
  if (np < LRU_THREADS)
    lru_kernel<1, LRU_BOTH><<<BG, LRU_THREADS, 0, (hipStream_t)stream>>>(P);
  else
    lru_kernel<4, LRU_BOTH><<<BG, LRU_THREADS, 0, (hipStream_t)stream>>>(P);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_lru_access(const ri_lru_t* s, ri_stream_t stream) {
  if (!s) return RI_ERR_ARG;
  const int rc = ri_lru_check(*s);
  if (rc) return rc;
  if (s->np < LRU_THREADS)
    lru_kernel<1, LRU_ACCESS><<<s->BG, LRU_THREADS, 0, (hipStream_t)stream>>>(*s);
  else
    lru_kernel<4, LRU_ACCESS><<<s->BG, LRU_THREADS, 0, (hipStream_t)stream>>>(*s);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_lru_stage_update(const ri_lru_t* s, ri_stream_t stream) {
  if (!s) return RI_ERR_ARG;
  const int rc = ri_lru_check(*s);
  if (rc) return rc;
  if (!s->row_src || !s->host_k || !s->host_v || !s->cache_k || !s->cache_v || s->host_stride <= 0 || s->BG > 65535 ||
      s->cache_stride < (int64_t)s->stage_row0 + (int64_t)s->buffer_size * s->block)
    return RI_ERR_ARG;
  if (ri_any_misaligned16(s->host_k, s->host_v, s->cache_k, s->cache_v)) return RI_ERR_ARG;
  const dim3 grid(s->BG + LRU_COPIERS);
  if (s->np < LRU_THREADS) lru_stage_kernel<1><<<grid, LRU_THREADS, 0, (hipStream_t)stream>>>(*s);
  else lru_stage_kernel<4><<<grid, LRU_THREADS, 0, (hipStream_t)stream>>>(*s);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

// Selection and look-up of a host-resident decode step in one launch.  It stands here because a file's kernels are loaded together,
// when the first of them is launched, and a host step launches those above too (a process's first pass, 2 layers 2.9 ms, 3.1 from a
// file of its own).
//
// Both halves are one workgroup per group and a chain of scans and dependent loads, and the second begins with the first one's
// ranks: a thread has its rank's cluster at hand, and a launch and a round trip for the ids are left out.
// What bounds it is the two chains. Selection and look-up apart / together, us: 32 groups of 7 heads, 3840 clusters 8.4 + 6.4 / 13.0.  Steps
// whose misses are few, apart / together: 1 group of 7 heads, 704 clusters 33.8 / 30.8; 6 of 8 in half, 1152 40.7 / 38.3; 64 of 8, 3456 46.4 / 43.2;
// 16 of 1, 1760 69.9 / 68.5.  (Nothing more by requesting the look-up's words in front of the selection's stores, or by barriers that
// do not wait for those.)
template <int NT, int E, int GSM, bool HALF, int SRC>
__global__ __launch_bounds__(NT) void select_access_kernel(ri_ptr4 in, ri_int4 n, int ntiles, SelectArgs A, ri_lru_t L) {
  SelectArgs P = A;
  if (SRC == SEL_LOGITS) {
    P.logits = ri_global<float>(in[0]);
    P.tile_max = ri_global<float>(in[1]);
    P.tile_sum = ri_global<float>(in[2]);
  } else {
    P.cent = ri_global<const uint16_t>(in[0]);
    P.q = ri_global<const uint16_t>(in[1]);
  }
  P.mask = ri_global<const uint8_t>(in[3]);
  P.nc = n[0];
  P.gs = n[1];
  P.np = n[2];
  P.es = n[3];
  P.ntiles = ntiles;
  const int own = select_group<NT, E, GSM, HALF, SRC, KEEP_NONE>(P, blockIdx.x, SelectKept{}, [] {});
  lru_group<1, LRU_ACCESS, NT, LRU_OWN>(L, blockIdx.x, own);
}

template <int NT, int E, int GSM, int SRC>
static void launch_access(const SelectArgs& P, const ri_lru_t& L, int BG, bool half, hipStream_t s) {
  const void* a = SRC == SEL_LOGITS ? (const void*)P.logits : (const void*)P.cent;
  const void* b = SRC == SEL_LOGITS ? (const void*)P.tile_max : (const void*)P.q;
  auto* kernel = half ? select_access_kernel<NT, E, GSM, true, SRC> : select_access_kernel<NT, E, GSM, false, SRC>;
  kernel<<<BG, NT, 0, s>>>(ri_pack_ptrs(a, b, P.tile_sum, P.mask), (ri_int4){P.nc, P.gs, P.np, P.es}, P.ntiles, P, L);
}
template <int NT, int E, int SRC>
static void launch_heads(const SelectArgs& P, const ri_lru_t& L, int BG, bool half, hipStream_t s) {
  if (P.gs <= 4) launch_access<NT, E, 4, SRC>(P, L, BG, half, s);
  else if (P.gs <= 8) launch_access<NT, E, 8, SRC>(P, L, BG, half, s);
  else launch_access<NT, E, 16, SRC>(P, L, BG, half, s);
}

// The selection's forms are those of ri_score_select where it makes the scores' sums itself, up to four clusters to a thread: 4096
// clusters, 2048 with more than eight heads (with up to four heads ri_score_select sums further).  A thread has one rank, and
// one thread at least has none: up to 255, 511 or 1023 probes.  *taken tells the caller of the rest to launch both halves apart.
int ri_launch_select_access(const SelectArgs& P, const ri_lru_t& L, int BG, bool half, bool* taken, hipStream_t s) {
  *taken = false;
  const int nc = P.nc, np = P.np;
  if (L.ret_ids != P.ret_ids || L.np != np || L.BG != BG || P.cluster_size || P.cI) return RI_OK;
  if (nc <= 512) {
    if (np >= (nc <= 256 ? 256 : 512)) return RI_OK;
    if (nc <= 256) launch_heads<256, 1, SEL_SCORE>(P, L, BG, half, s);
    else launch_heads<512, 1, SEL_SCORE>(P, L, BG, half, s);
  } else {
    if (nc > (P.gs <= 8 ? 4096 : 2048) || np >= 1024) return RI_OK;
    const int rc = ri_launch_select_inputs(P, BG, half, false, s);
    if (rc) return rc;
    if (nc <= 1024 && np < 512) launch_heads<512, 2, SEL_LOGITS>(P, L, BG, half, s);
    else if (nc <= 2048 && np < 512) launch_heads<512, 4, SEL_LOGITS>(P, L, BG, half, s);
    else launch_heads<1024, 4, SEL_LOGITS>(P, L, BG, half, s);
  }
  RI_HIP_CHECK_LAUNCH();
  *taken = true;
  return RI_OK;
}
