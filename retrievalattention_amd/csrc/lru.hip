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
#include "ri_common.h"

#define LRU_THREADS 1024
#define LRU_WAVES (LRU_THREADS / 64)
#define LRU_DIGIT 256
#define LRU_COPIES 8        // of the age histogram: a step's clusters share their age
#define LRU_HELD 4          // clusters per thread whose stamps and blocks stay in registers
#define LRU_COPIERS 64      // workgroups that copy missed rows

enum { LRU_BOTH, LRU_ACCESS, LRU_UPDATE };

// exclusive prefix sums of N values over the 1024 threads; totals in tot.  Wave scans on DPP, the sixteen
// wave totals scanned by the lanes of every wave (one LDS read, one DPP scan, two lane reads).
template <int N>
__device__ __forceinline__ void lru_scan(const int (&v)[N], int (&pre)[N], int (&tot)[N], int* sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    inc[k] = (int)ri_wave_incl_scan((uint32_t)v[k]);
    if (lane == 63) sh[k * LRU_WAVES + wave] = inc[k];
  }
  __syncthreads();
  const int wv = __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const uint32_t x = (lane < LRU_WAVES) ? (uint32_t)sh[k * LRU_WAVES + lane] : 0u;
    const uint32_t sc = ri_wave_incl_scan(x);
    tot[k] = __builtin_amdgcn_readlane((int)sc, LRU_WAVES - 1);
    const int woff = wv > 0 ? __builtin_amdgcn_readlane((int)sc, wv - 1) : 0;
    pre[k] = woff + inc[k] - v[k];
  }
  __syncthreads();
}

// R: ranks of the probe list a thread owns (thread t: ranks [t*R, t*R + R)); 1 up to 1023 probes, 4 up to 4096.
// LRU_UPDATE sees the state that LRU_ACCESS left: the hits carry this step's stamp, so every rank finds itself as before.
template <int R, int PHASE>
__device__ __forceinline__ void lru_group(const ri_lru_t& P, int g) {
  constexpr int NPMAX = LRU_THREADS * R;
  constexpr bool ACCESS = PHASE != LRU_UPDATE, UPDATE = PHASE != LRU_ACCESS;
  __shared__ int sh_scan[7 * LRU_WAVES];
  __shared__ __attribute__((aligned(16))) int sh_hist[UPDATE ? LRU_DIGIT * LRU_COPIES : 4];
  __shared__ int sh_cut[2];  // selected digit, blocks freed by clusters with a larger one
  // token offsets and sources of the ranks for the row table; later the blocks of the boundary step's
  // clusters by their order inside the step (2 * NPMAX entries: hits below, admitted misses above)
  __shared__ int sh_tab[2 * NPMAX];
  int* const sh_off = sh_tab;
  int* const sh_src = sh_tab + NPMAX;
  const int tid = threadIdx.x;
  const int block = P.block;
  const int32_t* sizes = P.sizes + (size_t)g * P.meta_stride;
  const int32_t* starts = P.starts + (size_t)g * P.meta_stride;
  const int32_t* boff = P.blk_off + (size_t)g * P.blk_off_stride;
  int32_t* stamp = P.stamp + (size_t)g * P.stamp_stride;
  int32_t* order = P.order + (size_t)g * P.stamp_stride;
  int32_t* bids = P.blk_ids + (size_t)g * P.blk_ids_stride;
  int32_t* flist = P.free_list + (size_t)g * P.capacity;
  const size_t lo = (size_t)g * P.buffer_size;
  const int E = P.epoch[g] + 1;
  const int F0 = P.free_count[g];
  const int rb = tid * R;
  if (PHASE == LRU_UPDATE && P.miss_num[g] == 0) {   // (uniform) nothing to admit
    if (tid == 0) {
      P.upd_num[g] = 0;
      P.epoch[g] = E;
    }
    return;
  }
  // thread t owns the ids [t*K, t*K + K) for the eviction; up to LRU_HELD of them stay in registers
  const int K = (P.ncl + LRU_THREADS - 1) / LRU_THREADS;
  const bool held = K <= LRU_HELD;   // uniform
  const int c0 = tid * K, c1 = min(P.ncl, c0 + K);
  int h_stamp[LRU_HELD], h_nb[LRU_HELD];
  auto hold = [&]() {
#pragma unroll
    for (int i = 0; i < LRU_HELD; ++i) {
      const int cc = min(c0 + i, P.ncl - 1);
      h_stamp[i] = stamp[cc];
      h_nb[i] = boff[cc + 1] - boff[cc];
    }
#pragma unroll
    for (int i = 0; i < LRU_HELD; ++i)
      if (c0 + i >= c1) h_stamp[i] = 0;
  };
  if (PHASE == LRU_UPDATE && held) hold();   // (in flight under the ranks' own loads)

  // ---- access: every rank looks at its cluster ----
  // (everything the rank needs to know about its cluster is requested in one go: loads issued after a
  // barrier would each put another round trip to global memory on the kernel's critical path)
  int c[R], nb[R], sz[R], stamp_c[R], boff_c[R], start_c[R];
  int nb_sum = 0;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    c[i] = -1; nb[i] = 0; sz[i] = 0; stamp_c[i] = 0; boff_c[i] = 0; start_c[i] = 0;
    if (rb + i < P.np) {
      c[i] = P.ret_ids[(size_t)g * P.np + rb + i];
      if (c[i] < 0 || c[i] >= P.ncl) {
        c[i] = -1;
      } else {
        sz[i] = sizes[c[i]];
        stamp_c[i] = stamp[c[i]];
        boff_c[i] = boff[c[i]];
        start_c[i] = starts[c[i]];
        nb[i] = (sz[i] + block - 1) / block;
      }
    }
    nb_sum += nb[i];
  }
  // The walk stops at the first cluster whose blocks no longer fit: everything after it is dropped.  Whether
  // anything is dropped is only known from the block prefix, so the counts are first taken as if nothing were
  // (one scan for the block prefix and the counts together) and only recounted when the list was cut.
  bool keep[R], hit[R], miss[R];
  int v5[6], p5[6], t5[6];
  auto count = [&](int run) {
#pragma unroll
    for (int k = 0; k < 6; ++k) v5[k] = 0;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      keep[i] = c[i] >= 0 && nb[i] > 0 && run + nb[i] <= P.buffer_size;
      hit[i] = keep[i] && stamp_c[i] != 0;
      miss[i] = keep[i] && !hit[i];
      run += nb[i];
      v5[0] += hit[i] ? nb[i] : 0;
      v5[1] += keep[i] ? sz[i] : 0;
      v5[2] += miss[i] ? nb[i] : 0;
      v5[3] += miss[i] ? sz[i] : 0;
      v5[4] += keep[i] ? 1 : 0;
      v5[5] += hit[i] ? 1 : 0;
    }
  };
  {
    count(INT32_MIN / 2);   // no cut-off: every valid cluster with blocks is kept
    int v7[7], p7[7], t7[7];
#pragma unroll
    for (int k = 0; k < 6; ++k) v7[k] = v5[k];
    v7[6] = nb_sum;
    lru_scan<7>(v7, p7, t7, sh_scan);
    if (t7[6] <= P.buffer_size) {   // uniform: the whole list fits
#pragma unroll
      for (int k = 0; k < 6; ++k) { p5[k] = p7[k]; t5[k] = t7[k]; }
    } else {
      count(p7[6]);
      lru_scan<6>(v5, p5, t5, sh_scan);
    }
  }
  // per rank: hit blocks, kept tokens, miss blocks, miss tokens, hits of the lower ranks
  int hb_pre[R], tok_pre[R], mb_pre[R], mt_pre[R], hit_idx[R];
  {
    int a = p5[0], b = p5[1], cc = p5[2], d = p5[3], h = p5[5];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      hb_pre[i] = a; tok_pre[i] = b; mb_pre[i] = cc; mt_pre[i] = d; hit_idx[i] = h;
      a += hit[i] ? nb[i] : 0;
      b += keep[i] ? sz[i] : 0;
      cc += miss[i] ? nb[i] : 0;
      d += miss[i] ? sz[i] : 0;
      h += hit[i] ? 1 : 0;
    }
  }
  const int nhits = t5[5];
  // tok_pre: tokens of kept clusters of lower rank (position in the row table); the hit list's own
  // token offsets are only needed without a row table
  int hit_tok[R];
#pragma unroll
  for (int i = 0; i < R; ++i) hit_tok[i] = 0;
  if (ACCESS && !P.row_src) {
    int vh[1] = {0}, ph[1], th[1];
#pragma unroll
    for (int i = 0; i < R; ++i) vh[0] += hit[i] ? sz[i] : 0;
    lru_scan<1>(vh, ph, th, sh_scan);
    int a = ph[0];
#pragma unroll
    for (int i = 0; i < R; ++i) { hit_tok[i] = a; a += hit[i] ? sz[i] : 0; }
  }
  // the longest prefix of the misses whose blocks fit the whole cache may be admitted (none when the cache
  // has no blocks: every retrieved cluster then stays a miss, wave_buffer_cpu.cpp:119-130 with capacity 0)
  // (a step whose clusters all hit — the steady state of a warm cache — admits nothing and skips the scans)
  const bool any_miss = t5[2] > 0;  // uniform
  bool adm[R];
  int adm_pre[R];
  int need = 0;
#pragma unroll
  for (int i = 0; i < R; ++i) { adm[i] = false; adm_pre[i] = 0; }
  if (any_miss) {
    int va[1] = {0}, pa[1], ta[1];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      adm[i] = miss[i] && mb_pre[i] + nb[i] <= P.capacity;
      va[0] += adm[i] ? nb[i] : 0;
    }
    lru_scan<1>(va, pa, ta, sh_scan);
    need = ta[0];
    int a = pa[0];
#pragma unroll
    for (int i = 0; i < R; ++i) { adm_pre[i] = a; a += adm[i] ? nb[i] : 0; }
  }

  if (ACCESS) {
    const bool rows = P.row_src != nullptr;
    if (rows) {
      // row table: every thread takes tokens t, t + 1024, ... and finds the rank that owns them by
      // bisection over the token offsets of the ranks (clusters that were dropped have no tokens)
#pragma unroll
      for (int i = 0; i < R; ++i) {
        sh_off[rb + i] = tok_pre[i];
        sh_src[rb + i] = hit[i] ? -(boff_c[i] + 1) : P.stage_row0 + mt_pre[i];  // hits: where their block ids are
      }
      __syncthreads();
      int32_t* table = P.row_src + (size_t)g * P.row_src_stride;
      for (int t = tid; t < t5[1]; t += LRU_THREADS) {
        int lo_r = 0, hi_r = min(NPMAX, P.np);  // first rank whose offset exceeds t (ranks past the list hold the total)
        while (lo_r < hi_r) {
          const int mid = (lo_r + hi_r) >> 1;
          if (sh_off[mid] > t) hi_r = mid; else lo_r = mid + 1;
        }
        const int r = lo_r - 1, i = t - sh_off[r], src = sh_src[r];
        table[t] = src < 0 ? bids[-src - 1 + i / block] * block + i % block : src + i;
      }
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (hit[i]) {
        const int32_t* ids = bids + boff_c[i];
        if (!rows) {
          for (int j = 0; j < nb[i]; ++j) {
            P.hit_ids[lo + hb_pre[i] + j] = ids[j];
            P.hit_sizes[lo + hb_pre[i] + j] = (j == nb[i] - 1) ? sz[i] - (nb[i] - 1) * block : block;
            P.hit_cumsum[lo + hb_pre[i] + j] = hit_tok[i] + j * block;
          }
        }
        stamp[c[i]] = E;
        order[c[i]] = nhits - 1 - hit_idx[i];   // hits are moved to the front in reverse rank order
      }
      if (miss[i]) {
        const int row = start_c[i];
        for (int j = 0; j < nb[i]; ++j) {
          P.miss_ids[lo + mb_pre[i] + j] = row + j * block;
          P.miss_sizes[lo + mb_pre[i] + j] = (j == nb[i] - 1) ? sz[i] - (nb[i] - 1) * block : block;
          P.miss_cumsum[lo + mb_pre[i] + j] = mt_pre[i] + j * block;
        }
      }
    }
    if (tid == 0) {
      P.hit_num[g] = rows ? 0 : t5[0];
      P.miss_num[g] = t5[2];
      if (P.meta) {
        P.meta[g * 4 + 0] = t5[4];
        P.meta[g * 4 + 1] = t5[1];
        P.meta[g * 4 + 2] = t5[0] + t5[2];
        P.meta[g * 4 + 3] = 0;
      }
    }
  }
  if (!UPDATE) return;
  if (PHASE == LRU_BOTH) __syncthreads();  // the hits carry this step's stamp and order before anybody looks for victims

  // ---- eviction: free (need - F0) blocks from the least recently used clusters ----
  const int to_free = need - F0;  // uniform
  int F = F0;
  if (to_free > 0) {
    if (PHASE == LRU_BOTH && held) hold();
    // fn(cluster, stamp, blocks) for every resident cluster of this thread, in id order
    auto resident = [&](auto&& fn) {
      if (held) {
#pragma unroll
        for (int i = 0; i < LRU_HELD; ++i)
          if (h_stamp[i] != 0) fn(c0 + i, h_stamp[i], h_nb[i]);
      } else {
        for (int cc = c0; cc < c1; ++cc) {
          const int st = stamp[cc];
          if (st != 0) fn(cc, st, boff[cc + 1] - boff[cc]);
        }
      }
    };
    // boundary step: the age A such that every resident cluster older than A goes and the clusters of age A
    // cover the remaining `rem` blocks; radix selection over the bytes of the age, oldest first.  No age has a byte
    // above the step number's: the first 255 steps take one round.
    uint32_t sel_mask = 0, sel_val = 0;
    int rem = to_free;
    for (int b = (31 - __clz(E)) >> 3; b >= 0; --b) {
#pragma unroll
      for (int i = 0; i < LRU_DIGIT * LRU_COPIES / LRU_THREADS; ++i) sh_hist[i * LRU_THREADS + tid] = 0;
      if (tid == 0) { sh_cut[0] = 0; sh_cut[1] = 0; }
      __syncthreads();
      resident([&](int, int st, int nbc) {
        const uint32_t age = (uint32_t)(E - st);
        if ((age & sel_mask) == sel_val)
          atomicAdd(&sh_hist[((age >> (8 * b)) & 255u) * LRU_COPIES + (tid & (LRU_COPIES - 1))], nbc);
      });
      __syncthreads();
      if (tid < 64) {
        // lane l holds the digits 255 - 4l .. 252 - 4l (oldest first); the lane whose running total crosses
        // rem holds the boundary digit
        int h[4], sum = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int4* hp = reinterpret_cast<const int4*>(sh_hist + (255 - (4 * tid + i)) * LRU_COPIES);
          const int4 x = hp[0], y = hp[1];
          h[i] = x.x + x.y + x.z + x.w + y.x + y.y + y.z + y.w;
          sum += h[i];
        }
        const int incl = (int)ri_wave_incl_scan((uint32_t)sum);
        int acc = incl - sum;
        if (acc < rem && rem <= incl) {
          int sel = 0;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (acc < rem && rem <= acc + h[i]) { sel = 255 - (4 * tid + i); sh_cut[1] = acc; }
            acc += h[i];
          }
          sh_cut[0] = sel;
        }
      }
      __syncthreads();
      sel_val |= (uint32_t)sh_cut[0] << (8 * b);
      sel_mask |= 255u << (8 * b);
      rem -= sh_cut[1];
      __syncthreads();
    }
    const uint32_t cut = sel_val;   // boundary age; rem blocks are still wanted from the clusters of that age
    // the clusters of the boundary step, least recent first = ascending order inside the step
    for (int i = tid; i < 2 * NPMAX; i += LRU_THREADS) sh_tab[i] = 0;
    __syncthreads();
    resident([&](int cc, int st, int nbc) {
      if ((uint32_t)(E - st) == cut) sh_tab[min(max(order[cc], 0), 2 * NPMAX - 1)] = nbc;
    });
    __syncthreads();
    {
      // exclusive prefix of the table in place: thread t owns the entries [t * 2R, t * 2R + 2R)
      int own[2 * R], vt[1] = {0}, pt[1], tt[1];
#pragma unroll
      for (int i = 0; i < 2 * R; ++i) { own[i] = sh_tab[tid * 2 * R + i]; vt[0] += own[i]; }
      lru_scan<1>(vt, pt, tt, sh_scan);
      int run = pt[0];
#pragma unroll
      for (int i = 0; i < 2 * R; ++i) { sh_tab[tid * 2 * R + i] = run; run += own[i]; }
    }
    __syncthreads();
    int ev = 0;
    uint64_t ev_bits = 0;  // K <= 64 ids per thread
    resident([&](int cc, int st, int nbc) {
      const uint32_t age = (uint32_t)(E - st);
      const bool out = age > cut || (age == cut && sh_tab[min(max(order[cc], 0), 2 * NPMAX - 1)] < rem);
      if (out) {
        ev_bits |= 1ull << (cc - c0);
        ev += nbc;
      }
    });
    int ve[1] = {ev}, pe[1], te[1];
    lru_scan<1>(ve, pe, te, sh_scan);
    int w = F0 + pe[0];
    for (int cc = c0; cc < c1; ++cc) {
      if (!((ev_bits >> (cc - c0)) & 1ull)) continue;
      const int nbc = boff[cc + 1] - boff[cc];
      for (int j = 0; j < nbc; ++j) flist[w++] = bids[boff[cc] + j];
      stamp[cc] = 0;
    }
    F = F0 + te[0];
    __syncthreads();  // the freed ids are in the list before they are handed out
  }

  // ---- admission: block ids come off the end of the free list in rank order ----
  int vb[2] = {0, 0}, pb[2] = {0, 0}, tb[2] = {0, 0};
#pragma unroll
  for (int i = 0; i < R; ++i) {
    adm[i] = adm[i] && adm_pre[i] + nb[i] <= F;  // (always true: everything resident can be evicted)
    vb[0] += adm[i] ? nb[i] : 0;
    vb[1] += adm[i] ? 1 : 0;
  }
  if (any_miss) lru_scan<2>(vb, pb, tb, sh_scan);
  int adm_idx = pb[1];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (adm[i]) {
      order[c[i]] = nhits + adm_idx++;   // pushed to the front in rank order, after the hits
      int32_t* ids = bids + boff_c[i];
      for (int j = 0; j < nb[i]; ++j) {
        const int id = flist[F - 1 - (adm_pre[i] + j)];
        ids[j] = id;
        P.upd_cache[lo + adm_pre[i] + j] = id;
        P.upd_sizes[lo + adm_pre[i] + j] = (j == nb[i] - 1) ? sz[i] - (nb[i] - 1) * block : block;
        P.upd_buf[lo + adm_pre[i] + j] = mt_pre[i] + j * block;  // admitted misses lead the miss list
      }
      stamp[c[i]] = E;
    }
  }
  if (tid == 0) {
    P.upd_num[g] = tb[0];
    P.free_count[g] = F - tb[0];
    P.epoch[g] = E;
  }
}

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

static int lru_check(const ri_lru_t& P) {
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
  const int rc = lru_check(P);
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
  const int rc = lru_check(*s);
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
  const int rc = lru_check(*s);
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
