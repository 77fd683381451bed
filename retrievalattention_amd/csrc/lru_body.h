// The group's half of the device-side block cache manager (see lru.hip), also behind a selection.
#pragma once
#include "ri_common.h"

#define LRU_THREADS 1024
#define LRU_DIGIT 256
#define LRU_COPIES 8        // of the age histogram: a step's clusters share their age
#define LRU_HELD 4          // clusters per thread whose stamps and blocks stay in registers

enum { LRU_BOTH, LRU_ACCESS, LRU_UPDATE };

// exclusive prefix sums of N values over the NT threads; totals in tot.  Wave scans on DPP, the (at most sixteen)
// wave totals scanned by the lanes of every wave (one LDS read, one DPP scan, two lane reads).
template <int NT, int N>
__device__ __forceinline__ void lru_scan(const int (&v)[N], int (&pre)[N], int (&tot)[N], int* sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    inc[k] = (int)ri_wave_incl_scan((uint32_t)v[k]);
    if (lane == 63) sh[k * (NT / 64) + wave] = inc[k];
  }
  __syncthreads();
  const int wv = __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const uint32_t x = (lane < (NT / 64)) ? (uint32_t)sh[k * (NT / 64) + lane] : 0u;
    const uint32_t sc = ri_wave_incl_scan(x);
    tot[k] = __builtin_amdgcn_readlane((int)sc, (NT / 64) - 1);
    const int woff = wv > 0 ? __builtin_amdgcn_readlane((int)sc, wv - 1) : 0;
    pre[k] = woff + inc[k] - v[k];
  }
  __syncthreads();
}

// R: ranks of the probe list a thread owns (thread t: ranks [t*R, t*R + R)); 1 up to NT - 1 probes, 4 up to 4096.  own: with
// R = 1 the cluster of the thread's rank (-1: none), where the caller has it.
// LRU_UPDATE sees the state that LRU_ACCESS left: the hits carry this step's stamp, so every rank finds itself as before.
enum { LRU_LISTED, LRU_OWN };   // IDS: who knows the ranks' clusters
template <int R, int PHASE, int NT = LRU_THREADS, int IDS = LRU_LISTED>
__device__ __forceinline__ void lru_group(const ri_lru_t& P, int g, int own = -1) {
  static_assert(IDS == LRU_LISTED || R == 1, "an id per thread");
  static_assert(PHASE == LRU_ACCESS || NT == LRU_THREADS, "the update's histogram is dealt to 1024 threads");
  constexpr int NPMAX = NT * R;
  constexpr bool ACCESS = PHASE != LRU_UPDATE, UPDATE = PHASE != LRU_ACCESS;
  __shared__ int sh_scan[7 * (NT / 64)];
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
  const int K = (P.ncl + NT - 1) / NT;
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
      c[i] = IDS == LRU_OWN ? own : P.ret_ids[(size_t)g * P.np + rb + i];
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
    lru_scan<NT, 7>(v7, p7, t7, sh_scan);
    if (t7[6] <= P.buffer_size) {   // uniform: the whole list fits
#pragma unroll
      for (int k = 0; k < 6; ++k) { p5[k] = p7[k]; t5[k] = t7[k]; }
    } else {
      count(p7[6]);
      lru_scan<NT, 6>(v5, p5, t5, sh_scan);
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
    lru_scan<NT, 1>(vh, ph, th, sh_scan);
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
    lru_scan<NT, 1>(va, pa, ta, sh_scan);
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
      for (int t = tid; t < t5[1]; t += NT) {
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
      for (int i = 0; i < LRU_DIGIT * LRU_COPIES / NT; ++i) sh_hist[i * NT + tid] = 0;
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
    for (int i = tid; i < 2 * NPMAX; i += NT) sh_tab[i] = 0;
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
      lru_scan<NT, 1>(vt, pt, tt, sh_scan);
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
    lru_scan<NT, 1>(ve, pe, te, sh_scan);
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
  if (any_miss) lru_scan<NT, 2>(vb, pb, tb, sh_scan);
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

// Whether a manager's arguments are in order (lru.hip): RI_OK or RI_ERR_ARG.
int ri_lru_check(const ri_lru_t& P);
