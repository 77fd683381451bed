// Cluster selection for the decode step (gfx950): from the fp32 logits of the scoring pass to
// the retrieval zone (top nprobe clusters in rank order), the estimation zone (next es) and
// the layout of the retrieved tokens (rank tables, optionally a row table).  Follows cache_hub/retroinfer_cache.py:572-575
// (sum over the query group of the bf16 softmax, empty-cluster mask, top-k) and the buffer
// cut-off of library/retroinfer/retroinfer_kernels/src/wave_buffer_cpu.cpp:207-216.
//
// Up to three launches:
//   score_kernel   (score.hip) the logits and per-tile softmax statistics, unless the selection scores for itself;
//   dist_kernel    many workgroups per group: score = bf16(sum_j bf16(exp(bf16(x_j)-m_j)/Z_j)),
//                  mapped to a 16-bit key whose unsigned order is the score order, unless the selection does it itself;
//   a selection    one workgroup per group: exact rank thresholds from histograms of the keys, zone
//                  membership with ties resolved by ascending id, rank order of the retrieval
//                  zone, and the token layout (page cut-off; token prefix and first store row per rank, a row per
//                  token on request).  select_radix_kernel serves up to 1024 probes of up to 16384 clusters,
//                  select_kernel the longer lists.
#include <type_traits>

#include "ri_common.h"

#define SEL_THREADS 1024
#define SEL_MAX_PROBES 4096  // ranks of the retrieval zone one workgroup can lay out (four per thread)
#define SEL_WAVES (SEL_THREADS / 64)
#define DIST_IDS 1024  // ids per dist workgroup (4 per thread)

// Histogram add that survives a degenerate distribution: when the whole wave hits one bin
// (for instance every score equal) a single lane adds the lane count.
__device__ __forceinline__ void hist_add(uint32_t* hist, uint32_t bin, bool active) {
  const uint64_t act = __ballot(active);
  if (act == 0) return;
  const int lead = __ffsll((long long)act) - 1;
  const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)bin, lead);
  const uint64_t same = __ballot(active && bin == first);
  if (same == act) {
    if ((int)(threadIdx.x & 63) == lead) atomicAdd(&hist[first], (uint32_t)__popcll(act));
  } else if (active) {
    atomicAdd(&hist[bin], 1u);
  }
}

// ------------------------------------------------------------------------------------
// dist_kernel: grid (ceil(nc / 1024), BG), 256 threads, 4 consecutive ids per thread.
// ------------------------------------------------------------------------------------
// HALF: scores are rounded to IEEE half instead of bfloat16 wherever the reference's tensors are (the D and
// Softmax outputs of batch_gemm_softmax and the score sum carry the cache's element type).
template <int GSM, bool HALF>
__global__ __launch_bounds__(256) void dist_kernel(const float* __restrict__ logits,
                                                   const float* __restrict__ tile_max,
                                                   const float* __restrict__ tile_sum,
                                                   const uint8_t* __restrict__ mask, uint16_t* __restrict__ keys,
                                                   uint16_t* __restrict__ dist_out, int gs, int nc, int ntiles) {
  __shared__ float sh_m[16], sh_iz[16];
  const int g = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = blockIdx.x * DIST_IDS + tid * 4;
  const bool in = c < nc;  // nc % 4 == 0

  // loads first, so that the row statistics below hide behind their latency; heads past gs and ids past nc read a valid
  // place instead (a load under a condition became a branch that also waited for it: one round trip per head)
  const int cc = min(c, nc - 4);
  float4 x4[GSM];
#pragma unroll
  for (int j = 0; j < GSM; ++j)
    x4[j] = *reinterpret_cast<const float4*>(logits + ((size_t)g * gs + min(j, gs - 1)) * nc + cc);
  const uint32_t mk = mask ? *reinterpret_cast<const uint32_t*>(mask + (size_t)g * nc + cc) : 0u;

  for (int j = wave; j < gs; j += 4) {
    float m, iz;
    ri_wave_reduce_partials(tile_max + (size_t)g * ntiles * gs, tile_sum + (size_t)g * ntiles * gs, ntiles, gs, j,
                            lane, &m, &iz);
    if (lane == 0) { sh_m[j] = m; sh_iz[j] = iz; }
  }
  __syncthreads();

  float d[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < GSM; ++j) {
    const float x[4] = {x4[j].x, x4[j].y, x4[j].z, x4[j].w};
    const float m = sh_m[j], iz = sh_iz[j];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p = ri_round_e16<HALF>(__expf(ri_round_e16<HALF>(x[i]) - m) * iz);
      d[i] += j < gs ? p : 0.f;
    }
  }
  uint16_t bits[4], key[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    bits[i] = ri_f32_to_e16<HALF>(d[i]);
    if ((mk >> (8 * i)) & 0xffu) bits[i] = ri_e16_lowest<HALF>();  // finfo(type).min
    key[i] = (uint16_t)ri_bf16_sort_key(bits[i]);
  }
  if (in) {
    uint2 w;
    w.x = (uint32_t)key[0] | ((uint32_t)key[1] << 16);
    w.y = (uint32_t)key[2] | ((uint32_t)key[3] << 16);
    *reinterpret_cast<uint2*>(keys + (size_t)g * nc + c) = w;
    if (dist_out) {
      w.x = (uint32_t)bits[0] | ((uint32_t)bits[1] << 16);
      w.y = (uint32_t)bits[2] | ((uint32_t)bits[3] << 16);
      *reinterpret_cast<uint2*>(dist_out + (size_t)g * nc + c) = w;
    }
  }
}

// ------------------------------------------------------------------------------------
// select_kernel helpers
// ------------------------------------------------------------------------------------
// Exclusive prefix sums of N values over the threads of the block with one barrier.
// sh: N * SEL_WAVES words that no other scan of the same parity is still reading: callers
// alternate between two buffers.  tot[] receives the block totals.
template <int N>
__device__ __forceinline__ void block_excl_scan(const uint32_t (&v)[N], uint32_t (&pre)[N], uint32_t (&tot)[N],
                                                uint32_t* sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t inc[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    inc[k] = ri_wave_incl_scan(v[k]);
    if (lane == 63) sh[k * SEL_WAVES + wave] = inc[k];
  }
  __syncthreads();
  // the sixteen wave totals are scanned by the lanes (one LDS read, one DPP scan, two lane reads) instead of
  // being walked by every thread: a third of the kernel's vector instructions were that walk, and the kernel
  // is bound by instruction issue on its one compute unit as much as by latency
  const int wv = __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const uint32_t x = (lane < SEL_WAVES) ? sh[k * SEL_WAVES + lane] : 0u;
    const uint32_t sc = ri_wave_incl_scan(x);
    tot[k] = (uint32_t)__builtin_amdgcn_readlane((int)sc, SEL_WAVES - 1);
    const uint32_t woff = wv > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)sc, wv - 1) : 0u;
    pre[k] = woff + inc[k] - v[k];
  }
}

// Scores are sums of at most 16 probabilities, so their keys span a small range: key 0x8000
// (score +0) .. 0xC180 (score 16), plus the masked value far below.  One histogram bin per
// distinct key makes the rank search exact in a single pass.
// (IEEE half: 0x8000 .. 0xCC00, so 17 bins per thread cover bfloat16 scores and 20 cover half scores.)
#define SEL_KEY_LO 0x8000u
#define SEL_BPT_BF16 17                     // bins per thread: 17 * 1024 = 17408 >= 0x4181 + 1
#define SEL_BPT_F16 20                      //                  20 * 1024 = 20480 >= 0x4C01 + 1
template <int BPT>
__device__ __forceinline__ uint32_t sel_bin(uint32_t key) {
  constexpr uint32_t BINS = SEL_THREADS * BPT;
  const uint32_t b = key >= SEL_KEY_LO ? key - SEL_KEY_LO + 1u : 0u;
  return b < BINS ? b : BINS - 1;
}

// ------------------------------------------------------------------------------------
// select_kernel: one 1024-thread workgroup per group, for more than 1024 probes or more than 16384 clusters; one histogram
// bin per distinct key (scores lie in [0, 16], so ~16.8k bins cover every key), rank order from the histogram prefix.
// The sizes of the retrieved clusters are read from global memory by the threads that own a rank (staging
// all nc sizes in LDS up front put 4 nc bytes per group on the load phase of the one compute unit that runs
// the group: 0.9 us slower per step at 8192 clusters, 2.2 us at 16384).
// Thread t owns the contiguous id range [t*E, t*E+E) and keeps those keys in registers: ties
// are ranked by ascending id with plain prefix sums.
// ------------------------------------------------------------------------------------
// E8: eights of keys a thread owns (2 up to 16384 clusters, 4 up to 32768, 8 up to 65536): the
// loops over the owned keys are unrolled E8 times, so the common sizes do not carry (and fetch) the code of
// sixty-four keys per thread.
// R: ranks of the retrieval zone a thread owns in the token-layout phase (1 up to 1023 probes, 4 up to 4096).
// BPT: histogram bins per thread (SEL_BPT_BF16 or SEL_BPT_F16).
template <int E8, int R, int BPT>
__global__ __launch_bounds__(SEL_THREADS) void select_kernel(
    const uint16_t* __restrict__ keys, const int32_t* __restrict__ cluster_size,
    const int32_t* __restrict__ cluster_start, int64_t* __restrict__ cI, int32_t* __restrict__ ret_ids,
    int32_t* __restrict__ est_ids, int32_t* __restrict__ ret_tok_off, int32_t* __restrict__ ret_start,
    int32_t* __restrict__ row_src, int row_src_stride, int32_t* __restrict__ meta, int nc, int np, int es, int page, int max_pages) {
  constexpr int SEL_BPT = BPT;
  constexpr int SEL_BINS = SEL_THREADS * BPT;
  __shared__ uint32_t hist[SEL_BINS];
  __shared__ uint32_t sh_scan[2][3 * SEL_WAVES];  // two buffers, used alternately
  __shared__ uint32_t sh_sel[4];  // bin of T1, entries above it, bin of T2, entries above it
  constexpr int NPMAX = SEL_THREADS * R;
  __shared__ uint32_t sh_ret[NPMAX];
  // rank-ordered entries, then size and first store row of the cluster at each rank: arrays of their own for
  // the common case, laid over the histogram (which is dead by then) when a thread owns several ranks
  __shared__ uint32_t sh_lay[R == 1 ? 3 * NPMAX : 1];
  static_assert(R == 1 || 3 * NPMAX <= SEL_BINS, "the rank arrays must fit the histogram they are laid over");
  uint32_t* const sh_sorted = R == 1 ? sh_lay : hist;
  uint32_t* const sh_size = sh_sorted + NPMAX;
  int32_t* const sh_start = reinterpret_cast<int32_t*>(sh_sorted + 2 * NPMAX);
  __shared__ uint32_t sh_pages, sh_tret, sh_nkeep;

  const int g = blockIdx.x;
  const int tid = threadIdx.x;
  const int k2 = np + es;

  // ---- loads: this thread's keys (registers) ----
  // thread t owns the contiguous id range [t*E, t*E+E), E a multiple of 8 (nc % 8 == 0), E <= 64
  const int E = 8 * E8;  // >= ceil(nc / SEL_THREADS), a multiple of 8
  const int cbeg = min(tid * E, nc);
  const int cend = min(cbeg + E, nc);
  uint4 kreg[E8];
#pragma unroll
  for (int i = 0; i < E8; ++i)
    kreg[i] = (cbeg + 8 * i < cend) ? *reinterpret_cast<const uint4*>(keys + (size_t)g * nc + cbeg + 8 * i)
                                     : ri_zero16();
#pragma unroll
  for (int i = 0; i < SEL_BPT; ++i) hist[tid * SEL_BPT + i] = 0u;
  if (tid == 0) { sh_pages = 0; sh_tret = 0; sh_nkeep = 0; }
  __syncthreads();
  // calls f(id, key) for every owned key in ascending id order
  auto for_each_key = [&](auto&& f) {
#pragma unroll
    for (int i = 0; i < E8; ++i) {
      if (cbeg + 8 * i < cend) {
        const uint32_t w[4] = {kreg[i].x, kreg[i].y, kreg[i].z, kreg[i].w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f(cbeg + 8 * i + 2 * q, w[q] & 0xffffu);
          f(cbeg + 8 * i + 2 * q + 1, w[q] >> 16);
        }
      }
    }
  };
  for_each_key([&](int, uint32_t key) { hist_add(hist, sel_bin<BPT>(key), true); });
  __syncthreads();

  // ---- rank thresholds: T1 = key of descending rank np-1, T2 = key of rank k2-1 ----
  // thread t owns bins [t*17, t*17+17); afterwards hist[b] holds the number of keys above bin b
  {
    uint32_t hb[SEL_BPT], mine = 0;
#pragma unroll
    for (int i = 0; i < SEL_BPT; ++i) { hb[i] = hist[tid * SEL_BPT + i]; mine += hb[i]; }
    uint32_t vin[1] = {mine}, below[1], tot[1];
    block_excl_scan<1>(vin, below, tot, sh_scan[0]);
    uint32_t above = tot[0] - below[0] - mine;  // entries in bins above this thread's
    const uint32_t rankA = (uint32_t)(np - 1), rankB = (uint32_t)(k2 - 1);
    // only threads that hold keys of the retrieval zone (their bins' ranks are needed below) or one of
    // the two threshold ranks walk their bins
    if (mine > 0 && (above < (uint32_t)np || (above <= rankB && rankB < above + mine))) {
#pragma unroll
      for (int i = SEL_BPT - 1; i >= 0; --i) {
        if (above <= rankA && rankA < above + hb[i]) { sh_sel[0] = tid * SEL_BPT + i; sh_sel[1] = above; }
        if (above <= rankB && rankB < above + hb[i]) { sh_sel[2] = tid * SEL_BPT + i; sh_sel[3] = above; }
        hist[tid * SEL_BPT + i] = above;
        above += hb[i];
      }
    }
  }
  __syncthreads();
  const uint32_t B1 = sh_sel[0], B2 = sh_sel[2];  // threshold bins (bins order like keys)
  const uint32_t g1 = sh_sel[1], g2 = sh_sel[3];  // keys strictly above T1 / T2

  // ---- one scan ranks everything: ties at T1, ties at T2 and the keys strictly between ----
  // Tied keys are taken in ascending id order: tie rank r at T1 belongs to the retrieval zone
  // while g1 + r < np, then to the estimation zone while g1 + r < k2; at T2 while g2 + r < k2.
  // The owned keys are classified once, without branches, into four bit masks (bit i = owned key i); the
  // rare cases (keys of the retrieval zone: np of nc; ties at a threshold) are then walked bit by bit.
  typedef typename std::conditional<(E8 <= 4), uint32_t, uint64_t>::type mask_t;
  mask_t m_gt1 = 0, m_eq1 = 0, m_gt2 = 0, m_eq2 = 0;
  for_each_key([&](int c, uint32_t key) {
    const uint32_t bin = sel_bin<BPT>(key);
    const int i = c - cbeg;
    m_gt1 |= (mask_t)(bin > B1) << i;
    m_eq1 |= (mask_t)(bin == B1) << i;
    m_gt2 |= (mask_t)(bin > B2) << i;
    m_eq2 |= (mask_t)(bin == B2) << i;
  });
  if (B2 == B1) m_eq2 = 0;
  const mask_t m_mid = m_gt2 & ~m_gt1 & ~m_eq1;  // strictly between the thresholds: estimation zone
  auto popc = [](mask_t m) { return (uint32_t)(sizeof(mask_t) == 8 ? __popcll((unsigned long long)m) : __popc((unsigned)m)); };
  auto lowest = [](mask_t m) { return sizeof(mask_t) == 8 ? __ffsll((long long)m) - 1 : __ffs((int)m) - 1; };
  uint32_t cnt3[3] = {popc(m_eq1), popc(m_eq2), popc(m_mid)}, pre3[3], tot3[3];
  block_excl_scan<3>(cnt3, pre3, tot3, sh_scan[1]);
  const uint32_t r1 = pre3[0], r2 = pre3[1];
  const uint32_t mid_before = pre3[2];
  const uint32_t lo1 = (uint32_t)np > g1 ? (uint32_t)np - g1 : 0u;   // first tie rank of T1 in the est zone
  const uint32_t hi1r = (uint32_t)k2 > g1 ? (uint32_t)k2 - g1 : 0u;  // one past the last
  const uint32_t hi2r = (uint32_t)k2 > g2 ? (uint32_t)k2 - g2 : 0u;
  // Global stores are kept for the end of the kernel: a barrier waits for every outstanding
  // memory operation of the wave, stores included, so a store issued here would put its round
  // trip on the critical path of each later phase.
  const uint32_t est_first = mid_before + (min(max(r1, lo1), hi1r) - lo1) + min(r2, hi2r);
  // owned key i (a register half chosen at run time: only the rare walks below need it)
  auto key_at = [&](int i) {
    uint32_t w = 0;
#pragma unroll
    for (int v = 0; v < E8; ++v) {
      const uint32_t q[4] = {kreg[v].x, kreg[v].y, kreg[v].z, kreg[v].w};
#pragma unroll
      for (int u = 0; u < 4; ++u) w = ((i >> 1) == 4 * v + u) ? q[u] : w;
    }
    return (i & 1) ? (w >> 16) : (w & 0xffffu);
  };
  mask_t est_bits = m_mid;  // bit i: owned key i is in the estimation zone
  for (mask_t m = m_gt1; m; m &= m - 1) {  // above T1: the ranks of a bin start at hist[bin] = keys above it
    const int i = lowest(m);
    const uint32_t key = key_at(i);
    const uint32_t slot = atomicAdd(&hist[sel_bin<BPT>(key)], 1u);
    sh_ret[slot] = (key << 16) | (0xffffu - (uint32_t)(cbeg + i));
  }
  {
    uint32_t rk = r1;  // ties at T1 enter in id order
    for (mask_t m = m_eq1; m; m &= m - 1, ++rk) {
      const int i = lowest(m);
      if (rk < lo1) sh_ret[g1 + rk] = (key_at(i) << 16) | (0xffffu - (uint32_t)(cbeg + i));
      else if (rk < hi1r) est_bits |= (mask_t)1 << i;
    }
    rk = r2;
    for (mask_t m = m_eq2; m && rk < hi2r; m &= m - 1, ++rk) est_bits |= (mask_t)1 << lowest(m);
  }
  __syncthreads();

  // ---- rank order: sh_ret is ordered by score; order runs of equal scores by ascending id ----
  // The size and first store row of the entry's cluster are requested before the walk over its run and
  // travel to the entry's final rank through LDS: their round trip to global memory runs under the walk
  // instead of after the next barrier.
  for (int r = tid; r < np; r += SEL_THREADS) {
    const uint32_t mine = sh_ret[r];
    const uint32_t kk = mine >> 16;
    uint32_t sz_e = 0;
    int32_t st_e = 0;
    if (cluster_size) {
      const size_t at = (size_t)g * nc + (0xffffu - (mine & 0xffffu));
      sz_e = (uint32_t)cluster_size[at];
      if (cluster_start) st_e = cluster_start[at];
    }
    int lo = r, rank_in_run = 0;
    while (lo > 0 && (sh_ret[lo - 1] >> 16) == kk) { --lo; rank_in_run += (sh_ret[lo] > mine); }
    int hi = r;
    while (hi + 1 < np && (sh_ret[hi + 1] >> 16) == kk) { ++hi; rank_in_run += (sh_ret[hi] > mine); }
    sh_sorted[lo + rank_in_run] = mine;
    sh_size[lo + rank_in_run] = sz_e;
    sh_start[lo + rank_in_run] = st_e;
  }
  __syncthreads();

  // ---- token layout of the retrieved clusters with the page cut-off ----
  // thread t owns the ranks [t*R, t*R + R)
  const int rb = tid * R;
  uint32_t sz[R], pg[R];
  int32_t st[R];
  int my_c[R];
  uint32_t pg_sum = 0, sz_sum = 0;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    sz[i] = 0; pg[i] = 0; st[i] = 0; my_c[i] = -1;
    if (rb + i < np) {
      my_c[i] = (int)(0xffffu - (sh_sorted[rb + i] & 0xffffu));
      st[i] = sh_start[rb + i];
      sz[i] = sh_size[rb + i];
      pg[i] = (sz[i] + page - 1) / page;
    }
    pg_sum += pg[i];
    sz_sum += sz[i];
  }
  uint32_t tok_run[R];
  uint32_t keep_bits = 0;
  int nkeep = 0;
  int32_t T_ret = 0;
  if (cluster_size) {
    uint32_t lay[2] = {pg_sum, sz_sum}, layp[2], layt[2];
    block_excl_scan<2>(lay, layp, layt, sh_scan[0]);
    uint32_t pg_run = layp[0], tk = layp[1];
    // kept clusters form a prefix because the page prefix is monotone; tokens before a kept
    // cluster all belong to kept clusters
#pragma unroll
    for (int i = 0; i < R; ++i) {
      tok_run[i] = tk;
      const int r = rb + i;
      const bool keep = r < np && pg_run + pg[i] <= (uint32_t)max_pages;
      // the kept clusters are the ranks 0 .. nkeep-1: the last of them publishes the totals
      if (keep) {
        keep_bits |= 1u << i;
        const uint32_t next_pg = (i + 1 < R) ? pg[i + 1] : (r + 1 < np ? (sh_size[r + 1] + page - 1) / page : 0u);
        const bool next_keep = r + 1 < np && pg_run + pg[i] + next_pg <= (uint32_t)max_pages;
        if (!next_keep) {
          sh_pages = pg_run + pg[i];
          sh_tret = tk + sz[i];
          sh_nkeep = (uint32_t)r + 1u;
        }
      }
      pg_run += pg[i];
      tk += sz[i];
    }
    __syncthreads();
    nkeep = (int)sh_nkeep;
    T_ret = (int32_t)sh_tret;
  }

  // ---- all global stores ----
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (rb + i < np) {
      ret_ids[(size_t)g * np + rb + i] = my_c[i];
      if (cI) cI[(size_t)g * k2 + rb + i] = my_c[i];
    }
  }
  {
    uint32_t est_off = est_first;
    for (int i = 0; i < E; ++i) {
      if ((est_bits >> i) & 1u) {
        est_ids[(size_t)g * es + est_off] = cbeg + i;
        if (cI) cI[(size_t)g * k2 + np + est_off] = cbeg + i;
        ++est_off;
      }
    }
  }
  if (!cluster_size) return;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int r = rb + i;
    if (r < np) {
      ret_tok_off[(size_t)g * (np + 1) + r] = (r < nkeep) ? (int32_t)tok_run[i] : T_ret;
      if (ret_start) ret_start[(size_t)g * np + r] = st[i];
    }
  }
  if (tid == 0) {
    ret_tok_off[(size_t)g * (np + 1) + np] = T_ret;
    meta[g * 4 + 0] = nkeep;
    meta[g * 4 + 1] = T_ret;
    meta[g * 4 + 2] = (int32_t)sh_pages;
    meta[g * 4 + 3] = 0;
  }
  // row table: each kept cluster writes the rows of its tokens
  if (!row_src || !cluster_start) return;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (!((keep_bits >> i) & 1u)) continue;
    int32_t* dst = row_src + (size_t)g * row_src_stride + tok_run[i];
    const int room = row_src_stride - (int)tok_run[i];
    for (int k = 0; k < (int)sz[i] && k < room; ++k) dst[k] = st[i] + k;
  }
}

// ------------------------------------------------------------------------------------
// select_radix_kernel: the selection of a group in one workgroup of NT threads, for up to NT probes.
//
// One compute unit works for a group, so what bounds it is the number of instructions its waves issue, then the barriers
// between the phases.  The rank thresholds come from two small histograms instead of one with a bin per key: 4 NT coarse
// bins (the key's upper bits; one 16-byte LDS access per thread to clear and to read them), then the keys inside the two
// threshold bins by their lower bits, which every wave scans for itself.  The retrieval zone (np of nc clusters) is
// gathered and sorted as (key, id) pairs in registers, so the rank order needs no histogram either.
// SRC says where the keys come from:
//   SEL_KEYS    16-bit keys of a preceding dist_kernel (many clusters times heads: the score sums want many compute units)
//   SEL_LOGITS  the logits and tile partials of a preceding score_kernel: the score sums are made here, one launch less
//   SEL_SCORE   the centroids (few clusters): the workgroup scores them with score_kernel's MFMA chain, two launches less
// Thread t owns the contiguous ids [t * E, t * E + E): ties are ranked by ascending id with plain prefix sums.  (Ids strided
// by 64, whose comparisons are masks in scalar registers, were slower from eight keys per thread on: the scalar unit
// issues one instruction per cycle for the whole compute unit as well.)
// ------------------------------------------------------------------------------------
#define SEL_KEYS 0
#define SEL_LOGITS 1
#define SEL_SCORE 2

struct SelectArgs {
  const uint16_t* keys;
  const uint16_t* q;
  const uint16_t* cent;
  float* logits;
  const float* tile_max;
  const float* tile_sum;
  const uint8_t* mask;
  const int32_t* cluster_size;
  const int32_t* cluster_start;
  uint16_t* dist_out;
  int64_t* cI;
  int32_t* ret_ids;
  int32_t* est_ids;
  int32_t* ret_tok_off;
  int32_t* ret_start;
  int32_t* row_src;
  int32_t* meta;
  int row_src_stride, gs, nc, ntiles, np, es, page, max_pages;
  float scale;
};

// Barrier over LDS traffic only: global stores issued before it stay in flight (__syncthreads waits for them as well).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// {a, b} = this lane's value and that of lane (lane ^ D), in either order; register moves only
template <int D>
__device__ __forceinline__ void lane_pair(uint32_t v, uint32_t& a, uint32_t& b) {
  typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
  a = v;
  if constexpr (D == 1) b = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true);   // quad_perm 1,0,3,2
  if constexpr (D == 2) b = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true);   // quad_perm 2,3,0,1
  if constexpr (D == 4) {
    const int m = __builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true);                      // half row mirrored: ^ 7
    b = (uint32_t)__builtin_amdgcn_update_dpp(0, m, 0x1B, 0xf, 0xf, true);                            // quad_perm 3,2,1,0: ^ 3
  }
  if constexpr (D == 8) b = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, true);  // row_ror:8
  if constexpr (D == 16) {   // rows 1 and 3 of one copy against rows 0 and 2 of the other
    const u32x2_t p = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_permlane16_swap(v, v, false, false));
    a = p.x; b = p.y;
  }
  if constexpr (D == 32) {
    const u32x2_t p = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_permlane32_swap(v, v, false, false));
    a = p.x; b = p.y;
  }
}

// lanes whose bit K and bit D are equal: those that keep the larger value of an exchange over 2^D in a merge of 2^K
constexpr uint64_t keep_mask(int K, int D) {
  uint64_t m = 0;
  for (int l = 0; l < 64; ++l)
    if (((l >> K) & 1) == ((l >> D) & 1)) m |= 1ull << l;
  return m;
}

// One exchange of a bitonic merge of 2^LK values over the distance 2^LD, then the shorter distances.  BUF: which of the
// two exchange buffers the next exchange between waves uses (they alternate: one barrier per exchange).
template <int LOG, int LK, int LD, int BUF>
__device__ __forceinline__ void bitonic_step(uint32_t& v, bool active, uint32_t* sh) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tid = threadIdx.x;
  constexpr bool ACROSS = LD >= 6;   // the other value is in another wave
  if constexpr (ACROSS) {
    if (active) sh[(BUF << LOG) + tid] = v;
    lds_barrier();
    if (active) {   // uniform in a wave, as is who keeps what
      const uint32_t o = sh[(BUF << LOG) + (tid ^ (1 << LD))];
      v = (((wave >> (LK - 6)) & 1) == ((wave >> (ACROSS ? LD - 6 : 0)) & 1)) ? max(v, o) : min(v, o);
    }
  } else if (active) {
    uint32_t a, b;
    lane_pair<(1 << LD)>(v, a, b);
    const uint32_t hi = max(a, b), lo = min(a, b);
    uint64_t keep = keep_mask(LK, LD);   // (bit LK of a lane is 0 when LK >= 6: bit LK of tid is the wave's)
    if (LK >= 6 && ((wave >> (LK >= 6 ? LK - 6 : 0)) & 1)) keep = ~keep;
    v = __builtin_amdgcn_inverse_ballot_w64(keep) ? hi : lo;
  }
  if constexpr (LD > 0) bitonic_step<LOG, LK, LD - 1, ACROSS ? 1 - BUF : BUF>(v, active, sh);
}

// Sorts the values of the threads tid < n in descending order (n a power of two, 64 <= n <= 2^LOG);
// sh: 2 * 2^LOG words.
template <int LOG, int LK = 1, int BUF = 0>
__device__ __forceinline__ void block_sort_desc(uint32_t& v, int n, uint32_t* sh) {
  if ((1 << LK) > n) return;   // uniform
  bitonic_step<LOG, LK, LK - 1, BUF>(v, (int)threadIdx.x < n, sh);
  constexpr int N = LK > 6 ? LK - 6 : 0;   // exchanges between waves of this merge
  if constexpr (LK < LOG) block_sort_desc<LOG, LK + 1, (N & 1) ? 1 - BUF : BUF>(v, n, sh);
}

// exclusive prefix sums over the NW waves of the block: inc[k] the wave-inclusive sums whose totals sit in sh[k * 16 + wave]
template <int NW>
__device__ __forceinline__ uint32_t wave_offset(const uint32_t* sh, uint32_t* total) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t sc = ri_wave_incl_scan(lane < NW ? sh[lane] : 0u);
  *total = (uint32_t)__builtin_amdgcn_readlane((int)sc, NW - 1);
  return wv > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)sc, wv - 1) : 0u;
}

// GSM: query heads padded to 4, 8 or 16 (SEL_LOGITS, SEL_SCORE).
template <int NT, int E, int GSM, bool HALF, int SRC>
__global__ __launch_bounds__(NT) void select_radix_kernel(SelectArgs P) {
  constexpr int NW = NT / 64, IDS = NT * E;
  constexpr int LOGT = NT == 256 ? 8 : (NT == 512 ? 9 : 10);
  constexpr int SHIFT = 16 - (LOGT + 2), FB = 1 << SHIFT;   // lower bits of a key, fine bins
  __shared__ __attribute__((aligned(16))) uint32_t hist[4 * NT];   // coarse bins; later the exchange area of the sort
  __shared__ uint32_t sh_fine[2][64], sh_scan[3][16], sh_sel[4], sh_tot[3], sh_ret[NT];
  __shared__ __attribute__((aligned(16))) uint16_t sh_p[SRC == SEL_SCORE ? IDS * GSM : 8];
  __shared__ float sh_a[SRC == SEL_SCORE ? NW : 1][16], sh_b[SRC == SEL_SCORE ? NW : 1][16];
  __shared__ __attribute__((aligned(16))) uint4 sh_rows[SRC == SEL_SCORE ? NW : 1][SRC == SEL_SCORE ? 256 : 1];
  const int g = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nc = P.nc, np = P.np, es = P.es, k2 = np + es, gs = P.gs;
  const int cbeg = tid * E;   // nc % 8 == 0: a thread's ids exist together, from E = 16 on in eights
  typedef typename std::conditional<(E <= 32), uint32_t, uint64_t>::type mask_t;

  *reinterpret_cast<uint4*>(&hist[4 * tid]) = ri_zero16();
  if (tid < 128) sh_fine[tid >> 6][lane] = 0u;
  if (tid < 3) sh_tot[tid] = 0u;
  sh_ret[tid] = 0u;

  // ---- this thread's keys, two per word ----
  uint32_t kw[(E + 1) / 2];
  if constexpr (SRC == SEL_KEYS) {
#pragma unroll
    for (int i = 0; i < E / 8; ++i) {
      const uint4 k = *reinterpret_cast<const uint4*>(P.keys + (size_t)g * nc + min(cbeg + 8 * i, nc - 8));
      kw[4 * i] = k.x; kw[4 * i + 1] = k.y; kw[4 * i + 2] = k.z; kw[4 * i + 3] = k.w;
    }
  } else {
    float d[E];
    const int cc = min(cbeg, nc - E);
    constexpr int MB = E < 4 ? E : 4;   // mask bytes per load
    typedef typename std::conditional<(MB == 4), uint32_t,
                                      typename std::conditional<(MB == 2), uint16_t, uint8_t>::type>::type mask_ld;
    uint32_t mk[E / MB];
#pragma unroll
    for (int i = 0; i < E / MB; ++i)
      mk[i] = P.mask ? *reinterpret_cast<const mask_ld*>(P.mask + (size_t)g * nc + cc + MB * i) : 0u;
    if constexpr (SRC == SEL_SCORE) {
      static_assert(E == 1, "a wave scores four tiles of 16 centroids: its own 64 ids' worth");
      const int r = lane & 15, h = lane >> 4;
      const uint16_t* cg = P.cent + (size_t)g * nc * RI_DIM;
      uint4 a[4][4], bq[4];
      // tile t of this wave: rows [16 * (wave + NW * t), + 16), so that few clusters still occupy every wave; rows past
      // the last centroid and heads past gs read a valid row (never used)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          a[t][i] = ri_ld16(cg + (size_t)min(16 * (wave + NW * t) + 4 * i + h, nc - 1) * RI_DIM + r * 8);
      }
      {
        const uint16_t* p = P.q + ((size_t)g * gs + min(r, gs - 1)) * RI_DIM + h * 8;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) bq[kk] = ri_ld16(p + kk * 32);
      }
      __builtin_amdgcn_sched_barrier(0);   // every load is in flight before the first product
      f32x4_t acc[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        uint4 at[4];
        ri_rows_put(sh_rows[wave], a[t]);
        ri_wave_sync();
        ri_rows_get(sh_rows[wave], at);
        ri_wave_sync();   // (a wave's LDS accesses happen in order: the next rows need not wait for these)
        f32x4_t x = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          x = HALF ? __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, at[kk]),
                                                            __builtin_bit_cast(f16x8_t, bq[kk]), x, 0, 0, 0)
                   : __builtin_amdgcn_mfma_f32_16x16x32_bf16(ri_as_bf16x8(at[kk]), ri_as_bf16x8(bq[kk]), x, 0, 0, 0);
        acc[t] = x * P.scale;
      }
      // softmax statistics: every wave's maximum and sum relative to it, folded by every lane for its head
      float lmax = -INFINITY, lsum = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (16 * (wave + NW * t) + 4 * h < nc)   // nc % 4 == 0: the four rows are valid together
#pragma unroll
          for (int i = 0; i < 4; ++i) lmax = fmaxf(lmax, acc[t][i]);
      lmax = fmaxf(lmax, __shfl_xor(lmax, 16));
      lmax = fmaxf(lmax, __shfl_xor(lmax, 32));
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (16 * (wave + NW * t) + 4 * h < nc)
#pragma unroll
          for (int i = 0; i < 4; ++i) lsum += __expf(acc[t][i] - lmax);
      lsum += __shfl_xor(lsum, 16);
      lsum += __shfl_xor(lsum, 32);
      if (h == 0) {
        sh_a[wave][r] = lmax;
        sh_b[wave][r] = lsum;
      }
      lds_barrier();
      float m = sh_a[0][r], z = 0.f;
#pragma unroll
      for (int w = 1; w < NW; ++w) m = fmaxf(m, sh_a[w][r]);
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float mw = sh_a[w][r];
        z += (mw == -INFINITY) ? 0.f : sh_b[w][r] * __expf(mw - m);   // a wave past the last centroid holds nothing
      }
      const float iz = 1.0f / z;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int c = 16 * (wave + NW * t) + 4 * h;
        if (r < gs && c < nc) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            sh_p[(c + i) * GSM + r] = ri_f32_to_e16<HALF>(__expf(ri_round_e16<HALF>(acc[t][i]) - m) * iz);
          *reinterpret_cast<f32x4_t*>(P.logits + ((size_t)g * gs + r) * nc + c) = acc[t];
        }
      }
      lds_barrier();
      d[0] = 0.f;
#pragma unroll
      for (int j = 0; j < GSM; ++j) {
        const float p = ri_e16_to_f32<HALF>(sh_p[cc * GSM + j]);
        d[0] += j < gs ? p : 0.f;
      }
    } else {
      constexpr int V = E < 4 ? E : 4;   // columns per load
      typedef float vec_t __attribute__((ext_vector_type(V)));
      vec_t x[GSM][E / V];
#pragma unroll
      for (int j = 0; j < GSM; ++j)
#pragma unroll
        for (int i = 0; i < E / V; ++i)
          x[j][i] = *reinterpret_cast<const vec_t*>(P.logits + ((size_t)g * gs + min(j, gs - 1)) * nc + cc + V * i);
      for (int j = wave; j < gs; j += NW) {
        float m, iz;
        ri_wave_reduce_partials(P.tile_max + (size_t)g * P.ntiles * gs, P.tile_sum + (size_t)g * P.ntiles * gs,
                                P.ntiles, gs, j, lane, &m, &iz);
        if (lane == 0) {
          sh_a[0][j] = m;
          sh_b[0][j] = iz;
        }
      }
      lds_barrier();
#pragma unroll
      for (int i = 0; i < E; ++i) d[i] = 0.f;
#pragma unroll
      for (int j = 0; j < GSM; ++j) {
        const float m = sh_a[0][j], iz = sh_b[0][j];
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const float p = ri_round_e16<HALF>(__expf(ri_round_e16<HALF>(x[j][i / V][i % V]) - m) * iz);
          d[i] += j < gs ? p : 0.f;
        }
      }
    }
    uint16_t bits[E + 1] = {};
#pragma unroll
    for (int i = 0; i < E; ++i) {
      bits[i] = ri_f32_to_e16<HALF>(d[i]);
      if ((mk[i / MB] >> (8 * (i % MB))) & 0xffu) bits[i] = ri_e16_lowest<HALF>();  // finfo(type).min
      if (P.dist_out && cbeg < nc) P.dist_out[(size_t)g * nc + cbeg + i] = bits[i];
    }
#pragma unroll
    for (int i = 0; i < (E + 1) / 2; ++i)
      kw[i] = ri_bf16_sort_key(bits[2 * i]) | ri_bf16_sort_key(bits[2 * i + 1]) << 16;
  }
  const int nown = min(max(nc - cbeg, 0), E);
  const auto key_of = [&](int i) { return (i & 1) ? kw[i >> 1] >> 16 : kw[i >> 1] & 0xffffu; };
  lds_barrier();

  // ---- rank thresholds: T1 = key of descending rank np-1, T2 = key of rank k2-1 ----
#pragma unroll
  for (int i = 0; i < E; ++i)
    if (i < nown) atomicAdd(&hist[key_of(i) >> SHIFT], 1u);
  lds_barrier();
  {
    const uint4 h4 = *reinterpret_cast<const uint4*>(&hist[4 * tid]);
    const uint32_t mine = h4.x + h4.y + h4.z + h4.w;
    const uint32_t inc = ri_wave_incl_scan(mine);
    if (lane == 63) sh_scan[0][wave] = inc;
    lds_barrier();
    uint32_t tot;
    const uint32_t above = (uint32_t)nc - wave_offset<NW>(sh_scan[0], &tot) - inc;   // keys in bins above this thread's
    // the thread whose bins hold the rank publishes the bin and the keys above it
    const auto find = [&](uint32_t rank, uint32_t* out) {
      if (rank - above < mine) {   // (unsigned: above <= rank < above + mine)
        const uint32_t hb[4] = {h4.x, h4.y, h4.z, h4.w};
        uint32_t a = above;
        int at = 3;
#pragma unroll
        for (int i = 3; i > 0; --i)
          if (at == i && rank - a >= hb[i]) { a += hb[i]; at = i - 1; }
        out[0] = tid * 4 + at;
        out[1] = a;
      }
    };
    find((uint32_t)(np - 1), sh_sel);
    find((uint32_t)(k2 - 1), sh_sel + 2);
  }
  lds_barrier();
  const uint32_t C1 = __builtin_amdgcn_readfirstlane(sh_sel[0]), C2 = __builtin_amdgcn_readfirstlane(sh_sel[2]);
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const uint32_t k = key_of(i), c = k >> SHIFT;
    if (i < nown && (c == C1 || c == C2)) atomicAdd(&sh_fine[c == C1 ? 0 : 1][k & (FB - 1)], 1u);
  }
  lds_barrier();
  // the fine bin of rank `rank` counted from the top of the coarse bin, and the keys above it
  const auto fine_bin = [&](const uint32_t* f, uint32_t rank, uint32_t& above) {
    const uint32_t c = lane < FB ? f[FB - 1 - (lane & (FB - 1))] : 0u;   // lane l: bin FB-1-l
    const uint32_t inc = ri_wave_incl_scan(c);
    const int at = __ffsll((long long)__ballot(inc > rank)) - 1;
    above = (uint32_t)__builtin_amdgcn_readlane((int)(inc - c), at);
    return (uint32_t)(FB - 1 - at);
  };
  const uint32_t s1 = __builtin_amdgcn_readfirstlane(sh_sel[1]), s2 = __builtin_amdgcn_readfirstlane(sh_sel[3]);
  uint32_t a1, a2;
  const uint32_t T1 = (C1 << SHIFT) | fine_bin(sh_fine[0], (uint32_t)(np - 1) - s1, a1);
  const uint32_t T2 = (C2 << SHIFT) | fine_bin(sh_fine[C1 == C2 ? 0 : 1], (uint32_t)(k2 - 1) - s2, a2);
  const uint32_t g1 = s1 + a1, g2 = s2 + a2;   // keys strictly above T1 / T2

  // ---- one scan places everything: keys above T1, ties at T1, ties at T2 and the keys strictly between ----
  // Tied keys are taken in ascending id order: tie rank r at T1 belongs to the retrieval zone
  // while g1 + r < np, then to the estimation zone while g1 + r < k2; at T2 while g2 + r < k2.
  // The owned keys are classified once, without branches, into bit masks (bit i = owned key i); the rare cases
  // (keys of the retrieval zone: np of nc; ties at a threshold) are then walked bit by bit.
  mask_t m_gt1 = 0, m_eq1 = 0, m_gt2 = 0, m_eq2 = 0;
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const uint32_t k = key_of(i);
    m_gt1 |= (mask_t)(k > T1) << i;
    m_eq1 |= (mask_t)(k == T1) << i;
    m_gt2 |= (mask_t)(k > T2) << i;
    m_eq2 |= (mask_t)(k == T2) << i;
  }
  {
    const mask_t ok = nown >= (int)(8 * sizeof(mask_t)) ? ~(mask_t)0 : ((mask_t)1 << nown) - 1;
    m_gt1 &= ok; m_eq1 &= ok; m_gt2 &= ok;
    m_eq2 &= T2 == T1 ? 0 : ok;
  }
  const mask_t m_mid = m_gt2 & ~m_gt1 & ~m_eq1;  // strictly between the thresholds: estimation zone
  const auto popc = [](mask_t m) { return (uint32_t)(sizeof(mask_t) == 8 ? __popcll((unsigned long long)m) : __popc((unsigned)m)); };
  const auto lowest = [](mask_t m) { return sizeof(mask_t) == 8 ? __ffsll((long long)m) - 1 : __ffs((int)m) - 1; };
  // keys above T1 are fewer than NT <= 1024, everything else is at most nc
  constexpr int NS = IDS <= 32768 ? 2 : 3;   // words: two counts share one while they fit
  uint32_t cnt[3] = {popc(m_gt1) | popc(m_eq1) << 12, popc(m_eq2), popc(m_mid)}, pre[3];
  if (NS == 2) cnt[1] |= cnt[2] << 16;
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    pre[k] = ri_wave_incl_scan(cnt[k]);
    if (lane == 63) sh_scan[k][wave] = pre[k];
  }
  lds_barrier();
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    uint32_t tot;
    pre[k] += wave_offset<NW>(sh_scan[k], &tot) - cnt[k];
  }
  const uint32_t r1 = pre[0] >> 12, r2 = NS == 2 ? pre[1] & 0xffffu : pre[1], mid_before = NS == 2 ? pre[1] >> 16 : pre[2];
  const uint32_t lo1 = (uint32_t)np - g1;                            // first tie rank of T1 in the est zone
  const uint32_t hi1r = (uint32_t)k2 > g1 ? (uint32_t)k2 - g1 : 0u;  // one past the last
  const uint32_t hi2r = (uint32_t)k2 > g2 ? (uint32_t)k2 - g2 : 0u;
  const uint32_t est_first = mid_before + (min(max(r1, lo1), hi1r) - lo1) + min(r2, hi2r);
  // owned key i (a register half chosen at run time: only the rare walks below need it)
  const auto key_at = [&](int i) {
    uint32_t w = 0;
#pragma unroll
    for (int v = 0; v < (E + 1) / 2; ++v) w = ((i >> 1) == v) ? kw[v] : w;
    return (i & 1) ? (w >> 16) : (w & 0xffffu);
  };
  mask_t est_bits = m_mid;  // bit i: owned key i is in the estimation zone
  {
    uint32_t slot = pre[0] & 0xfffu;
    for (mask_t m = m_gt1; m; m &= m - 1, ++slot) {
      const int i = lowest(m);
      sh_ret[slot] = (key_at(i) << 16) | (0xffffu - (uint32_t)(cbeg + i));
    }
    uint32_t rk = r1;  // ties at T1 enter in id order
    for (mask_t m = m_eq1; m && rk < hi1r; m &= m - 1, ++rk) {
      const int i = lowest(m);
      if (rk < lo1) sh_ret[g1 + rk] = (T1 << 16) | (0xffffu - (uint32_t)(cbeg + i));
      else est_bits |= (mask_t)1 << i;
    }
    rk = r2;
    for (mask_t m = m_eq2; m && rk < hi2r; m &= m - 1, ++rk) est_bits |= (mask_t)1 << lowest(m);
  }
  lds_barrier();

  // ---- rank order of the retrieval zone: descending score, ties by ascending id ----
  uint32_t v = sh_ret[tid];
  const bool in = tid < np;
  const auto id_of = [](uint32_t pair) { return (int)(0xffffu - (pair & 0xffffu)); };
  // (the sizes and first rows are requested for the unsorted entries, so that the loads behind the sort find them near)
  int32_t warm_size = 0, warm_start = 0;
  if (in && P.cluster_size) {
    warm_size = P.cluster_size[(size_t)g * nc + id_of(v)];
    if (P.cluster_start) warm_start = P.cluster_start[(size_t)g * nc + id_of(v)];
  }
  int n = 64;
  while (n < np) n <<= 1;
  block_sort_desc<LOGT>(v, n, hist);
  asm volatile("" : : "v"(warm_size), "v"(warm_start));
  const int my_c = id_of(v);
  uint32_t sz = 0;
  int32_t st = 0;
  if (in && P.cluster_size) {
    sz = (uint32_t)P.cluster_size[(size_t)g * nc + my_c];
    if (P.cluster_start) st = P.cluster_start[(size_t)g * nc + my_c];
  }

  // ---- token layout of the retrieved clusters with the page cut-off ----
  uint32_t tok = 0;
  int nkeep = 0;
  uint32_t T_ret = 0, pages = 0;
  bool keep = false;
  if (P.cluster_size) {
    const uint32_t pg = (sz + P.page - 1) / P.page;
    uint32_t pg_pre = ri_wave_incl_scan(pg);
    tok = ri_wave_incl_scan(sz);
    if (lane == 63) {
      sh_scan[0][wave] = pg_pre;
      sh_scan[1][wave] = tok;
    }
    lds_barrier();
    pg_pre += wave_offset<NW>(sh_scan[0], &pages) - pg;
    tok += wave_offset<NW>(sh_scan[1], &T_ret) - sz;
    nkeep = np;
    keep = in;
    if (pages > (uint32_t)P.max_pages) {   // uniform: the list is cut
      // the kept clusters are a prefix of the ranks (the page prefix is monotone): every wave reports its last one
      keep = in && pg_pre + pg <= (uint32_t)P.max_pages;
      const uint64_t kept = __ballot(keep);
      if (kept && lane == 63 - __clzll((long long)kept)) {
        atomicMax(&sh_tot[0], pg_pre + pg);
        atomicMax(&sh_tot[1], tok + sz);
        atomicMax(&sh_tot[2], (uint32_t)tid + 1u);
      }
      lds_barrier();
      pages = sh_tot[0];
      T_ret = sh_tot[1];
      nkeep = (int)sh_tot[2];
    }
  }

  // ---- all global stores ----
  // (behind every load: a load's wait covers the stores in front of it)
  if (in) {
    P.ret_ids[(size_t)g * np + tid] = my_c;
    if (P.cI) P.cI[(size_t)g * k2 + tid] = my_c;
  }
  {
    uint32_t at = est_first;
#pragma unroll
    for (int i = 0; i < E; ++i) {
      if ((est_bits >> i) & 1u) {
        P.est_ids[(size_t)g * es + at] = cbeg + i;
        if (P.cI) P.cI[(size_t)g * k2 + np + at] = cbeg + i;
        ++at;
      }
    }
  }
  if (!P.cluster_size) return;
  if (in) {
    P.ret_tok_off[(size_t)g * (np + 1) + tid] = (int32_t)((tid < nkeep) ? tok : T_ret);
    if (P.ret_start) P.ret_start[(size_t)g * np + tid] = st;
  }
  if (tid == 0) {
    P.ret_tok_off[(size_t)g * (np + 1) + np] = (int32_t)T_ret;
    P.meta[g * 4 + 0] = nkeep;
    P.meta[g * 4 + 1] = (int32_t)T_ret;
    P.meta[g * 4 + 2] = (int32_t)pages;
    P.meta[g * 4 + 3] = 0;
  }
  if (P.row_src && P.cluster_start && keep) {   // row table: each kept cluster writes the rows of its tokens
    int32_t* dst = P.row_src + (size_t)g * P.row_src_stride + tok;
    const int room = P.row_src_stride - (int)tok;
    for (int k = 0; k < (int)sz && k < room; ++k) dst[k] = st + k;
  }
}

// ------------------------------------------------------------------------------------
// C entry points
// ------------------------------------------------------------------------------------
static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

extern "C" size_t ri_score_select_workspace_bytes(int BG, int gs, int nc) {
  if (BG <= 0 || gs <= 0 || nc <= 0) return 0;
  const size_t ntiles = (size_t)(nc + RI_SCORE_TILE - 1) / RI_SCORE_TILE;
  return 2 * align256((size_t)BG * ntiles * gs * sizeof(float)) + align256((size_t)BG * nc * sizeof(uint16_t));
}

template <int NT, int E, int GSM, int SRC>
static void launch_select(const SelectArgs& P, int BG, bool half, hipStream_t s) {
  if (half) select_radix_kernel<NT, E, GSM, true, SRC><<<BG, NT, 0, s>>>(P);
  else select_radix_kernel<NT, E, GSM, false, SRC><<<BG, NT, 0, s>>>(P);
}
template <int NT, int E, int SRC>
static void launch_select_heads(const SelectArgs& P, int BG, bool half, hipStream_t s) {
  if (P.gs <= 4) launch_select<NT, E, 4, SRC>(P, BG, half, s);
  else if (P.gs <= 8) launch_select<NT, E, 8, SRC>(P, BG, half, s);
  else launch_select<NT, E, 16, SRC>(P, BG, half, s);
}

static int score_select_impl(const void* q, const void* centroids, const uint8_t* mask,
                             const int32_t* cluster_size_i32, const int32_t* cluster_start, float* logits, void* dist,
                             int64_t* cI, int32_t* ret_ids, int32_t* est_ids, int32_t* ret_tok_off, int32_t* ret_start,
                             int32_t* row_src, int row_src_stride, int32_t* meta, int BG, int gs, int nc, int np, int es,
                             int page, int max_pages, float scale, void* workspace, size_t workspace_bytes, bool half,
                             ri_stream_t stream) {
  if (!q || !centroids || !logits || !ret_ids || !workspace) return RI_ERR_ARG;
  if (ri_any_misaligned16(q, centroids, logits, workspace)) return RI_ERR_ARG;
  if (BG <= 0 || gs <= 0 || gs > 16 || nc <= 0 || (nc % 8) != 0) return RI_ERR_ARG;
  if (np <= 0 || np > SEL_MAX_PROBES || es < 0 || np + es > nc || nc > 65536) return RI_ERR_ARG;
  if (es > 0 && !est_ids) return RI_ERR_ARG;
  if (cluster_size_i32 && (!ret_tok_off || !meta || page <= 0 || max_pages <= 0)) return RI_ERR_ARG;
  if (workspace_bytes < ri_score_select_workspace_bytes(BG, gs, nc)) return RI_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  const int ntiles = (nc + RI_SCORE_TILE - 1) / RI_SCORE_TILE;
  char* w = (char*)workspace;
  float* tmax = (float*)w;
  w += align256((size_t)BG * ntiles * gs * sizeof(float));
  float* tsum = (float*)w;
  w += align256((size_t)BG * ntiles * gs * sizeof(float));
  uint16_t* keys = (uint16_t*)w;
  const SelectArgs P = {keys, (const uint16_t*)q, (const uint16_t*)centroids, logits, tmax, tsum, mask,
                        cluster_size_i32, cluster_start, (uint16_t*)dist, cI, ret_ids, est_ids, ret_tok_off, ret_start,
                        row_src, meta, row_src_stride, gs, nc, ntiles, np, es, page, max_pages, scale};
  // One compute unit reads 20 KB per microsecond from memory and up to 100 from its L2.  Its own scoring therefore pays up to
  // 512 clusters (8 groups of 4 heads: 8.0 us; 640 clusters 10.3 against 10.0 for two launches, 16 groups of 1024 11.8
  // against 10.7; for 128 groups of 8 heads it is still ahead there, 14.0 against 16.0, but not by what the rule would
  // cost), its own score sums up to about 112 KB of logits (8 groups of 4 heads, 4096 clusters: 14.4 against 15.5 us; 32 groups of
  // 4 heads, 8192 clusters: 26.7 against 26.1).  Past 4096 clusters a thread holds eight of them: with more than four
  // heads that is 64 logits in registers, and many compute units are the faster ones again (4 .. 32 groups of 5 and 6
  // heads, 4104 .. 5728 clusters: 16.1 .. 22.6 us with dist_kernel, 20.0 .. 26.2 without).
  if (nc <= 512) {
    if (nc <= 256) launch_select_heads<256, 1, SEL_SCORE>(P, BG, half, s);
    else launch_select_heads<512, 1, SEL_SCORE>(P, BG, half, s);
    RI_HIP_CHECK_LAUNCH();
    return RI_OK;
  }
  int rc = ri_launch_score(q, centroids, logits, tmax, tsum, BG, gs, nc, scale, half, s);
  if (rc) return rc;
  if (nc * gs <= 28 * 1024 && nc <= (gs <= 4 ? 8192 : 4096) && np <= SEL_THREADS) {
    // as few waves as the clusters and the probes leave room for: what a wave does once costs all of them
    if (nc <= 1024 && np <= 512) launch_select_heads<512, 2, SEL_LOGITS>(P, BG, half, s);
    else if (nc <= 2048 && np <= 512) launch_select_heads<512, 4, SEL_LOGITS>(P, BG, half, s);
    else if (nc <= 4096) launch_select_heads<SEL_THREADS, 4, SEL_LOGITS>(P, BG, half, s);
    else launch_select<SEL_THREADS, 8, 4, SEL_LOGITS>(P, BG, half, s);   // gs <= 4 here, the heads this one holds
    RI_HIP_CHECK_LAUNCH();
    return RI_OK;
  }
  const dim3 dgrid((nc + DIST_IDS - 1) / DIST_IDS, BG);
#define RI_DIST_LAUNCH(GSM)                                                                                       \
  do {                                                                                                            \
    if (half)                                                                                                     \
      dist_kernel<GSM, true><<<dgrid, 256, 0, s>>>(logits, tmax, tsum, mask, keys, (uint16_t*)dist, gs, nc, ntiles); \
    else                                                                                                          \
      dist_kernel<GSM, false><<<dgrid, 256, 0, s>>>(logits, tmax, tsum, mask, keys, (uint16_t*)dist, gs, nc, ntiles); \
  } while (0)
  if (gs <= 4) RI_DIST_LAUNCH(4);
  else if (gs <= 8) RI_DIST_LAUNCH(8);
  else RI_DIST_LAUNCH(16);
#undef RI_DIST_LAUNCH
  RI_HIP_CHECK_LAUNCH();
  const int per_thread = (nc + SEL_THREADS - 1) / SEL_THREADS;
#define RI_SELECT_LAUNCH_T(E8, R, BPT)                                                                               \
  select_kernel<E8, R, BPT><<<BG, SEL_THREADS, 0, s>>>(keys, cluster_size_i32, cluster_start, cI, ret_ids, est_ids,  \
                                                       ret_tok_off, ret_start, row_src, row_src_stride, meta, nc, np, \
                                                       es, page, max_pages)
#define RI_SELECT_LAUNCH(E8, R)                             \
  do {                                                      \
    if (half) RI_SELECT_LAUNCH_T(E8, R, SEL_BPT_F16);       \
    else RI_SELECT_LAUNCH_T(E8, R, SEL_BPT_BF16);           \
  } while (0)
  if (np <= SEL_THREADS && per_thread <= 8) {
    launch_select<SEL_THREADS, 8, 4, SEL_KEYS>(P, BG, half, s);
  } else if (np <= SEL_THREADS && per_thread <= 16) {
    launch_select<SEL_THREADS, 16, 4, SEL_KEYS>(P, BG, half, s);
  } else if (np < SEL_THREADS) {
    if (per_thread <= 32) RI_SELECT_LAUNCH(4, 1);
    else RI_SELECT_LAUNCH(8, 1);
  } else {  // long probe lists only occur with many clusters
    if (per_thread <= 16) RI_SELECT_LAUNCH(2, 4);
    else if (per_thread <= 32) RI_SELECT_LAUNCH(4, 4);
    else RI_SELECT_LAUNCH(8, 4);
  }
#undef RI_SELECT_LAUNCH
#undef RI_SELECT_LAUNCH_T
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_score_select(const void* q, const void* centroids, const uint8_t* mask,
                               const int32_t* cluster_size_i32, const int32_t* cluster_start,
                               float* logits, void* dist, int64_t* cI, int32_t* ret_ids,
                               int32_t* est_ids, int32_t* ret_tok_off, int32_t* ret_start,
                               int32_t* row_src, int row_src_stride, int32_t* meta, int BG, int gs, int nc, int np,
                               int es, int page, int max_pages, float scale, void* workspace,
                               size_t workspace_bytes, ri_stream_t stream) {
  return score_select_impl(q, centroids, mask, cluster_size_i32, cluster_start, logits, dist, cI, ret_ids, est_ids,
                           ret_tok_off, ret_start, row_src, row_src_stride, meta, BG, gs, nc, np, es, page, max_pages,
                           scale, workspace, workspace_bytes, false, stream);
}

extern "C" int ri_score_select_f16(const void* q, const void* centroids, const uint8_t* mask,
                                   const int32_t* cluster_size_i32, const int32_t* cluster_start,
                                   float* logits, void* dist, int64_t* cI, int32_t* ret_ids,
                                   int32_t* est_ids, int32_t* ret_tok_off, int32_t* ret_start,
                                   int32_t* row_src, int row_src_stride, int32_t* meta, int BG, int gs, int nc, int np,
                                   int es, int page, int max_pages, float scale, void* workspace,
                                   size_t workspace_bytes, ri_stream_t stream) {
  return score_select_impl(q, centroids, mask, cluster_size_i32, cluster_start, logits, dist, cI, ret_ids, est_ids,
                           ret_tok_off, ret_start, row_src, row_src_stride, meta, BG, gs, nc, np, es, page, max_pages,
                           scale, workspace, workspace_bytes, true, stream);
}

static int score_logits_impl(const void* q, const void* centroids, float* logits, int BG, int gs, int nc, float scale,
                             void* workspace, size_t workspace_bytes, bool half, ri_stream_t stream) {
  if (!q || !centroids || !logits || !workspace) return RI_ERR_ARG;
  if (ri_any_misaligned16(q, centroids, logits, workspace)) return RI_ERR_ARG;
  if (BG <= 0 || gs <= 0 || gs > 16 || nc <= 0 || (nc % 4) != 0) return RI_ERR_ARG;
  if (workspace_bytes < ri_score_select_workspace_bytes(BG, gs, nc)) return RI_ERR_WORKSPACE;
  const int ntiles = (nc + RI_SCORE_TILE - 1) / RI_SCORE_TILE;
  float* tmax = (float*)workspace;
  float* tsum = (float*)((char*)workspace + align256((size_t)BG * ntiles * gs * sizeof(float)));
  return ri_launch_score(q, centroids, logits, tmax, tsum, BG, gs, nc, scale, half, (hipStream_t)stream);
}

extern "C" int ri_score_logits(const void* q, const void* centroids, float* logits, int BG, int gs, int nc,
                               float scale, void* workspace, size_t workspace_bytes, ri_stream_t stream) {
  return score_logits_impl(q, centroids, logits, BG, gs, nc, scale, workspace, workspace_bytes, false, stream);
}

extern "C" int ri_score_logits_f16(const void* q, const void* centroids, float* logits, int BG, int gs, int nc,
                                   float scale, void* workspace, size_t workspace_bytes, ri_stream_t stream) {
  return score_logits_impl(q, centroids, logits, BG, gs, nc, scale, workspace, workspace_bytes, true, stream);
}
