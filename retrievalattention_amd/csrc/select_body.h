// Device code of the cluster selection that select.hip and step.hip share (gfx950).
#pragma once
#include <type_traits>

#include "ri_common.h"

// ------------------------------------------------------------------------------------
// select_group: the selection of a group by one workgroup of NT threads, for up to NT probes (select_radix_kernel, and the
// first half of step_kernel).
//
// One compute unit works for a group, so what bounds it is the number of instructions its waves issue, then the barriers
// between the phases.  The rank thresholds come from one histogram with a bin per key over the octaves that scores are found in
// (SEL_SPAN below), or from the keys' upper bits and then the lower ones of the two threshold bins; bins of one key are also hit
// by fewer lanes at once.  The places above a bin stay in its word, so a key of the retrieval zone (np of nc) takes its place by
// one atomic, and the few that share a bin are put in order by looking at each other.  In two histograms always, with the
// retrieval zone sorted as pairs (36 exchanges for 256 of them), cycles of one of two waves of a SIMD: 32 groups of 4 heads, 8192
// clusters, 147 probes 18800 -> 14000 from the first load to the tables, steps of four layers 187.8 -> 179.3 us; 64 of 8, 16384,
// 294: 27300 -> 19500, a step 131.9 -> 128.4.
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
  uint16_t* keys;
  const uint16_t* q;
  const uint16_t* cent;
  float* logits;
  float* tile_max;
  float* tile_sum;
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
  int row_src_stride, gs, nc, ntiles, np, es, page, max_pages, tile;
  float scale;
};

// Barrier over LDS traffic only: global stores issued before it stay in flight (__syncthreads waits for them as well).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

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
    ri_lane_pair<(1 << LD)>(v, a, b);
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

// Where the rest of a workgroup that goes on with the attention finds the selection (LDS).
struct SelectKept {
  float* logits;   // [nc][GSM]: SEL_SCORE
  int* est;        // [es]
  int* off;        // [np + 1]
  int* start;      // [np]
  int* ids;        // [np]
  int* meta;       // [4]
  uint32_t* scratch;   // [SEL_SCRATCH<NT>] what the attention has not laid anything in yet
  uint4* area;         // SEL_SCORE of more than eight heads: SEL_AREA<NT, GSM> bytes, the same (their logits go to memory)
};
template <int NT, int GSM>
constexpr size_t SEL_AREA = NT / 64 * 256 * sizeof(uint4) + (size_t)NT * GSM * sizeof(uint16_t);
enum { KEEP_NONE, KEEP_TABLES };

// Bins of the rank search.  Scores are sums of at most sixteen probabilities: in bfloat16 (128 keys to an octave) a bin for
// each of the 4031 keys up to that of 16, 1.5 * 2^-28 the lowest, finds a rank in one pass; the first 64 bins and the last hold what
// lies beyond, and where a rank falls there the search is made again by the keys' upper bits.  Half has too many keys for that.
// 64: what lies below is dealt to them by lane.  Peaked heads leave most of their clusters there, and on one bin those are one
// atomic after the other.  Where only the estimation zone's rank falls there and a thread has one key or two (BYTES), the keys below
// are searched by their upper bytes and then by the lower ones, which is less than the whole search again; of more keys the code of it
// costs all other steps more (16 groups of 2 heads, 10 % of 2496 clusters 25.2 -> 25.5).  Captured layers whose heads are as
// peaked, us, always two histograms / one bin below and the whole search again / as it is: 2 groups of 8 heads, 8192 clusters 27.7 / 33.3 /
// 27.0; 32 of 4, 8192 47.1 / 52.7 / 45.0; 16 of 4, 1024 18.8 / 19.9 / 18.9; 8 of 4, 512 17.2 / 17.7 / 16.7; a selection by itself, 8 of
// 8, 4096 14.1 / 18.4 / 15.3.  Keys inside cost an instruction for two.
#define SEL_SPAN 4096
#define SEL_WINDOW 0xB182u   // keys from here on have a bin, but see SEL_BELOW; bin SEL_SPAN - 2: the key of 16.0, 0xC180
#define SEL_BELOW 64         // bins that what lies below the next one's key shares
#define SEL_SHIFT 4          // by the upper bits: lower bits of a key
#define SEL_RUN 32u          // longest run of a bin that its entries put in order by looking at all of it
template <int NT>
constexpr int SEL_SCRATCH = SEL_SPAN + 3 * NT;

typedef uint16_t sel_pair __attribute__((ext_vector_type(2)));
// the bins of two keys
__device__ __forceinline__ uint32_t sel_bins(uint32_t keys, bool window) {
  const sel_pair k = __builtin_bit_cast(sel_pair, keys), lo = {SEL_WINDOW, SEL_WINDOW}, last = {SEL_SPAN - 1, SEL_SPAN - 1};
  const sel_pair w = __builtin_elementwise_min(__builtin_elementwise_sub_sat(k, lo), last), u = k >> (sel_pair){SEL_SHIFT, SEL_SHIFT};
  return __builtin_bit_cast(uint32_t, window ? w : u);
}
// 1 in the halves where a is above b (written out: the compiler makes two comparisons and two selects of it)
__device__ __forceinline__ uint32_t sel_above(uint32_t a, uint32_t b) {
  uint32_t m;
  asm("v_pk_sub_u16 %0, %1, %2 clamp\n\tv_pk_min_u16 %0, %0, 1 op_sel_hi:[1,0]" : "=&v"(m) : "v"(a), "v"(b));
  return m;
}

// GSM: query heads padded to 4, 8 or 16 (SEL_LOGITS, SEL_SCORE).  KEEP: the results are left in K in place of
// memory (a load's wait covers the stores in front of it: the caller stores behind the attention).
// ahead(): what the caller wants on its way behind the selection's first loads.  Returns the cluster of the thread's rank, -1
// past the list.
template <int NT, int E, int GSM, bool HALF, int SRC, int KEEP, typename Ahead>
__device__ __forceinline__ int select_group(const SelectArgs& P, const int g, const SelectKept& K, Ahead&& ahead) {
  constexpr bool STORE = !KEEP;
  constexpr int NW = NT / 64, IDS = NT * E;
  constexpr int LOGT = NT == 256 ? 8 : (NT == 512 ? 9 : 10);
  constexpr int BPT = SEL_SPAN / NT, FB = 1 << SEL_SHIFT;   // bins of a thread, fine bins
  static_assert(IDS <= 16384 * 2 && E <= 32, "counts in half a word, owned keys in one");
  constexpr bool BYTES = E <= 2;   // the estimation zone's rank below the window is found by two small passes, see SEL_BELOW
  __shared__ __attribute__((aligned(16))) uint32_t sh_own[KEEP ? 4 : SEL_SCRATCH<NT>];
  uint32_t* const hist = KEEP ? K.scratch : sh_own;   // bins; also the exchange area of the sort
  uint32_t* const sh_rank = hist + SEL_SPAN;          // [3][NT] entries, sizes and first rows in rank order
  __shared__ uint32_t sh_fine[2][FB], sh_scan[3][16], sh_sel[5], sh_tot[3], sh_ret[NT];
  // Sizes and first rows of all clusters, requested with the first loads: the ones of the retrieval zone are only known
  // after the sort, and a round trip for them there is a tenth of the kernel.  (With more clusters that is more than it saves:
  // 16 groups of 1024 10.4 us either way.)
  constexpr bool STAGED = SRC == SEL_SCORE;
  constexpr bool OWN = GSM <= 8;   // who computes the probabilities, see below
  __shared__ __attribute__((aligned(16))) int32_t sh_size[STAGED ? IDS : 4], sh_row[STAGED ? IDS : 4];
  __shared__ __attribute__((aligned(16))) float sh_x[SRC == SEL_SCORE && OWN && !KEEP ? IDS * GSM : 4];
  constexpr bool LENT = KEEP && SRC == SEL_SCORE && !OWN;   // the rows' turn and the probabilities lie in what the attention lends
  __shared__ __attribute__((aligned(16))) uint16_t sh_p_own[SRC == SEL_SCORE && !OWN && !LENT ? IDS * GSM : 8];
  __shared__ float sh_a[SRC == SEL_SCORE ? NW : 1][16], sh_b[SRC == SEL_SCORE ? NW : 1][16];
  __shared__ __attribute__((aligned(16))) uint4 sh_rows_own[SRC == SEL_SCORE && !LENT ? NW : 1][SRC == SEL_SCORE ? 256 : 1];
  auto* const sh_rows = LENT ? reinterpret_cast<uint4 (*)[SRC == SEL_SCORE ? 256 : 1]>(K.area) : sh_rows_own;
  uint16_t* const sh_p = LENT ? reinterpret_cast<uint16_t*>(K.area + NW * 256) : sh_p_own;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nc = P.nc, np = P.np, es = P.es, k2 = np + es, gs = P.gs;
  const int cbeg = tid * E;   // nc % 8 == 0: a thread's ids exist together, from E = 16 on in eights
  typedef uint32_t mask_t;

  const auto clear_bins = [&]() {
#pragma unroll
    for (int i = 0; i < BPT; i += 4) *reinterpret_cast<uint4*>(&hist[BPT * tid + i]) = ri_zero16();
  };
  clear_bins();
  if (tid < 2 * FB) sh_fine[tid / FB][tid % FB] = 0u;
  if (tid < 3) sh_tot[tid] = 0u;
  if (tid == 3) sh_sel[4] = 0u;
  sh_ret[tid] = 0u;

  int32_t own_size = 0, own_row = 0;
  if (STAGED && P.cluster_size) {
    own_size = P.cluster_size[(size_t)g * nc + min(tid, nc - 1)];
    if (P.cluster_start) own_row = P.cluster_start[(size_t)g * nc + min(tid, nc - 1)];
  }

  // ---- this thread's keys, two per word ----
  uint32_t kw[(E + 1) / 2];
  if constexpr (SRC == SEL_KEYS) {
#pragma unroll
    for (int i = 0; i < E / 8; ++i) {
      const uint4 k = *reinterpret_cast<const uint4*>(P.keys + (size_t)g * nc + min(cbeg + 8 * i, nc - 8));
      kw[4 * i] = k.x; kw[4 * i + 1] = k.y; kw[4 * i + 2] = k.z; kw[4 * i + 3] = k.w;
    }
    ahead();
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
      {
        const uint16_t* p = P.q + ((size_t)g * gs + min(r, gs - 1)) * RI_DIM + h * 8;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) bq[kk] = ri_ld16(p + kk * 32);
      }
      // tile t of this wave: rows [16 * (wave + NW * t), + 16), so that few clusters still occupy every wave; rows past
      // the last centroid and heads past gs read a valid row (never used)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          a[t][i] = ri_ld16(cg + (size_t)min(16 * (wave + NW * t) + 4 * i + h, nc - 1) * RI_DIM + r * 8);
      }
      ahead();
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
      // softmax statistics: every wave's maximum and sum relative to it, folded by every lane for its head.  (No branches: a
      // row past the last centroid scores -inf and weighs 0; nc % 4 == 0, the four rows are valid together.)
      float lmax = -INFINITY, lsum = 0.f;
      f32x4_t there[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bool in = 16 * (wave + NW * t) + 4 * h < nc;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          there[t][i] = in ? acc[t][i] : -INFINITY;
          lmax = fmaxf(lmax, there[t][i]);
        }
      }
      lmax = ri_xor_max<32>(ri_xor_max<16>(lmax));
      const float base = lmax == -INFINITY ? 0.f : lmax;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) lsum += __expf(there[t][i] - base);
      lsum = ri_xor_sum<32>(ri_xor_sum<16>(lsum));
      if (h == 0) {
        sh_a[wave][r] = lmax;
        sh_b[wave][r] = lsum;
      }
      // The products leave a cluster's heads to neighbouring lanes: with up to eight of them half of the lanes or more have
      // nothing, so the scores go through LDS to the thread that owns the cluster, which computes gs probabilities (8 groups
      // of 4 heads, 512 clusters with the sizes at hand: 7.9 -> 7.7 us, 256: 6.9 -> 6.6); with more heads the lanes that have
      // the scores compute sixteen each (8 groups of 12: 8.4, the other way 9.3).
      float* const xs = KEEP ? K.logits : sh_x;   // [cluster][GSM], of as many clusters as there are threads
      if (OWN && r < gs) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) xs[(16 * (wave + NW * t) + 4 * h + i) * GSM + r] = acc[t][i];
      }
      sh_size[tid] = own_size;
      sh_row[tid] = own_row;
      lds_barrier();
      float mw[NW], zw[NW], m, z = 0.f;   // of head r
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        mw[w] = sh_a[w][r];
        zw[w] = sh_b[w][r];
      }
      m = mw[0];
#pragma unroll
      for (int w = 1; w < NW; ++w) m = fmaxf(m, mw[w]);
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        float part = zw[w] * __expf(mw[w] - m);
        asm("" : "+v"(part));   // (else each becomes a branch with its own wait)
        z += (mw[w] == -INFINITY) ? 0.f : part;   // a wave past the last centroid holds nothing
      }
      const float iz = 1.0f / z;
      d[0] = 0.f;
      if constexpr (OWN) {
        float x[GSM];
#pragma unroll
        for (int j = 0; j < GSM; j += 4) {
          const float4 v = *reinterpret_cast<const float4*>(xs + cc * GSM + j);
          x[j] = v.x; x[j + 1] = v.y; x[j + 2] = v.z; x[j + 3] = v.w;
        }
#pragma unroll
        for (int j = 0; j < GSM; ++j) {
          const float mj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m), j));
          const float izj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(iz), j));
          const float p = ri_round_e16<HALF>(__expf(ri_round_e16<HALF>(x[j]) - mj) * izj);
          d[0] += j < gs ? p : 0.f;
        }
        if (STORE && cbeg < nc)
#pragma unroll
          for (int j = 0; j < GSM; ++j)
            if (j < gs) P.logits[((size_t)g * gs + j) * nc + cbeg] = x[j];
      } else {
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
#pragma unroll
        for (int j = 0; j < GSM; ++j) {
          const float p = ri_e16_to_f32<HALF>(sh_p[cc * GSM + j]);
          d[0] += j < gs ? p : 0.f;
        }
      }
    } else {
      constexpr int V = E < 4 ? E : 4;   // columns per load
      typedef float vec_t __attribute__((ext_vector_type(V)));
      vec_t x[GSM][E / V];
      // (a group's logits lie within 1 MB: 32-bit offsets from one base)
      const char* const lg = reinterpret_cast<const char*>(P.logits + (size_t)g * gs * nc);
#pragma unroll
      for (int j = 0; j < GSM; ++j)
#pragma unroll
        for (int i = 0; i < E / V; ++i)
          x[j][i] = *reinterpret_cast<const vec_t*>(lg + (uint32_t)(min(j, gs - 1) * nc + cc + V * i) * 4u);
      // (at most 64 partials: narrow tiles up to 4096 clusters, wide ones past them.  All on their way before any is looked at.)
      constexpr int HPW = (GSM + NW - 1) / NW;
      const size_t part = (size_t)g * P.ntiles * gs;
      const char *const pm = reinterpret_cast<const char*>(P.tile_max + part), *const ps = reinterpret_cast<const char*>(P.tile_sum + part);
      float pm0[HPW], ps0[HPW];
#pragma unroll
      for (int k = 0; k < HPW; ++k) {
        const uint32_t at = (uint32_t)(min(lane, P.ntiles - 1) * gs + min(wave + k * NW, gs - 1)) * 4u;
        pm0[k] = *reinterpret_cast<const float*>(pm + at);
        ps0[k] = *reinterpret_cast<const float*>(ps + at);
      }
      ahead();
#pragma unroll
      for (int k = 0; k < HPW; ++k) {
        float m, iz;
        ri_wave_reduce_partials(lane < P.ntiles ? pm0[k] : -INFINITY, lane < P.ntiles ? ps0[k] : 0.f, &m, &iz);
        if (lane == 0 && wave + k * NW < gs) {
          sh_a[0][wave + k * NW] = m;
          sh_b[0][wave + k * NW] = iz;
        }
      }
      lds_barrier();
#pragma unroll
      for (int i = 0; i < E; ++i) d[i] = 0.f;
#pragma unroll
      for (int j = 0; j < GSM; ++j) {
        // (uniform; of sixteen the compiler moves every load behind its branch, so there the heads past gs count for nothing)
        if (GSM <= 8 && j >= gs) break;
        const float m = sh_a[0][j], iz = sh_b[0][j];
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const float p = ri_round_e16<HALF>(__expf(ri_round_e16<HALF>(x[j][i / V][i % V]) - m) * iz);
          d[i] += GSM <= 8 || j < gs ? p : 0.f;
        }
      }
    }
    // (looked at here: the compiler compares where it loads, which is a wait in front of every other load)
    if (SRC == SEL_SCORE) asm volatile("" : "+v"(mk[0]));
    uint16_t bits[E + 1] = {};
#pragma unroll
    for (int i = 0; i < E; ++i) {
      bits[i] = ri_f32_to_e16<HALF>(d[i]);
      if ((mk[i / MB] >> (8 * (i % MB))) & 0xffu) bits[i] = ri_e16_lowest<HALF>();  // finfo(type).min
      if (!KEEP && P.dist_out && cbeg < nc) P.dist_out[(size_t)g * nc + cbeg + i] = bits[i];
    }
#pragma unroll
    for (int i = 0; i < (E + 1) / 2; ++i)
      kw[i] = ri_bf16_sort_key(bits[2 * i]) | ri_bf16_sort_key(bits[2 * i + 1]) << 16;
  }
  const auto key_of = [&](int i) { return (i & 1) ? kw[i >> 1] >> 16 : kw[i >> 1] & 0xffffu; };
  const int nown = min(max(nc - cbeg, 0), E);
  constexpr int KW = (E + 1) / 2, EIGHTS = (E + 7) / 8;   // (nc % 8 == 0: a thread's keys exist together, or eight by eight)
  lds_barrier();

  // ---- rank thresholds: T1 = key of descending rank np-1, T2 = key of rank k2-1 ----
  // Afterwards a bin's word holds the keys above the bin, and in the upper half its own.
  bool window = !HALF;
  uint32_t spread = window ? (uint32_t)lane * 0x10001u : 0u;   // the least bin of either key
  uint32_t C1, s1, C2, s2;
  for (;;) {   // (twice at most: by the window, then by the upper bits)
#pragma unroll
    for (int o = 0; o < EIGHTS; ++o)
      if (8 * o < nown) {
#pragma unroll
        for (int v = 4 * o; v < 4 * o + 4 && v < KW; ++v) {
          const uint32_t b = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(sel_pair, sel_bins(kw[v], window)),
                                                                                     __builtin_bit_cast(sel_pair, spread)));
          atomicAdd(&hist[b & 0xffffu], 1u);
          if (E > 1) atomicAdd(&hist[b >> 16], 1u);
        }
      }
    lds_barrier();
    {
      uint32_t h[BPT], mine = 0;
#pragma unroll
      for (int i = 0; i < BPT; i += 4) {
        const uint4 h4 = *reinterpret_cast<const uint4*>(&hist[BPT * tid + i]);
        h[i] = h4.x; h[i + 1] = h4.y; h[i + 2] = h4.z; h[i + 3] = h4.w;
      }
#pragma unroll
      for (int i = 0; i < BPT; ++i) mine += h[i];
      const uint32_t inc = ri_wave_incl_scan(mine);
      if (lane == 63) sh_scan[0][wave] = inc;
      lds_barrier();
      uint32_t tot;
      const uint32_t above = (uint32_t)nc - wave_offset<NW>(sh_scan[0], &tot) - inc;   // keys in bins above this thread's
      uint32_t a[BPT];
      a[BPT - 1] = above;
#pragma unroll
      for (int i = BPT - 1; i > 0; --i) a[i - 1] = a[i] + h[i];
#pragma unroll
      for (int i = 0; i < BPT; i += 4)
        *reinterpret_cast<uint4*>(&hist[BPT * tid + i]) = make_uint4(a[i] | h[i] << 16, a[i + 1] | h[i + 1] << 16,
                                                                     a[i + 2] | h[i + 2] << 16, a[i + 3] | h[i + 3] << 16);
      // the thread whose bins hold the rank publishes the bin and the keys above it
      const auto find = [&](uint32_t rank, uint32_t* out) {
        if (rank - above < mine) {   // (unsigned: above <= rank < above + mine)
          uint32_t at = 0, up = a[0];
#pragma unroll
          for (int i = 1; i < BPT; ++i) {
            at += rank < a[i - 1];
            up = rank < a[i - 1] ? a[i] : up;
          }
          out[0] = tid * BPT + at;
          out[1] = up;
        }
      };
      find((uint32_t)(np - 1), sh_sel);
      find((uint32_t)(k2 - 1), sh_sel + 2);
      uint32_t most = h[0];
#pragma unroll
      for (int i = 1; i < BPT; ++i) most = max(most, h[i]);
      // a bin of the retrieval zone that is long to put in order (or one just below it)
      if (above < (uint32_t)np && most > SEL_RUN) sh_sel[4] = 1u;
    }
    lds_barrier();
    C1 = __builtin_amdgcn_readfirstlane(sh_sel[0]);
    s1 = __builtin_amdgcn_readfirstlane(sh_sel[1]);
    C2 = __builtin_amdgcn_readfirstlane(sh_sel[2]);
    s2 = __builtin_amdgcn_readfirstlane(sh_sel[3]);
    // (the last bin holds everything above the window, the first ones everything below)
    if (__builtin_expect(!window || ((BYTES ? C1 : C2) >= SEL_BELOW && C1 < SEL_SPAN - 1), 1)) break;
    window = false;
    spread = 0u;
    clear_bins();
    if (tid == 0) sh_sel[4] = 0u;
    lds_barrier();
  }
  uint32_t T1, T2, g1, g2;   // g1, g2: keys strictly above T1 / T2
  if (window) {
    T1 = SEL_WINDOW + C1;
    T2 = SEL_WINDOW + C2;
    g1 = s1;
    g2 = s2;
    if (BYTES && __builtin_expect(C2 < SEL_BELOW, 0)) {   // of the keys below, by their upper bytes, then the lower ones of the rank's
      uint32_t* const byte = sh_rank;   // [2][256]
      static_assert(3 * NT >= 512, "room for them");
      for (int i = tid; i < 512; i += NT) byte[i] = 0u;
      lds_barrier();
      const auto count = [&](auto&& at) {
#pragma unroll
        for (int o = 0; o < EIGHTS; ++o)
          if (8 * o < nown) {
#pragma unroll
            for (int i = 8 * o; i < 8 * o + 8 && i < E; ++i)
              if (key_of(i) < SEL_WINDOW + SEL_BELOW) at(key_of(i));
          }
        lds_barrier();
      };
      // the bin of rank `rank` counted from the top, which becomes the rank in the bin
      const auto find = [&](const uint32_t* f, uint32_t& rank) {
        const uint4 x = *reinterpret_cast<const uint4*>(f + 252 - 4 * lane);   // lane l: bins 255 - 4 l to 252 - 4 l
        const uint32_t n = x.x + x.y + x.z + x.w, inc = ri_wave_incl_scan(n);
        const int l = __ffsll((long long)__ballot(inc > rank)) - 1;
        rank -= (uint32_t)__builtin_amdgcn_readlane((int)(inc - n), l);
        uint32_t bin = 255 - 4 * l;
        const uint32_t c[3] = {(uint32_t)__builtin_amdgcn_readlane((int)x.w, l), (uint32_t)__builtin_amdgcn_readlane((int)x.z, l),
                               (uint32_t)__builtin_amdgcn_readlane((int)x.y, l)};
        for (int i = 0; i < 3 && rank >= c[i]; ++i) { rank -= c[i]; --bin; }
        return bin;
      };
      uint32_t rank = (uint32_t)k2 - 1 - (hist[SEL_BELOW - 1] & 0xffffu);   // (keys above the last of the shared bins)
      count([&](uint32_t k) { atomicAdd(&byte[k >> 8], 1u); });
      const uint32_t upper = find(byte, rank);
      count([&](uint32_t k) { if (k >> 8 == upper) atomicAdd(&byte[256 + (k & 255)], 1u); });
      T2 = upper << 8 | find(byte + 256, rank);
      g2 = (uint32_t)k2 - 1 - rank;   // (rank: of the last key among those equal to T2)
    }
  } else {
#pragma unroll
    for (int o = 0; o < EIGHTS; ++o)
      if (8 * o < nown) {
#pragma unroll
        for (int i = 8 * o; i < 8 * o + 8 && i < E; ++i) {
          const uint32_t k = key_of(i), c = k >> SEL_SHIFT;
          if (c == C1 || c == C2) atomicAdd(&sh_fine[c == C1 ? 0 : 1][k & (FB - 1)], 1u);
        }
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
    uint32_t a1, a2;
    T1 = (C1 << SEL_SHIFT) | fine_bin(sh_fine[0], (uint32_t)(np - 1) - s1, a1);
    T2 = (C2 << SEL_SHIFT) | fine_bin(sh_fine[C1 == C2 ? 0 : 1], (uint32_t)(k2 - 1) - s2, a2);
    g1 = s1 + a1;
    g2 = s2 + a2;
  }

  // ---- one scan places the ties and the keys between the thresholds ----
  // Tied keys are taken in ascending id order: tie rank r at T1 belongs to the retrieval zone
  // while g1 + r < np, then to the estimation zone while g1 + r < k2; at T2 while g2 + r < k2.
  // The owned keys are classified once, two at a time and without branches, into bit masks (bit i = owned key i); the rare
  // cases (keys of the retrieval zone: np of nc; ties at a threshold) are then walked bit by bit.
  mask_t m_gt1 = 0, m_lt1 = 0, m_gt2 = 0, m_lt2 = 0;
  {
    const uint32_t t1 = T1 | T1 << 16, t2 = T2 | T2 << 16;
#pragma unroll
    for (int w = 0; w < KW; w += 8) {
      uint32_t gt1 = 0, lt1 = 0, gt2 = 0, lt2 = 0;   // bit 2 v: key 2 v, bit 16 + 2 v: key 2 v + 1
#pragma unroll
      for (int v = 0; v < 8 && w + v < KW; ++v) {
        const uint32_t k = kw[w + v];
        gt1 |= sel_above(k, t1) << (2 * v);
        lt1 |= sel_above(t1, k) << (2 * v);
        gt2 |= sel_above(k, t2) << (2 * v);
        lt2 |= sel_above(t2, k) << (2 * v);
      }
      const auto in_order = [&](uint32_t m) { return (mask_t)((m & 0x5555u) | m >> 15) << (2 * w); };
      m_gt1 |= in_order(gt1);
      m_lt1 |= in_order(lt1);
      m_gt2 |= in_order(gt2);
      m_lt2 |= in_order(lt2);
    }
  }
  const mask_t ok = nown >= (int)(8 * sizeof(mask_t)) ? ~(mask_t)0 : ((mask_t)1 << nown) - 1;
  const mask_t m_eq1 = ~(m_gt1 | m_lt1) & ok, m_eq2 = T2 == T1 ? 0 : ~(m_gt2 | m_lt2) & ok;
  m_gt1 &= ok;
  const mask_t m_mid = m_gt2 & ~m_gt1 & ~m_eq1 & ok;  // strictly between the thresholds: estimation zone
  const auto popc = [](mask_t m) { return (uint32_t)__popc((unsigned)m); };
  const auto lowest = [](mask_t m) { return __ffs((int)m) - 1; };
  uint32_t cnt[2] = {popc(m_eq1), popc(m_eq2) | popc(m_mid) << 16}, pre[2];   // (each at most nc <= 16384)
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    pre[k] = ri_wave_incl_scan(cnt[k]);
    if (lane == 63) sh_scan[k + 1][wave] = pre[k];
  }
  // owned key i (a register half chosen at run time: only the rare walks below need it)
  const auto key_at = [&](int i) {
    uint32_t w = 0;
#pragma unroll
    for (int v = 0; v < KW; ++v) w = ((i >> 1) == v) ? kw[v] : w;
    return (i & 1) ? (w >> 16) : (w & 0xffffu);
  };
  // keys above T1 take the places of their bin in whatever order they come
  for (mask_t m = m_gt1; m; m &= m - 1) {
    const int i = lowest(m);
    const uint32_t k = key_at(i);
    const uint32_t slot = atomicAdd(&hist[sel_bins(k, window) & 0xffffu], 1u) & 0xffffu;
    sh_ret[slot] = (k << 16) | (0xffffu - (uint32_t)(cbeg + i));
  }
  lds_barrier();
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    uint32_t tot;
    pre[k] += wave_offset<NW>(sh_scan[k + 1], &tot) - cnt[k];
  }
  const uint32_t r1 = pre[0], r2 = pre[1] & 0xffffu, mid_before = pre[1] >> 16;
  const uint32_t lo1 = (uint32_t)np - g1;                            // first tie rank of T1 in the est zone
  const uint32_t hi1r = (uint32_t)k2 > g1 ? (uint32_t)k2 - g1 : 0u;  // one past the last
  const uint32_t hi2r = (uint32_t)k2 > g2 ? (uint32_t)k2 - g2 : 0u;
  const uint32_t est_first = mid_before + (min(max(r1, lo1), hi1r) - lo1) + min(r2, hi2r);
  mask_t est_bits = m_mid;  // bit i: owned key i is in the estimation zone
  {
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
  // (the sizes and first rows are requested for the unsorted entries: they go to the entry's rank with it, or the loads behind
  // the sort find them near)
  uint32_t sz = 0;
  int32_t st = 0;
  if (!STAGED && in && P.cluster_size) {
    sz = (uint32_t)P.cluster_size[(size_t)g * nc + id_of(v)];
    if (P.cluster_start) st = P.cluster_start[(size_t)g * nc + id_of(v)];
  }
  if (KEEP) {   // (in front of the wait for them)
    uint32_t at = est_first;
    for (mask_t m = est_bits; m; m &= m - 1) K.est[at++] = cbeg + lowest(m);
  }
  const bool sorted = __builtin_amdgcn_readfirstlane(sh_sel[4]) != 0 || g1 - s1 > SEL_RUN;   // uniform
  int my_c;
  if (!sorted) {
    // An entry above T1 is in its bin's run of places already; its place there is the number of entries that come before it.
    // (Ties at T1 are in theirs.)
    int rank = tid;
    if (tid < (int)g1) {
      const uint32_t b = sel_bins(v >> 16, window) & 0xffffu, w = hist[b];
      const bool cut = !window && b == C1;   // (its keys above T1 only)
      const int end = cut ? (int)g1 : (int)(w & 0xffffu), start = cut ? (int)s1 : end - (int)(w >> 16);
      if (end - start > 1) {
        rank = start;
        for (int e = start; e < end; e += 4) {
          uint32_t o[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) o[u] = sh_ret[min(e + u, end - 1)];
#pragma unroll
          for (int u = 0; u < 4; ++u) rank += e + u < end && o[u] > v;
        }
      }
    }
    if (in) {
      sh_rank[rank] = v;
      if (!STAGED) {
        sh_rank[NT + rank] = sz;
        sh_rank[2 * NT + rank] = (uint32_t)st;
      }
    }
    lds_barrier();
    v = in ? sh_rank[tid] : 0u;
    my_c = id_of(v);
    if (!STAGED && in) {
      sz = sh_rank[NT + tid];
      st = (int32_t)sh_rank[2 * NT + tid];
    }
  } else {
    int n = 64;
    while (n < np) n <<= 1;
    block_sort_desc<LOGT>(v, n, hist);
    if (!STAGED) asm volatile("" : : "v"(sz), "v"(st));
    my_c = id_of(v);
    if (!STAGED && in && P.cluster_size) {
      sz = (uint32_t)P.cluster_size[(size_t)g * nc + my_c];
      if (P.cluster_start) st = P.cluster_start[(size_t)g * nc + my_c];
    }
  }
  if (STAGED && in && P.cluster_size) {
    sz = (uint32_t)sh_size[my_c];
    if (P.cluster_start) st = sh_row[my_c];
  }

  // ---- token layout of the retrieved clusters with the page cut-off ----
  uint32_t tok = 0;
  int nkeep = 0;
  uint32_t T_ret = 0, pages = 0;
  bool keep = false;
  if (P.cluster_size) {
    // (a division by what is not known when this is built takes forty instructions)
    const uint32_t up = sz + P.page - 1;
    const uint32_t pg = (P.page & (P.page - 1)) == 0 ? up >> __builtin_ctz(P.page) : up / P.page;
    uint32_t pg_pre = 0;
    if (wave * 64 < np) {   // uniform
      pg_pre = ri_wave_incl_scan(pg);
      tok = ri_wave_incl_scan(sz);
    }
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
    if (STORE) P.ret_ids[(size_t)g * np + tid] = my_c;
    else K.ids[tid] = my_c;
    if (STORE && P.cI) P.cI[(size_t)g * k2 + tid] = my_c;
  }
  if (STORE) {
    uint32_t at = est_first;
    for (mask_t m = est_bits; m; m &= m - 1, ++at) {
      const int c = cbeg + lowest(m);
      P.est_ids[(size_t)g * es + at] = c;
      if (P.cI) P.cI[(size_t)g * k2 + np + at] = c;
    }
  }
  if (!P.cluster_size) return in ? my_c : -1;
  if (in) {
    if (STORE) P.ret_tok_off[(size_t)g * (np + 1) + tid] = (int32_t)((tid < nkeep) ? tok : T_ret);
    if (STORE && P.ret_start) P.ret_start[(size_t)g * np + tid] = st;
    if (KEEP) {
      K.off[tid] = (int)((tid < nkeep) ? tok : T_ret);
      K.start[tid] = st;
    }
  }
  if (tid == 0) {
    if (KEEP) K.off[np] = (int)T_ret;
    int32_t* const meta = STORE ? P.meta + g * 4 : K.meta;
    if (STORE) P.ret_tok_off[(size_t)g * (np + 1) + np] = (int32_t)T_ret;
    meta[0] = nkeep;
    meta[1] = (int32_t)T_ret;
    meta[2] = (int32_t)pages;
    meta[3] = 0;
  }
  if (STORE && P.row_src && P.cluster_start && keep) {   // row table: each kept cluster writes the rows of its tokens
    int32_t* dst = P.row_src + (size_t)g * P.row_src_stride + tok;
    const int room = P.row_src_stride - (int)tok;
    for (int k = 0; k < (int)sz && k < room; ++k) dst[k] = st + k;
  }
  return in ? my_c : -1;
}

// Checks the arguments of ri_score_select and lays them down (select.hip).
int ri_prepare_select(SelectArgs* P, const void* q, const void* centroids, const uint8_t* mask,
                      const int32_t* cluster_size_i32, const int32_t* cluster_start, float* logits, void* dist, int64_t* cI,
                      int32_t* ret_ids, int32_t* est_ids, int32_t* ret_tok_off, int32_t* ret_start, int32_t* row_src,
                      int row_src_stride, int32_t* meta, int BG, int gs, int nc, int np, int es, int page, int max_pages,
                      float scale, void* workspace, size_t workspace_bytes);

// Scoring, and the scores' sums and keys if `keys` (select.hip)
int ri_launch_select_inputs(const SelectArgs& P, int BG, bool half, bool keys, hipStream_t s);

// Scoring, selection and the block cache's look-up of the selected clusters (lru.hip); `taken`: false, and nothing launched,
// where that is not worth a launch of its own kind.
int ri_launch_select_access(const SelectArgs& P, const ri_lru_t& lru, int BG, bool half, bool* taken, hipStream_t s);
