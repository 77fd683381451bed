// Device code of the attention that attend.hip and step.hip share (gfx950): the per-wave online-softmax state, the
// update for one chunk of 16 rows (softmax bookkeeping, P·V on the matrix cores), the coherent load of split partials, and
// a group's attention by one workgroup of it.
#pragma once
#include <math.h>

#include "ri_common.h"

// Softmax bookkeeping is spread over the four 16-lane groups of a wave: group h keeps
// NH = GS_PAD/4 heads (the MFMA hands every group four heads; with GS_PAD = 4 all groups see the
// same four, so each keeps one).  ri_head_reg(h) is the first accumulator register group h keeps,
// ri_head_of(h, i) the head held in kept slot i.
template <int GS_PAD>
__device__ __forceinline__ int ri_head_reg(int h) {
  return GS_PAD == 4 ? h : (GS_PAD == 8 ? (h >> 1) * 2 : 0);
}
template <int GS_PAD>
__device__ __forceinline__ int ri_head_of(int h, int i) {
  return (4 * h + ri_head_reg<GS_PAD>(h) + i) % GS_PAD;
}

typedef short bf16x4s_t __attribute__((ext_vector_type(4)));

#define ATT_VT_STRIDE 144  // LDS row stride of the 16 x 128 value tile in bf16 elements (288 bytes)

template <int GS_PAD>
struct WaveState {
  float m[GS_PAD / 4];
  float l[GS_PAD / 4];
  // P·V accumulators in MFMA 16x16 layout: acc[dt][i] of lane l = head 4*(l/16)+i, dim 16*dt + l%16
  f32x4_t acc[8];
};

// probability -> the 16-bit element type of the P.V operands (hardware conversion, round to nearest even)
template <bool HALF>
__device__ __forceinline__ uint16_t ri_p_to_e16(float x) {
  if (HALF) return __builtin_bit_cast(uint16_t, (_Float16)x);
  const __bf16 b = (__bf16)x;
  return __builtin_bit_cast(uint16_t, b);
}

// maximum / sum over the 16 lanes of a row, in every lane (register moves within the row, no LDS crossbar)
__device__ __forceinline__ float ri_row_max(float x) {
  x = fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xf, 0xf, true)));   // quad_perm 1,0,3,2
  x = fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xf, 0xf, true)));   // quad_perm 2,3,0,1
  x = fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x141, 0xf, 0xf, true)));  // half row mirrored
  return fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x140, 0xf, 0xf, true)));  // row mirrored
}
__device__ __forceinline__ float ri_row_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xf, 0xf, true));
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xf, 0xf, true));
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x141, 0xf, 0xf, true));
  return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x140, 0xf, 0xf, true));
}

// The value rows h, h+4, h+8, h+12 of a chunk (dims 8n..8n+7, as loaded) -> row-major 16 x 128 tile in LDS.
__device__ __forceinline__ void chunk_values(const uint4 v[4], uint16_t* vt, int lane) {
  const int n = lane & 15, h = lane >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) *reinterpret_cast<uint4*>(vt + (h + 4 * i) * ATT_VT_STRIDE + 8 * n) = v[i];
}

// One chunk of 16 rows whose value tile is in LDS.
//   sv[NH]  scores of the heads this lane keeps for row n = lane%16 (lane group h = lane/16)
// Softmax bookkeeping in fp32 per lane; P goes to LDS as bf16 [head][row]; P·V = 8 MFMA 16x16x16 whose B
// operands come from LDS transpose reads
// (ds_read_b64_tr_b16: lane l of a 16-lane group receives element l%4 of the 8-byte pieces
// addressed by lanes l/4, l/4+4, l/4+8, l/4+12 — four consecutive rows of one column).
template <int GS_PAD, bool HALF>
__device__ __forceinline__ void chunk_update(WaveState<GS_PAD>& st, const float* sv, bool valid, float w,
                                             const uint16_t* vt, uint16_t* pb, float* al_sh, int lane) {
  constexpr int NH = GS_PAD / 4;
  const int n = lane & 15, h = lane >> 4;
  float al[NH];
  bool rescale = false;
#pragma unroll
  for (int i = 0; i < NH; ++i) {
    const float s = valid ? sv[i] : -INFINITY;
    const float mn = fmaxf(st.m[i], ri_row_max(s));
    // No finite score so far (no valid row, a head that does not exist, keys with infinite elements): relative to 0 such
    // scores weigh exp(-inf) = 0, as the rows that are not valid always do; relative to -inf they would weigh NaN.
    const bool none = mn == -INFINITY;
    al[i] = none ? 1.f : __expf(st.m[i] - mn);
    const float p = __expf(s - (none ? 0.f : mn));
    rescale |= (al[i] != 1.f);
    st.l[i] = st.l[i] * al[i] + w * p;
    st.m[i] = mn;
    pb[ri_head_of<GS_PAD>(h, i) * 16 + n] = ri_p_to_e16<HALF>(p);
  }
  // the running maximum rarely moves after the first chunks: rescale only when some head's did
  const bool any_rescale = __builtin_amdgcn_ballot_w64(rescale) != 0;
  if (any_rescale && n == 0) {
#pragma unroll
    for (int i = 0; i < NH; ++i) al_sh[ri_head_of<GS_PAD>(h, i)] = al[i];
  }
  ri_wave_sync();
  if (any_rescale) {
    const float4 a4 = *reinterpret_cast<const float4*>(al_sh + 4 * h);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      st.acc[dt][0] *= a4.x; st.acc[dt][1] *= a4.y; st.acc[dt][2] *= a4.z; st.acc[dt][3] *= a4.w;
    }
  }
  // A operand: P[head n][rows 4h..4h+3]
  const bf16x4s_t pa = *reinterpret_cast<const bf16x4s_t*>(pb + n * 16 + 4 * h);
  const uint16_t* vsrc = vt + (4 * h + (n >> 2)) * ATT_VT_STRIDE + 4 * (n & 3);
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) {
    const bf16x4s_t vb = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (bf16x4s_t __attribute__((address_space(3)))*)(vsrc + 16 * dt));
    if (HALF)
      st.acc[dt] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4_t, pa), __builtin_bit_cast(f16x4_t, vb),
                                                         st.acc[dt], 0, 0, 0);
    else
      st.acc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pa, vb, st.acc[dt], 0, 0, 0);
  }
  ri_wave_sync();   // the tile and P are rewritten by the next chunk
}

// The partials were written by other workgroups of the same launch; they are read with
// device-scope loads (which go past this compute unit's non-coherent cache lines) instead of
// an acquire fence that would drop the whole cache.
__device__ __forceinline__ float2 ri_ld_partial(const float* p) {
  const uint64_t v = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  return make_float2(__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32)));
}

#define ATT_WAVES 8                // waves of a workgroup
#define ATT_FLAG_A 0x40000000     // descriptor bit: row lives in region A
#define ATT_SKIP (int)0x80000000  // descriptor bit (the sign): the row is read but not attended

struct AttendParams {
  const uint16_t* q;  // [BG, gs, 128]
  // region A: rows [0, lenA) at kA/vA + (g*strideA + row)*128
  const uint16_t* kA;
  const uint16_t* vA;
  int64_t strideA;
  int lenA;
  const int32_t* lenA_ptr;  // when given: lenA is read here at launch time (clamped to [0, strideA])
  // region B: rows [0, lenB(g)) at kB/vB + (g*strideB + src(row))*128,
  // src(row) = row_src ? row_src[g*rs_stride + row] : row
  const uint16_t* kB;
  const uint16_t* vB;
  int64_t strideB;
  const int32_t* row_src;
  int rs_stride;
  // with a row table: only rows whose source row lies in [src_lo, src_hi), src_lo >= 0, are attended; the others are
  // skipped like padding rows (a second launch takes them, merging this one's result as its previous one).  Their entries
  // may be anything: row 0 is read in their place.
  int src_lo, src_hi;
  // or, without a row table: rank r of np clusters covers rows [ret_off[r], ret_off[r+1]) of region B,
  // stored contiguously from row ret_start[r] (ret_off has np + 1 entries, constant from the last kept rank on)
  const int32_t* ret_off;
  const int32_t* ret_start;
  int np;
  const int32_t* lenB_ptr;  // lenB(g) = lenB_ptr ? lenB_ptr[g*lenB_ptr_stride] : lenB_const
  int lenB_ptr_stride;
  int lenB_const;
  const uint16_t* weightB;  // [BG, weight_stride] bf16 per region-B row, or null
  int weight_stride;
  // estimation rows
  const int32_t* est_ids;     // [BG, es]
  const float* logits;        // [BG, gs, nc] scores of the estimation rows, or null:
  const uint16_t* est_cent;   // [BG, nc, 128] then the scores are computed here from the centroid rows
  const uint16_t* value_sum;  // [BG, nc, 128]
  const uint16_t* csize;      // [BG, nc] bf16
  int nc;
  int es;
  // partials and the arrival counters (zero between launches)
  float* part_ml;   // [BG, S, GS_PAD, 2]
  float* part_acc;  // [BG, S, GS_PAD, 128]
  int* counters;    // [BG, ATT_WAVES] pitch words apart (attend_counter_pitch)
  int pitch;
  int S;     // workgroups per group
  int W_kv;  // of the group's S * ATT_WAVES waves the first W_kv take key/value rows, the others estimation rows
  int W_one; // the same of one workgroup's waves, if it takes the whole group
  uint32_t inv_kv, inv_es;           // ATT_INVERSE of the waves of either kind
  uint32_t inv_kv_one, inv_es_one;   // and of one workgroup's
  int gs;
  float scale;
  // epilogue
  const uint16_t* prev_out;  // [BG, gs, 128] or null
  const float* prev_lse;     // [BG, gs] or null
  uint16_t* out;             // [BG, gs, 128]
  float* lse_out;            // [BG, gs] or null
  int32_t* valid_lengths;    // [BG] or null: lenA + lenB(g)
};

// Rows of a wave: the group's `total` rows are cut into `nwaves` runs of a multiple of 16 rows.  inv: ATT_INVERSE(nwaves), made by
// the host, because a division by what is not known when this is built is thirty instructions in front of a wave's first load.
#define ATT_INVERSE(nwaves) ((uint32_t)((0x80000000u + (uint32_t)(nwaves) - 1u) / (uint32_t)(nwaves)))
__device__ __forceinline__ void wave_rows(int total, int nwaves, uint32_t inv, int wid, int* r0, int* r1) {
  const uint32_t n = ((uint32_t)(total + 15) >> 4) + nwaves - 1;   // (exact below 2^31 / nwaves, of which there are 512)
  const int rpw = 16 * (int)(n < (1u << 22) ? (uint32_t)(((uint64_t)n * inv) >> 31) : n / (uint32_t)nwaves);
  *r0 = min(total, wid * rpw);
  *r1 = min(total, *r0 + rpw);
}

// The output row of head j: A / L merged with an earlier part (its output po, its log-sum-exp pl) under the maximum M.
// Lane l holds dims 2l and 2l + 1.
template <bool HALF>
__device__ __forceinline__ void write_head(const AttendParams& P, int g, int j, float M, float L, float A0, float A1) {
  const int lane = threadIdx.x & 63;
  const size_t o = (size_t)g * P.gs + j, at = o * RI_DIM + 2 * lane;
  if (P.prev_lse) {
    const float pl = P.prev_lse[o];
    if (pl != -INFINITY) {  // an empty earlier part carries no weight, whatever its output holds
      float p0, p1;
      ri_unpack2<HALF>(*reinterpret_cast<const uint32_t*>(P.prev_out + at), p0, p1);
      const float M2 = fmaxf(M, pl);
      const float f = M == -INFINITY ? 0.f : __expf(M - M2), fp = __expf(pl - M2);
      L = L * f + fp;
      A0 = A0 * f + fp * p0;
      A1 = A1 * f + fp * p1;
      M = M2;
    }
  }
  // nothing attended at all (an empty part): zeros and a log-sum-exp of -inf, not 0/0
  const bool any = L > 0.f;
  *reinterpret_cast<uint32_t*>(P.out + at) =
      (uint32_t)ri_f32_to_e16<HALF>(any ? A0 / L : 0.f) | ((uint32_t)ri_f32_to_e16<HALF>(any ? A1 / L : 0.f) << 16);
  if (lane == 0 && P.lse_out) P.lse_out[o] = M + __logf(L);
}

// The eight waves share the heads when they merge: wave w takes heads w, w + ATT_WAVES, ..., a lane two dims.  (With up to four
// heads, two waves to a head and a dim per lane would be twice the stores, arrivals and requests: eight captured layers of 16
// groups of 4 heads, 1024 clusters 136.0 us instead of 134.3, the five operators over 32 groups 63.1 instead of 62.6.)
template <int GS_PAD>
constexpr int ATT_HEADS_OF_WAVE = (GS_PAD + ATT_WAVES - 1) / ATT_WAVES;

// Merges a wave's share of the S split partials of group g (and the optional previous result) and writes the output: lanes
// first cover the splits (statistics), then two dims each.
// The partials come from the memory side, where a load takes about a microsecond and one compute unit gets 20 KB per
// microsecond: a wave requests the statistics of its heads and then eight splits of them at a time.  (One head after the other:
// 13600 cycles for 16 heads over 3 splits.  Sixteen splits on their way: their registers and conditions cost more than the round trips,
// the attention by itself 1 group of 16 heads, 100000 rows 30.9 -> 32.8 us, 4 of 12, 24000 19.4 -> 20.3, 8 of 8, 6000 10.5 -> 10.9.)
template <int GS_PAD, bool HALF>
__device__ __forceinline__ void combine_share(const AttendParams& P, int g, int wave) {
  constexpr int HPW = ATT_HEADS_OF_WAVE<GS_PAD>, U = 8;   // U: splits requested at a time
  const int gs = P.gs, S = P.S;
  const int lane = threadIdx.x & 63;
  int head[HPW];
#pragma unroll
  for (int k = 0; k < HPW; ++k) head[k] = min(wave + k * ATT_WAVES, gs - 1);
  const float* ml = P.part_ml + (size_t)g * S * GS_PAD * 2;
  const float* pa = P.part_acc + (size_t)g * S * GS_PAD * RI_DIM + 2 * lane;
  float2 ms[HPW];
#pragma unroll
  for (int k = 0; k < HPW; ++k) ms[k] = ri_ld_partial(ml + ((size_t)min(lane, S - 1) * GS_PAD + head[k]) * 2);
  float2 a[U][HPW];
  const auto request = [&](int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < HPW; ++k) a[u][k] = ri_ld_partial(pa + ((size_t)min(s0 + u, S - 1) * GS_PAD + head[k]) * RI_DIM);
  };
  request(0);
  float f[HPW], M[HPW], L[HPW], A0[HPW], A1[HPW];
#pragma unroll
  for (int k = 0; k < HPW; ++k) {
    const float m = lane < S ? ms[k].x : -INFINITY;
    M[k] = ri_row_max(m);
    M[k] = ri_xor_max<32>(ri_xor_max<16>(M[k]));
    f[k] = m == -INFINITY ? 0.f : __expf(m - M[k]);
    L[k] = ri_row_sum(ms[k].y * f[k]);
    L[k] = ri_xor_sum<32>(ri_xor_sum<16>(L[k]));
    A0[k] = A1[k] = 0.f;
  }
  for (int s0 = 0; s0 < S; s0 += U) {   // (a split past the last has no weight: f of its lane is 0)
    if (s0) request(s0);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < HPW; ++k) {
        const float fs = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f[k]), (s0 + u) & 63));
        const float w = s0 + u < S ? fs : 0.f;
        A0[k] += a[u][k].x * w;
        A1[k] += a[u][k].y * w;
      }
  }
#pragma unroll
  for (int k = 0; k < HPW; ++k)
    if (wave + k * ATT_WAVES < gs) write_head<HALF>(P, g, head[k], M[k], L[k], A0[k], A1[k]);
}

#define ATT_DESC_MAX 64  // rows of one wave whose descriptors are staged in LDS at a time (32 and 128 measured slower)

// A wave's LDS: value tile, probabilities, rescale factors, row descriptors and weights.
struct WaveLds {
  uint16_t* vt;
  uint16_t* pb;
  float* al;
  int* dsc;
  float* w;
};

// Rows [r0, r1) of one wave in batches of 64.  `stage(row, weight)` returns where the row lives (a descriptor) and may set
// the row's weight; `load(d, dv, k, v)` requests the score operand and the four value rows of a chunk, `score` turns
// the operand into the scores of this lane's heads.
// The next chunk is requested as soon as the registers of this one are free (keys after their products, values after
// they are in LDS), so that its loads run under the softmax and the P.V products without a second set of registers.
template <int GS_PAD, bool HALF, typename K, typename Stage, typename Load, typename Score>
__device__ __forceinline__ void attend_rows(WaveState<GS_PAD>& st, const WaveLds& sh, int r0, int r1, Stage&& stage,
                                            Load&& load, Score&& score) {
  const int lane = threadIdx.x & 63;
  const int n = lane & 15, h = lane >> 4;
  for (int s0 = r0; s0 < r1; s0 += ATT_DESC_MAX) {
    const int s1 = min(r1, s0 + ATT_DESC_MAX);
    {
      float w = 1.f;
      // (a row past the last repeats it, marked: every load has a valid address and no load sits under a condition)
      const int d = stage(min(s0 + lane, s1 - 1), w);
      sh.dsc[lane] = s0 + lane < s1 ? d : d | ATT_SKIP;
      sh.w[lane] = w;
    }
    ri_wave_sync();
    const int nch = (s1 - s0 + 15) >> 4;
    K k;
    uint4 v[4];
    int dk, dv[4];
    const auto issue = [&](int j) {
      dk = sh.dsc[j * 16 + n];
#pragma unroll
      for (int i = 0; i < 4; ++i) dv[i] = sh.dsc[j * 16 + h + 4 * i];
      load(dk & ~ATT_SKIP, dv, k, v);
    };
    issue(0);
    for (int j = 0; j < nch; ++j) {
      const bool valid = dk >= 0;
      float sv[GS_PAD / 4], w = sh.w[j * 16 + n];
      score(k, sv, w);
      if (__builtin_amdgcn_ballot_w64(valid) != ~0ull) {   // rows that are not attended must not bring NaN into P.V
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (dv[i] < 0) v[i] = ri_zero16();
      }
      chunk_values(v, sh.vt, lane);
      if (j + 1 < nch) issue(j + 1);
      chunk_update<GS_PAD, HALF>(st, sv, valid, w, sh.vt, sh.pb, sh.al, lane);
    }
  }
}

// The eight waves of a workgroup merge in LDS, so a group split over S workgroups hands S partials to whichever waves come last.
// The rank tables of the retrieval zone (np + 1 token offsets, np first rows) live in dynamic LDS, sized by
// the launch, so that any number of probes the selection accepts can be attended.
// HALF: q, K, V, value sums, cluster sizes, weights and outputs are IEEE half instead of bfloat16.
// KEPT: the workgroup has just made the selection, whose tables and ids are in LDS (K), from KEPT_LOGITS on the logits too, and
// has laid down what att_clear and att_put_query do.  KEPT_ALL: it has the whole group.
enum { KEPT_NONE, KEPT_TABLES, KEPT_LOGITS, KEPT_ALL };
struct AttendKept {
  const float* logits;   // [nc][GS_PAD]
  const int* est;        // [es]
  int* off;              // [np + 1]
  int* start;            // [np]
  int lenA;              // the steady zone's rows
};

// The waves' value tiles.  (Of a workgroup that makes the selection first: what that lays in them is dead by then.)
__device__ __forceinline__ uint16_t (*att_tiles())[16 * ATT_VT_STRIDE] {
  __shared__ __attribute__((aligned(16))) uint16_t sh_vt[ATT_WAVES][16 * ATT_VT_STRIDE];
  static_assert(__alignof__(sh_vt) == 16, "pieces of 16 bytes");
  return sh_vt;
}

// What else a workgroup lays down in LDS before its rows: probabilities (of heads that do not exist they stay zero) and factors
// (theirs must not scale by garbage), a wave's own, and the query, read again per chunk so that the registers go to the loads.
template <int GS_PAD>
struct AttendLds {
  __attribute__((aligned(16))) uint16_t pb[ATT_WAVES][16 * 16];
  __attribute__((aligned(16))) uint16_t q[GS_PAD][RI_DIM];
  float al[ATT_WAVES][16];
};
template <int GS_PAD>
__device__ __forceinline__ AttendLds<GS_PAD>& att_lds() {
  __shared__ __attribute__((aligned(16))) AttendLds<GS_PAD> sh;
  return sh;
}
template <int GS_PAD>
__device__ __forceinline__ void att_clear() {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wave >= ATT_WAVES) return;
  AttendLds<GS_PAD>& sh = att_lds<GS_PAD>();
  reinterpret_cast<uint2*>(sh.pb[wave])[lane] = make_uint2(0u, 0u);
  if (lane < 16) sh.al[wave][lane] = 1.f;
}
// row m of the MFMA holds head m % GS_PAD, zero if >= gs
template <int GS_PAD>
__device__ __forceinline__ void att_put_query(uint4 piece_of, int gs) {
  static_assert(GS_PAD * (RI_DIM / 8) <= 64 * ATT_WAVES, "one piece of the query per thread");
  const int head = threadIdx.x / (RI_DIM / 8), piece = threadIdx.x % (RI_DIM / 8);
  if (head < GS_PAD) *reinterpret_cast<uint4*>(&att_lds<GS_PAD>().q[head][piece * 8]) = head < gs ? piece_of : ri_zero16();
}

// piece threadIdx.x % 16 of the query of head threadIdx.x / 16
__device__ __forceinline__ uint4 att_query_piece(const AttendParams& P, int g) {
  const int head = threadIdx.x / (RI_DIM / 8), piece = threadIdx.x % (RI_DIM / 8);
  return ri_ld16(P.q + ((size_t)g * P.gs + min(head, P.gs - 1)) * RI_DIM + piece * 8);
}
// the steady zone's rows (a vector load: the wait for a scalar one is a wait for every access to LDS as well)
__device__ __forceinline__ int att_steady_rows(const AttendParams& P) {
  int none = 0;
  asm("" : "+v"(none));
  const int32_t* const at = P.lenA_ptr ? P.lenA_ptr : reinterpret_cast<const int32_t*>(P.q);   // (any valid place)
  const int there = at[none];
  return P.lenA_ptr ? min(max(there, 0), (int)P.strideA) : P.lenA;
}

// The last of n ranks whose first row off[rank] is <= row (ranks of empty clusters share a first row with the next rank, which
// is the one found); off[0] is 0.  For whole waves, whose rows ascend with the lane and are at most a batch apart: the wave
// looks for the first one's rank together, 64 ranks per read, and counts on from there, the few ranks that begin behind it and
// not behind the last row.  (Every lane by bisection took eight reads one after the other, 2000 .. 2500 cycles of each
// wave's chain for 150 .. 300 ranks.)
__device__ __forceinline__ int rank_of(const int* off, int n, int row) {
  const int lane = threadIdx.x & 63;
  const int first = __builtin_amdgcn_readfirstlane(row), last = __builtin_amdgcn_readlane(row, 63);
  int base = 0, span = n;   // uniform: off[base] <= first < off[base + span]
  while (span > 64) {
    const int step = (span + 63) >> 6, at = lane * step;
    const uint64_t below = __builtin_amdgcn_ballot_w64(at < span && off[base + min(at, span - 1)] <= first);
    const int found = (__builtin_popcountll(below) - 1) * step;
    base += found;
    span = min(step, span - found);
  }
  int rank = base - 1;
  for (;;) {   // uniform: 64 ranks from base on, until one begins behind the last row
    const int o = base + lane < n ? off[base + lane] : 0x7fffffff;
    const uint64_t here = __builtin_amdgcn_ballot_w64(o <= last);
    for (uint64_t m = here; m; m &= m - 1) rank += __builtin_amdgcn_readlane(o, __builtin_ctzll(m)) <= row;
    if (~here) return rank;
    base += 64;
  }
}

// The waves' numerators for the merge where they do not fit the wave's own value tile (see attend_group): free until then.
template <int GS_PAD>
__device__ __forceinline__ float* att_numerators() {
  constexpr bool OWN = GS_PAD * RI_DIM * sizeof(float) > 16 * ATT_VT_STRIDE * sizeof(uint16_t);
  __shared__ __attribute__((aligned(16))) float sh_acc[OWN ? ATT_WAVES : 1][OWN ? GS_PAD : 1][RI_DIM];
  static_assert(__alignof__(sh_acc) == 16, "read two dims at a time");
  return &sh_acc[0][0][0];
}

template <int GS_PAD, bool HALF, int KEPT>
__device__ __forceinline__ void attend_group(const AttendParams& P, const int g, const int split, const AttendKept& K) {
  constexpr int NW = ATT_WAVES;
  constexpr int NH = GS_PAD / 4;
  constexpr int NT = 64 * NW;
  uint16_t (*const sh_vt)[16 * ATT_VT_STRIDE] = att_tiles();
  auto& sh_pb = att_lds<GS_PAD>().pb;
  auto& sh_al = att_lds<GS_PAD>().al;
  auto& sh_q = att_lds<GS_PAD>().q;
  __shared__ float sh_m[NW][GS_PAD];
  __shared__ float sh_l[NW][GS_PAD];
  // the waves' numerators for the merge: up to eight heads they are laid over the wave's own value tile (dead once its
  // rows are done), which keeps a workgroup at 48 KB of LDS, so that the two its registers leave room for fit a compute
  // unit (sixteen heads: 116 KB, one workgroup)
  constexpr bool ACC_OVER_VT = GS_PAD * RI_DIM * sizeof(float) <= 16 * ATT_VT_STRIDE * sizeof(uint16_t);
  auto acc_of = [&](int w) -> float* {
    return ACC_OVER_VT ? reinterpret_cast<float*>(sh_vt[w]) : att_numerators<GS_PAD>() + (size_t)w * GS_PAD * RI_DIM;
  };
  __shared__ int sh_desc[NW][ATT_DESC_MAX];
  __shared__ float sh_w[NW][ATT_DESC_MAX];
  extern __shared__ __attribute__((aligned(16))) int sh_tab[];
  int* const sh_roff = KEPT ? K.off : sh_tab;                // [np + 1]
  int* const sh_rst = KEPT ? K.start : sh_tab + P.np + 1;    // [np]

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, h = lane >> 4;
  const int gs = P.gs, S = KEPT == KEPT_ALL ? 1 : P.S;

  WaveState<GS_PAD> st;
#pragma unroll
  for (int i = 0; i < NH; ++i) { st.m[i] = -INFINITY; st.l[i] = 0.f; }
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) st.acc[dt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

  const WaveLds sh = {sh_vt[wave], sh_pb[wave], sh_al[wave], sh_desc[wave], sh_w[wave]};
  if (!KEPT) att_clear<GS_PAD>();
  const int lenB = KEPT ? K.off[P.np] : P.lenB_ptr ? P.lenB_ptr[(size_t)g * P.lenB_ptr_stride] : P.lenB_const;
  // (by itself the attention asks for the zone's length only where there is one to ask for: asked for always it is a round trip in
  // front of its rows, 11.6 instead of 11.3 us of 32 groups of 4 heads, 1900 rows)
  const int lenA = __builtin_amdgcn_readfirstlane(KEPT ? K.lenA : P.lenA_ptr ? min(max(P.lenA_ptr[0], 0), (int)P.strideA) : P.lenA);

  const int wid = split * NW + wave;            // wave of the group
  const bool kv_wave = wid < P.W_kv;
  const bool kv_wg = split * NW < P.W_kv;       // the workgroup has waves with key/value rows
  const int W_es = S * NW - P.W_kv;

  // ---------------- prologue: query and rank tables to LDS ----------------
  if (!KEPT && (kv_wg || P.est_cent)) {
    const bool tab = kv_wg && P.ret_off != nullptr;
    // every global load of the prologue is requested before the first of them is consumed
    // (up to 1023 probes the table entries pass through registers, TAB_U per thread; longer tables are
    // staged by a plain loop after the query)
    constexpr int TAB_U = 1024 / NT;
    const bool tab_fast = tab && P.np < 1024;
    int t_off[TAB_U], t_st[TAB_U];
    if (tab_fast) {
#pragma unroll
      for (int u = 0; u < TAB_U; ++u) {
        const int i = threadIdx.x + u * NT;
        t_off[u] = P.ret_off[(size_t)g * (P.np + 1) + min(i, P.np)];
        t_st[u] = P.ret_start[(size_t)g * P.np + min(i, P.np - 1)];
      }
    }
    att_put_query<GS_PAD>(att_query_piece(P, g), gs);
    if (tab_fast) {
#pragma unroll
      for (int u = 0; u < TAB_U; ++u) {
        const int i = threadIdx.x + u * NT;
        if (i <= P.np) sh_roff[i] = t_off[u];
        if (i < P.np) sh_rst[i] = t_st[u];
      }
    } else if (tab) {
      for (int i = threadIdx.x; i <= P.np; i += NT) {
        sh_roff[i] = P.ret_off[(size_t)g * (P.np + 1) + i];
        if (i < P.np) sh_rst[i] = P.ret_start[(size_t)g * P.np + i];
      }
    }
    __syncthreads();
  }

  if (kv_wave || (!KEPT && P.est_cent)) {
    // ---------------- rows with keys ----------------
    // Estimation rows whose scores are not handed in are key/value rows of their own: key = centroid,
    // value = value sum, weight = cluster size, located through the id list.
    const bool est = !kv_wave;
    int r0, r1;
    if (est) wave_rows(P.es, W_es, P.inv_es, wid - P.W_kv, &r0, &r1);
    else wave_rows(lenA + lenB, P.W_kv, P.inv_kv, wid, &r0, &r1);
    const uint16_t* qrow = &sh_q[n % GS_PAD][h * 8];
    const uint16_t* kA = P.kA + (size_t)g * P.strideA * RI_DIM;
    const uint16_t* vA = P.vA + (size_t)g * P.strideA * RI_DIM;
    const uint16_t* kB = est ? P.est_cent + (size_t)g * P.nc * RI_DIM : P.kB + (size_t)g * P.strideB * RI_DIM;
    const uint16_t* vB = est ? P.value_sum + (size_t)g * P.nc * RI_DIM : P.vB + (size_t)g * P.strideB * RI_DIM;
    const int32_t* rs = est ? P.est_ids + (size_t)g * P.es
                            : (P.row_src ? P.row_src + (size_t)g * P.rs_stride : nullptr);
    const uint16_t* wB = (!est && P.weightB) ? P.weightB + (size_t)g * P.weight_stride : nullptr;
    const uint16_t* wsrc = est ? P.csize + (size_t)g * P.nc : nullptr;  // weight by source row
    const int r_first = ri_head_reg<GS_PAD>(h);
    const int lead = est ? 0 : lenA;
    struct Keys { uint4 k[4]; };
    attend_rows<GS_PAD, HALF, Keys>(
        st, sh, r0, r1,
        [&](int row, float& w) {
          int d;
          if (KEPT || (!est && P.ret_off)) {
            if (__builtin_amdgcn_readlane(row, 63) < lead) return row | ATT_FLAG_A;   // (the batch's last row)
            const int rb = max(row - lead, 0), rank = rank_of(sh_roff, P.np, rb);
            d = sh_rst[rank] + rb - sh_roff[rank];
            return row < lead ? row | ATT_FLAG_A : d;   // (no weights with rank tables)
          }
          if (row < lead) return row | ATT_FLAG_A;
          const int rb = row - lead;
          d = rs ? rs[rb] : rb;
          if (!est && P.row_src && (d < P.src_lo || d >= P.src_hi)) d = ATT_SKIP;   // row 0, not attended
          if (wB) w = ri_e16_to_f32<HALF>(wB[rb]);
          if (wsrc) w = ri_e16_to_f32<HALF>(wsrc[d]);
          return d;
        },
        [&](int dk, const int* dv, Keys& k, uint4* v) {
          const uint16_t* kp = ((dk & ATT_FLAG_A) ? kA : kB) + (size_t)(dk & ~ATT_FLAG_A) * RI_DIM + h * 8;
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) k.k[kk] = ri_ld16(kp + kk * 32);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int d = dv[i] & ~ATT_SKIP;
            v[i] = ri_ld16(((d & ATT_FLAG_A) ? vA : vB) + (size_t)(d & ~ATT_FLAG_A) * RI_DIM + n * 8);
          }
        },
        [&](const Keys& k, float* sv, float&) {
          f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) {
            const uint4 qv = *reinterpret_cast<const uint4*>(qrow + kk * 32);
            acc = HALF ? __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, qv),
                                                                __builtin_bit_cast(f16x8_t, k.k[kk]), acc, 0, 0, 0)
                       : __builtin_amdgcn_mfma_f32_16x16x32_bf16(ri_as_bf16x8(qv), ri_as_bf16x8(k.k[kk]), acc, 0, 0, 0);
          }
#pragma unroll
          for (int i = 0; i < NH; ++i) {
            float x;
            if (GS_PAD == 16) {
              x = acc[i];
            } else {  // register r_first + i without dynamic indexing
              const int r = r_first + i;
              x = r == 0 ? acc[0] : (r == 1 ? acc[1] : (r == 2 ? acc[2] : acc[3]));
            }
            sv[i] = x * P.scale;
          }
        });
  } else {
    // ---------------- estimation rows with their logits at hand ----------------
    int r0, r1;
    wave_rows(P.es, W_es, P.inv_es, wid - P.W_kv, &r0, &r1);
    const int32_t* ids = P.est_ids + (size_t)g * P.es;
    const uint16_t* vs = P.value_sum + (size_t)g * P.nc * RI_DIM;
    const uint16_t* cs = P.csize + (size_t)g * P.nc;
    const float* lg = P.logits + (size_t)g * gs * P.nc;
    struct Logits { float x[NH]; uint16_t size; };
    attend_rows<GS_PAD, HALF, Logits>(
        st, sh, r0, r1, [&](int row, float&) { return KEPT ? K.est[row] : ids[row]; },
        [&](int dk, const int* dv, Logits& k, uint4* v) {
#pragma unroll
          for (int i = 0; i < NH; ++i) {
            const int head = min(ri_head_of<GS_PAD>(h, i), gs - 1);
            k.x[i] = KEPT >= KEPT_LOGITS ? K.logits[dk * GS_PAD + head] : lg[(size_t)head * P.nc + dk];
          }
          k.size = cs[dk];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = ri_ld16(vs + (size_t)(dv[i] & ~ATT_SKIP) * RI_DIM + n * 8);
        },
        [&](const Logits& k, float* sv, float& w) {
#pragma unroll
          for (int i = 0; i < NH; ++i) sv[i] = ri_head_of<GS_PAD>(h, i) < gs ? k.x[i] : -INFINITY;
          w = ri_e16_to_f32<HALF>(k.size);
        });
  }

  // ---------------- wave partial -> LDS ----------------
#pragma unroll
  for (int i = 0; i < NH; ++i) {
    const float l = ri_row_sum(st.l[i]);
    if (n == 0) {
      sh_m[wave][ri_head_of<GS_PAD>(h, i)] = st.m[i];
      sh_l[wave][ri_head_of<GS_PAD>(h, i)] = l;
    }
  }
  // accumulators are already summed over rows: lane (n, h) register i holds head 4h+i, dim 16*dt+n
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int head = 4 * h + i;
    if (head < GS_PAD) {
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) acc_of(wave)[head * RI_DIM + 16 * dt + n] = st.acc[dt][i];
    }
  }
  __syncthreads();

  // ---------------- merge the waves: each takes its share of the heads ----------------
#pragma unroll
  for (int k = 0; k < ATT_HEADS_OF_WAVE<GS_PAD>; ++k) {
    const int j = wave + k * NW;
    if (j >= gs) break;
    float m[NW], M = -INFINITY, a0 = 0.f, a1 = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      m[w] = sh_m[w][j];
      M = fmaxf(M, m[w]);
    }
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = m[w] == -INFINITY ? 0.f : __expf(m[w] - M);
      const float2 x = *reinterpret_cast<const float2*>(acc_of(w) + j * RI_DIM + 2 * lane);
      a0 += x.x * f;
      a1 += x.y * f;
      l += sh_l[w][j] * f;
    }
    if (S == 1) {   // the workgroup has the whole group: no partial leaves it
      write_head<HALF>(P, g, j, M, l, a0, a1);
      continue;
    }
    const size_t o = ((size_t)g * S + split) * GS_PAD + j;
    // device-coherent stores: another workgroup of this launch reads them
    __hip_atomic_store(reinterpret_cast<uint64_t*>(&P.part_acc[o * RI_DIM + 2 * lane]),
                       (uint64_t)__float_as_uint(a0) | (uint64_t)__float_as_uint(a1) << 32, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    if (lane == 0)
      __hip_atomic_store(reinterpret_cast<uint64_t*>(&P.part_ml[o * 2]),
                         (uint64_t)__float_as_uint(M) | (uint64_t)__float_as_uint(l) << 32, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  if (S == 1) {
    if (threadIdx.x == 0 && P.valid_lengths) P.valid_lengths[g] = lenA + lenB;
    return;
  }
  if constexpr (KEPT != KEPT_ALL) {

  // ---------------- the last wave of its share over all splits merges them ----------------
  // Hand-off of the partials between workgroups of one launch, wave by wave (no barrier, and a group's heads are merged
  // beside each other, by whichever workgroups come last: with the ranks found by whole waves, see rank_of, a layer of 16 groups
  // of 4 heads, 1024 clusters 17.8 -> 17.6 us, of 32 of 4, 8192 44.8 -> 44.4, of 64 of 8, 16384 128.4 -> 127.5) and without fences:
  //  * the partial was written above with agent-scope atomic stores: on gfx950 those are write-through
  //    stores (sc1) that complete in the memory-side cache every compute unit shares, not in this
  //    compute unit's L1 or this chiplet's L2;
  //  * s_waitcnt(0) returns when all of this wave's stores have been acknowledged there, and only then does the wave announce
  //    the arrival of its share with an agent-scope atomic increment (performed at the same shared level);
  //  * the wave that sees the count complete reads the partials of this share, and of no other, with agent-scope atomic
  //    loads (combine_share), which bypass the non-coherent cache levels.
  // So every partial is globally visible before its arrival can be counted, and the reader cannot hit a
  // stale line.  The C++ memory model would express this with a release increment and an acquire on the
  // last arriver; at agent scope those compile to a write-back and an invalidate of the whole L2, which
  // was measured at +15 us per launch (35.2 us instead of 20.0 us at the benchmark shape), while the
  // data that must be ordered is only this wave's own 2 KB.  Neither the wait nor relaxed atomics keep the compiler from moving
  // memory accesses over them, so empty asm statements do: the first keeps the stores above the wait, the second the increment
  // below it, the third the loads of the partials below the test of the count.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "the partial hand-off below relies on gfx950 cache behaviour: build this file for gfx950 only"
#endif
  if (wave >= gs) return;
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0);
  asm volatile("" ::: "memory");
  int* const arrived = P.counters + (g * NW + wave) * P.pitch;
  int before = 0;
  if (lane == 0) before = __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (__builtin_amdgcn_readfirstlane(before) != S - 1) return;
  asm volatile("" ::: "memory");
  combine_share<GS_PAD, HALF>(P, g, wave);
  if (threadIdx.x == 0 && P.valid_lengths) P.valid_lengths[g] = lenA + lenB;
  // ready for the next launch (every arrival of this launch has been counted; launches that share the
  // workspace do not overlap)
  if (lane == 0) __hip_atomic_store(arrived, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Checks the arguments of ri_wave_attention and lays them down with their split plan (attend.hip), as the launch plans it by
// itself, or with one workgroup per group, or without the rule that leaves a few rows to one.
enum { ATT_PLAN, ATT_ONE, ATT_SEVERAL };
int ri_prepare_wave_attention(AttendParams* P, const void* q, const void* steady_k, const void* steady_v,
                              int64_t steady_stride, int static_len, const int32_t* static_len_dev, const void* store_k,
                              const void* store_v, int64_t store_stride, const int32_t* row_src, int row_src_stride,
                              const int32_t* ret_tok_off, const int32_t* ret_start, int np, const int32_t* meta,
                              const int32_t* est_ids, const float* logits, const void* est_centroids, const void* value_sum,
                              const void* cluster_size_bf16, void* out, int32_t* valid_lengths, int BG, int gs, int nc,
                              int es, float scale, void* scratch, size_t scratch_bytes, int plan);
