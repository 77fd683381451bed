// Selection and block cache look-up of a host-resident decode step in one launch (gfx950).
#include "lru_body.h"
#include "select_body.h"

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
static void launch(const SelectArgs& P, const ri_lru_t& L, int BG, bool half, hipStream_t s) {
  const void* a = SRC == SEL_LOGITS ? (const void*)P.logits : (const void*)P.cent;
  const void* b = SRC == SEL_LOGITS ? (const void*)P.tile_max : (const void*)P.q;
  auto* kernel = half ? select_access_kernel<NT, E, GSM, true, SRC> : select_access_kernel<NT, E, GSM, false, SRC>;
  kernel<<<BG, NT, 0, s>>>(ri_pack_ptrs(a, b, P.tile_sum, P.mask), (ri_int4){P.nc, P.gs, P.np, P.es}, P.ntiles, P, L);
}
template <int NT, int E, int SRC>
static void launch_heads(const SelectArgs& P, const ri_lru_t& L, int BG, bool half, hipStream_t s) {
  if (P.gs <= 4) launch<NT, E, 4, SRC>(P, L, BG, half, s);
  else if (P.gs <= 8) launch<NT, E, 8, SRC>(P, L, BG, half, s);
  else launch<NT, E, 16, SRC>(P, L, BG, half, s);
}

// The selection's forms are those of ri_score_select, as far as it makes the scores' sums itself; a thread has one rank.
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
