// Centroid scoring and cluster selection for the decode step (gfx950).
//
// score_kernel    : logits[g,j,c] = scale * <q[g,j,:], centroid[g,c,:]> on bf16 MFMA, streamed
//                   once over the centroids, plus softmax partials per 256 or 64 columns.
// softmax_kernel  : the rest of the batch_gemm_softmax interface.
//
// Follows cache_hub/retroinfer_cache.py:569-575 and
// library/retroinfer/retroinfer_kernels/src/batch_gemm_softmax.h:222-243 (rounding pipeline).
#include "ri_common.h"

#define SCORE_TILE RI_SCORE_TILE  // columns of one softmax partial of the batch_gemm_softmax interface

// ------------------------------------------------------------------------------------
// score_kernel: grid (ntiles, BG), 256 threads = 4 waves, each wave owns 64 or 16 centroids.
// MFMA 16x16x32: A = 16 centroid rows, B = query heads (columns >= gs are zero).
// Accumulator register i of lane l holds row 4*(l/16)+i, column l%16.
// ------------------------------------------------------------------------------------
// HALF: the 16-bit element type of q, cent and the 16-bit logits is IEEE half instead of bfloat16
// (batch_gemm_softmax.cu:185-197 dispatches on Half and BFloat16).
template <bool HALF>
__device__ __forceinline__ uint16_t score_f32_to_16(float f) { return ri_f32_to_e16<HALF>(f); }

// TPW = 16-row centroid tiles per wave, NWV waves: a workgroup covers 16 TPW NWV centroids.
// Launched with 4 and 4 (SCORE_TILE, sixteen loads in flight per lane); eight waves with eight loads and sixteen with
// four were slower (29.96 and 32.1 us against 29.6 us for scoring + selection at 32 groups of 8192 centroids); where those
// workgroups are few with 1 and 4 (score_tile in select.hip).
// Softmax partials of the columns with one barrier: every wave reduces its own columns to a maximum and a
// sum of exponentials relative to that maximum, and after the barrier one thread per head folds the wave pairs
// (max of the maxima, sums rescaled by exp(m_w - M)).
template <bool HALF, int TPW, int NWV, bool STREAM>
__device__ __forceinline__ void score_body(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ cent, float* __restrict__ logits,
    uint16_t* __restrict__ logits_bf16, float* __restrict__ tile_max, float* __restrict__ tile_sum,
    int gs, int nc, int ntiles, float scale) {
  const int tile = blockIdx.x;
  const int g = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int r = lane & 15;
  const int h = lane >> 4;
  const int c0 = (tile * NWV + wave) * (16 * TPW);

  const uint16_t* cg = cent + (size_t)g * nc * RI_DIM;
  // Rows past the last centroid and query heads past gs read a valid row instead (their columns are never used): a load
  // under a condition is a branch of its own, and the compiler waited for everything before the last query pieces.
  uint4 a[TPW][4], bq[4];
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      a[t][i] = ri_ld16(cg + (size_t)min(c0 + t * 16 + 4 * i + h, nc - 1) * RI_DIM + r * 8);
  }
  {
    const uint16_t* p = q + ((size_t)g * gs + min(r, gs - 1)) * RI_DIM + h * 8;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) bq[kk] = ri_ld16(p + kk * 32);
  }
  __builtin_amdgcn_sched_barrier(0);   // every load is in flight before the first product

  __shared__ __attribute__((aligned(16))) uint4 sh_rows[NWV][256];
  f32x4_t acc[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    uint4 at[4];
    ri_rows_put(sh_rows[wave], a[t]);
    ri_wave_sync();
    ri_rows_get(sh_rows[wave], at);
    ri_wave_sync();   // (a wave's LDS accesses happen in order: the next rows need not wait for these)
    acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
      acc[t] = HALF ? __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, at[kk]),
                                                             __builtin_bit_cast(f16x8_t, bq[kk]), acc[t], 0, 0, 0)
                    : __builtin_amdgcn_mfma_f32_16x16x32_bf16(ri_as_bf16x8(at[kk]), ri_as_bf16x8(bq[kk]),
                                                              acc[t], 0, 0, 0);
  }

  // scale, and the wave's row maximum over its valid centroids.  The logits are stored at
  // the very end: a barrier waits for outstanding stores too.
  float lmax = -INFINITY;
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    const int cbase = c0 + t * 16 + 4 * h;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[t][i] *= scale;
      if (cbase + i < nc) lmax = fmaxf(lmax, acc[t][i]);
    }
  }
  __shared__ float sh_max[NWV][16];
  __shared__ float sh_sum[NWV][16];
  lmax = ri_xor_max<32>(ri_xor_max<16>(lmax));
  float lsum = 0.f;
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    const int cbase = c0 + t * 16 + 4 * h;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (cbase + i < nc) lsum += __expf(acc[t][i] - lmax);
  }
  lsum = ri_xor_sum<32>(ri_xor_sum<16>(lsum));
  if (h == 0) {
    sh_max[wave][r] = lmax;
    sh_sum[wave][r] = lsum;
  }
  __syncthreads();
  if ((int)threadIdx.x < gs) {
    const int j = threadIdx.x;
    float m = sh_max[0][j];
#pragma unroll
    for (int w = 1; w < NWV; ++w) m = fmaxf(m, sh_max[w][j]);
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      const float mw = sh_max[w][j];
      s += (mw == -INFINITY) ? 0.f : sh_sum[w][j] * __expf(mw - m);   // a wave past the last centroid holds nothing
    }
    const size_t o = ((size_t)g * ntiles + tile) * gs + j;
    tile_max[o] = m;
    tile_sum[o] = s;
  }
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    const int cbase = c0 + t * 16 + 4 * h;
    if (r < gs && cbase < nc) {  // nc % 4 == 0, so the four columns are valid together
      const size_t o = ((size_t)g * gs + r) * nc + cbase;
      if (logits) {
        // streaming store (STREAM): logits that leave the cache as they are written do not wait, dirty, for the write-back
        // at the end of the kernel (about 1 us per step at 32 groups of 8192 centroids)
        typedef float score_f4 __attribute__((ext_vector_type(4)));
        const score_f4 val = {acc[t][0], acc[t][1], acc[t][2], acc[t][3]};
        if (STREAM) __builtin_nontemporal_store(val, reinterpret_cast<score_f4*>(logits + o));
        else *reinterpret_cast<score_f4*>(logits + o) = val;
      }
      if (logits_bf16) {
        uint2 pk;
        pk.x = (uint32_t)score_f32_to_16<HALF>(acc[t][0]) | ((uint32_t)score_f32_to_16<HALF>(acc[t][1]) << 16);
        pk.y = (uint32_t)score_f32_to_16<HALF>(acc[t][2]) | ((uint32_t)score_f32_to_16<HALF>(acc[t][3]) << 16);
        *reinterpret_cast<uint2*>(logits_bf16 + o) = pk;
      }
    }
  }
}

template <bool HALF, int TPW, int NWV, bool STREAM>
__global__ __launch_bounds__(64 * NWV) void score_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ cent, float* __restrict__ logits,
    uint16_t* __restrict__ logits16, float* __restrict__ tile_max, float* __restrict__ tile_sum,
    int gs, int nc, int ntiles, float scale) {
  score_body<HALF, TPW, NWV, STREAM>(q, cent, logits, logits16, tile_max, tile_sum, gs, nc, ntiles, scale);
}

// Row statistics and softmax, a workgroup per row: every wave reduces the row's partials, with the workgroup's first 8
// elements per thread in flight, and the finals go to slot 0 once all have read it.  (One launch for two: 7 -> 4 us of 32
// groups of 4 x 8192, and the apply no longer waits for the reduction of every other row.)
template <bool HALF>
__global__ __launch_bounds__(1024) void softmax_kernel(const uint4* __restrict__ d, float* norm, float* sum,
                                                       uint4* __restrict__ soft, int ntiles, int gs, int pieces) {
  const int g = blockIdx.y, j = blockIdx.x;
  const size_t base = ((size_t)g * gs + j) * pieces;
  float* pm = norm + (size_t)g * ntiles * gs;
  float* ps = sum + (size_t)g * ntiles * gs;
  uint4 v = d[base + min((int)threadIdx.x, pieces - 1)];
  float m, iz;
  ri_wave_reduce_partials(pm, ps, ntiles, gs, j, threadIdx.x & 63, &m, &iz);
  __syncthreads();  // every wave has read slot 0 before it is overwritten
  if (threadIdx.x == 0) {
    pm[j] = m;
    ps[j] = iz;
  }
  for (int i = threadIdx.x; i < pieces; i += blockDim.x) {
    if (i != (int)threadIdx.x) v = d[base + i];
    const uint32_t in[4] = {v.x, v.y, v.z, v.w};
    uint32_t o[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float lo, hi;
      ri_unpack2<HALF>(in[u], lo, hi);
      o[u] = (uint32_t)score_f32_to_16<HALF>(__expf(lo - m) * iz) |
             ((uint32_t)score_f32_to_16<HALF>(__expf(hi - m) * iz) << 16);
    }
    soft[base + i] = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// LDS that a scoring launch asks for and does not use: from three rounds of workgroups on, two to a compute unit stream faster
// than the four that fit (128 KB of rows on their way to a unit, not 256; a kernel that only reads shows the same).  A step, us,
// four / two / one: 64 groups of 8 heads, 16384 clusters 125.7 / 123.1 / 140; four / two: 64 of 4, 16384 122.9 / 119.9, 128 of 4, 8192
// 121.1 / 118.3, 48 of 8, 16384 104.5 / 103.0, 64 of 12, 16384 138.3 / 137.3; two rounds: 64 of 4, 8192 70.3 / 69.7, 32 of 4, 16384 71.3 /
// 70.9, but 128 of 8, 4096 74.3 / 74.9; less: 24 of 4, 16384 59.7 / 59.9, 32 of 8, 8192 44.3 / 45.1.  (Three to a unit 126.2 in the first.)
// Where the scores go out in 16 bits and a softmax reads them back, only up to four heads, or from six rounds on.  Four / two to a
// unit, inputs in turn: 64 of 4, 16384 56.2 / 54.0, 96 of 4, 8192 43.6 / 42.9, but 96 of 8, 8192 47.8 / 48.0, 48 of 12, 16384 51.0 / 51.9, 128 of
// 16, 8192 71.9 / 72.3 (the same input again, 64 of 8, 16384 51.8 / 53.5); six rounds, 96 of 8, 16384 90.1 / 87.2, of 12 96.8 / 95.5.
static size_t score_spread(int64_t workgroups) { return workgroups >= 3 * 1024 ? 56 * 1024 : 0; }

// ------------------------------------------------------------------------------------
// C entry points
// ------------------------------------------------------------------------------------
static int check_score_shape(int BG, int gs, int nc, int k) {
  if (BG <= 0 || gs <= 0 || gs > 16 || nc <= 0 || (nc % 8) != 0 || k != RI_DIM) return RI_ERR_ARG;
  return RI_OK;
}

template <bool HALF>
static int batch_gemm_softmax_impl(const void* A, const void* B, void* D, float* Norm, float* Sum, void* Softmax,
                                   int batch_count, int m, int n, int k, float alpha, float beta,
                                   ri_stream_t stream) {
  if (!A || !B || !D || !Norm || !Sum || !Softmax || beta != 0.f) return RI_ERR_ARG;
  if (ri_any_misaligned16(A, B, D, Softmax)) return RI_ERR_ARG;
  int rc = check_score_shape(batch_count, m, n, k);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  const int ntiles = (n + SCORE_TILE - 1) / SCORE_TILE;
  // fp32 logits are not part of this interface: the partial statistics come from the fp32
  // accumulators inside the kernel, the softmax from the 16-bit D, as in the reference.
  const int64_t workgroups = (int64_t)ntiles * batch_count;
  const size_t spread = m <= 4 || workgroups >= 6 * 1024 ? score_spread(workgroups) : 0;
  score_kernel<HALF, 4, 4, false><<<dim3(ntiles, batch_count), 256, spread, s>>>(
      (const uint16_t*)A, (const uint16_t*)B, nullptr, (uint16_t*)D, Norm, Sum, m, n, ntiles, alpha);
  RI_HIP_CHECK_LAUNCH();
  const int threads = min(1024, (n / 8 + 63) / 64 * 64);
  softmax_kernel<HALF><<<dim3(m, batch_count), threads, 0, s>>>((const uint4*)D, Norm, Sum, (uint4*)Softmax, ntiles, m,
                                                                n / 8);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_batch_gemm_softmax(const void* A, const void* B, void* D, float* Norm, float* Sum,
                                     void* Softmax, int batch_count, int m, int n, int k, float alpha,
                                     float beta, ri_stream_t stream) {
  return batch_gemm_softmax_impl<false>(A, B, D, Norm, Sum, Softmax, batch_count, m, n, k, alpha, beta, stream);
}

extern "C" int ri_batch_gemm_softmax_f16(const void* A, const void* B, void* D, float* Norm, float* Sum,
                                         void* Softmax, int batch_count, int m, int n, int k, float alpha,
                                         float beta, ri_stream_t stream) {
  return batch_gemm_softmax_impl<true>(A, B, D, Norm, Sum, Softmax, batch_count, m, n, k, alpha, beta, stream);
}


// scoring pass used by the fused selection (select.hip)
int ri_launch_score(const void* q, const void* centroids, float* logits, float* tile_max, float* tile_sum,
                    int BG, int gs, int nc, int tile, float scale, bool half, hipStream_t s) {
  const int ntiles = (nc + tile - 1) / tile;
  const uint16_t *qq = (const uint16_t*)q, *cc = (const uint16_t*)centroids;
  // Up to 32 MB of centroids the logits are better left where the next kernels find them (whole steps: 8 groups of 8 heads,
  // 4096 centroids 25.9 -> 25.0 us, 16 of 16, 2048 32.0 -> 30.9, 12 of 7, 1856 24.8 -> 24.4; 16 of 4, 8192 34.7 either way);
  // with more the write-back is longer than that (32 of 4, 8192 46.1 streamed, 46.4 not).
  const bool stream = (size_t)BG * nc > 128 * 1024;
  auto* kernel = half ? (stream ? score_kernel<true, 4, 4, true> : score_kernel<true, 4, 4, false>)
                      : (stream ? score_kernel<false, 4, 4, true> : score_kernel<false, 4, 4, false>);
  if (tile == RI_SCORE_TILE_FEW) kernel = half ? score_kernel<true, 1, 4, false> : score_kernel<false, 1, 4, false>;
  const size_t spread = tile == RI_SCORE_TILE_FEW ? 0 : score_spread((int64_t)ntiles * BG);
  kernel<<<dim3(ntiles, BG), 256, spread, s>>>(qq, cc, logits, nullptr, tile_max, tile_sum, gs, nc, ntiles, scale);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}
