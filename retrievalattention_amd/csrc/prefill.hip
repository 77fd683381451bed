// What prefill does around the clustering (gfx950): taking a sequence's K and V apart into the clustered range and the
// steady zone, centring the keys, and writing the index entries of the finished clustering.
// (cache_hub/retroinfer_cache.py:384-436.)  Everything here is bound by the bytes it moves; the element-wise launches it
// replaces moved them at a third to a half of the copy rate (transposed copies of 268 MB: 173 us each) and the small ones
// cost 4.5 us apiece.
#include "ri_common.h"

// ------------------------------------------------------------------------------------
// split: keys[h, i] = K[first + i, h] for the clustered range, and the steady rows of K and V.
// 16 lanes per row, a workgroup moves 16 rows of one head: occupancy keeps more loads in flight than several rows per
// thread do (8 heads of 8K / 128K tokens: 6.7 / 93 us; two or four rows per thread 19 / 105).  Heads vary fastest over
// the workgroups, so those in flight together read whole tokens.  Workgroups behind the clustered range move the steady
// rows.
// ------------------------------------------------------------------------------------
struct SplitParams {
  const uint4* k;
  const uint4* v;
  uint4* keys;      // [H, N, 16] pieces
  uint4* zone_k;    // [H, zone_stride, 16]
  uint4* zone_v;
  int64_t k_row, k_head, v_row, v_head;   // pieces between tokens and between heads
  int64_t zone_stride;                    // rows between heads
  int first, N, start0, end0, n_start, n_end, H, blocks;   // blocks: of 16 clustered rows
};

__global__ __launch_bounds__(256) void split_kernel(SplitParams P) {
  const int h = blockIdx.x % P.H, blk = blockIdx.x / P.H;
  const int piece = threadIdx.x & 15, sub = threadIdx.x >> 4;
  if (blk < P.blocks) {
    const int i = blk * 16 + sub;
    if (i < P.N) P.keys[((int64_t)h * P.N + i) * 16 + piece] = P.k[h * P.k_head + (P.first + (int64_t)i) * P.k_row + piece];
    return;
  }
  const int i = (blk - P.blocks) * 16 + sub;
  if (i >= P.n_start + P.n_end) return;
  const int64_t tok = i < P.n_start ? P.start0 + i : P.end0 + (i - P.n_start);
  const uint4 xk = P.k[tok * P.k_row + h * P.k_head + piece], xv = P.v[tok * P.v_row + h * P.v_head + piece];
  const int64_t to = (h * P.zone_stride + i) * 16 + piece;
  P.zone_k[to] = xk;
  P.zone_v[to] = xv;
}

extern "C" int ri_prefill_split(const void* key, const void* value, int64_t key_row_stride, int64_t key_head_stride,
                                int64_t value_row_stride, int64_t value_head_stride, int first, int N, int start0,
                                int n_start, int end0, int n_end, int H, void* keys, void* steady_k, void* steady_v,
                                int64_t steady_stride, ri_stream_t stream) {
  if (!key || !value || !keys || !steady_k || !steady_v) return RI_ERR_ARG;
  if (ri_any_misaligned16(key, value, keys, steady_k, steady_v)) return RI_ERR_ARG;
  if (N <= 0 || H <= 0 || first < 0 || start0 < 0 || end0 < 0 || n_start < 0 || n_end < 0 ||
      steady_stride < n_start + n_end || key_row_stride < 0 || key_head_stride < 0 || value_row_stride < 0 ||
      value_head_stride < 0 || (key_row_stride | key_head_stride | value_row_stride | value_head_stride) % 8 != 0)
    return RI_ERR_ARG;
  const int blocks = N / 16 + (N % 16 != 0);
  const int64_t wgs = ((int64_t)blocks + ((int64_t)n_start + n_end + 15) / 16) * H;
  if (wgs > 0x7fffffffLL) return RI_ERR_ARG;
  const SplitParams P = {(const uint4*)key, (const uint4*)value, (uint4*)keys, (uint4*)steady_k, (uint4*)steady_v,
                         key_row_stride / 8, key_head_stride / 8, value_row_stride / 8, value_head_stride / 8,
                         steady_stride, first, N, start0, end0, n_start, n_end, H, blocks};
  split_kernel<<<dim3((unsigned)wgs), 256, 0, (hipStream_t)stream>>>(P);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

// ------------------------------------------------------------------------------------
// center: keys[h, i] -= mean[h] (16-bit arithmetic: both operands widened, the difference rounded), in place.
// grid (ceil(rows / 16), H), 16 lanes per row.
// ------------------------------------------------------------------------------------
template <bool HALF>
__global__ __launch_bounds__(256) void center_kernel(uint4* __restrict__ keys, const uint4* __restrict__ mean, int N) {
  const int i = blockIdx.x * 16 + (threadIdx.x >> 4), piece = threadIdx.x & 15;
  if (i >= N) return;
  uint4* kp = keys + ((size_t)blockIdx.y * N + i) * 16 + piece;
  const uint4 x = *kp, m = mean[(size_t)blockIdx.y * 16 + piece];
  *kp = make_uint4(ri_sub2<HALF>(x.x, m.x), ri_sub2<HALF>(x.y, m.y), ri_sub2<HALF>(x.z, m.z), ri_sub2<HALF>(x.w, m.w));
}

static int prefill_center(void* keys, const void* mean, int H, int N, bool half, ri_stream_t stream) {
  if (!keys || !mean || ri_any_misaligned16(keys, mean) || H <= 0 || H > 65535 || N <= 0) return RI_ERR_ARG;
  const dim3 grid(N / 16 + (N % 16 != 0), H);
  if (half) center_kernel<true><<<grid, 256, 0, (hipStream_t)stream>>>((uint4*)keys, (const uint4*)mean, N);
  else center_kernel<false><<<grid, 256, 0, (hipStream_t)stream>>>((uint4*)keys, (const uint4*)mean, N);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_prefill_center(void* keys, const void* mean, int H, int N, ri_stream_t stream) {
  return prefill_center(keys, mean, H, N, false, stream);
}

extern "C" int ri_prefill_center_f16(void* keys, const void* mean, int H, int N, ri_stream_t stream) {
  return prefill_center(keys, mean, H, N, true, stream);
}

// ------------------------------------------------------------------------------------
// index: the cache's entries of a finished clustering, one launch for all of them.
// grid (ceil(nc / 16), H), 16 lanes per cluster.
// ------------------------------------------------------------------------------------
template <bool HALF>
__device__ __forceinline__ uint32_t add2(uint32_t a, uint32_t b) {
  float a0, a1, b0, b1;
  ri_unpack2<HALF>(a, a0, a1);
  ri_unpack2<HALF>(b, b0, b1);
  return (uint32_t)ri_f32_to_e16<HALF>(a0 + b0) | ((uint32_t)ri_f32_to_e16<HALF>(a1 + b1) << 16);
}

template <bool HALF>
__global__ __launch_bounds__(256) void index_kernel(const uint4* __restrict__ cent, const uint4* __restrict__ mean,
                                                    const int32_t* __restrict__ counts,
                                                    const int32_t* __restrict__ offsets, uint4* __restrict__ out,
                                                    uint8_t* __restrict__ mask, uint16_t* __restrict__ size16,
                                                    int32_t* __restrict__ size, int32_t* __restrict__ start, int nc) {
  const int h = blockIdx.y, c = blockIdx.x * 16 + (threadIdx.x >> 4), piece = threadIdx.x & 15;
  if (c >= nc) return;
  const size_t at = (size_t)h * nc + c;
  const uint4 x = cent[at * 16 + piece], m = mean[(size_t)h * 16 + piece];
  out[at * 16 + piece] = make_uint4(add2<HALF>(x.x, m.x), add2<HALF>(x.y, m.y), add2<HALF>(x.z, m.z), add2<HALF>(x.w, m.w));
  if (piece == 0) {
    const int32_t n = counts[at];
    mask[at] = n == 0;
    size16[at] = ri_f32_to_e16<HALF>((float)n);
    size[at] = n;
    start[at] = offsets[(size_t)h * (nc + 1) + c];
  }
}

static int prefill_index(const void* centroids, const void* mean, const int32_t* counts, const int32_t* offsets, void* out,
                         uint8_t* mask, void* size16, int32_t* size, int32_t* start, int H, int nc, bool half,
                         ri_stream_t stream) {
  if (!centroids || !mean || !counts || !offsets || !out || !mask || !size16 || !size || !start) return RI_ERR_ARG;
  if (ri_any_misaligned16(centroids, mean, out) || H <= 0 || H > 65535 || nc <= 0) return RI_ERR_ARG;
  const dim3 grid((nc + 15) / 16, H);
  auto* kernel = half ? index_kernel<true> : index_kernel<false>;
  kernel<<<grid, 256, 0, (hipStream_t)stream>>>((const uint4*)centroids, (const uint4*)mean, counts, offsets, (uint4*)out,
                                                mask, (uint16_t*)size16, size, start, nc);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_prefill_index(const void* centroids, const void* mean, const int32_t* counts, const int32_t* offsets,
                                void* out, uint8_t* mask, void* size16, int32_t* size, int32_t* start, int H, int nc,
                                ri_stream_t stream) {
  return prefill_index(centroids, mean, counts, offsets, out, mask, size16, size, start, H, nc, false, stream);
}

extern "C" int ri_prefill_index_f16(const void* centroids, const void* mean, const int32_t* counts,
                                    const int32_t* offsets, void* out, uint8_t* mask, void* size16, int32_t* size,
                                    int32_t* start, int H, int nc, ri_stream_t stream) {
  return prefill_index(centroids, mean, counts, offsets, out, mask, size16, size, start, H, nc, true, stream);
}
