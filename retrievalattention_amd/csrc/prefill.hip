// What prefill does around the clustering (gfx950): taking a sequence's K and V apart into the clustered range and the
// steady zone, centring the keys, and writing the index entries of the finished clustering.
// (cache_hub/retroinfer_cache.py:384-436.)  Everything here is bound by the bytes it moves; the element-wise launches it
// replaces moved them at a third to a half of the copy rate (transposed copies of 268 MB: 173 us each) and the small ones
// cost 4.5 us apiece.
#include "ri_common.h"

// ------------------------------------------------------------------------------------
// mean: the mean of every head's keys over the clustered range, read from where the model left them.
//
// The centred keys, and with them every bit of the index, hang on the order of this sum, so the order is fixed: rows
// i = r, r + S, r + 2S ... are added one after the other (chain r of S = 4 Y C, in fp32), chains r + j Y C (j = 0 .. 3) in
// order of j; of the Y C sums left, those of a c (r = c Y + y) as a tree over y; these into Y sums over c = y', y' + Y ...
// in order, and those as a tree.  Y and C are mean_order's.  It is the order in which torch 2.10 adds on this device
// (torch.mean(keys, dim=1) over [H, N, 128]), found from its sums over chosen inputs, so that an index built with
// torch.mean and one built here are the same to the bit.  The product with 1 / N is torch's as well: in half rounded once, to
// the element type, in bfloat16 first to fp32.
//
// mean_chain_kernel: a wave per chain and head, two dims per lane, MEAN_DEEP rows of it in flight (an addition waits for
// the one before, so a chain cannot be split: the rows in flight are what fills the link to memory).  Heads vary fastest:
// workgroups next to each other read whole tokens.
// mean_fold_kernel: a workgroup per head and 32 dims puts the chains together.
// Inside a prefill, 8 heads of 8192 / 131072 tokens and 4 of 48719: chains 6.6, 69 and 11.2 us, fold 2.4, 4.8 and 4.5, where
// torch.mean took 54, 168 and 157.  Bound by the rows in flight, there are only H S waves of 256 bytes a row: 268 MB at 3.9
// TB/s, where reading alone reaches 5.7.  (Over the same rows again and again, some of them in the memory-side cache: 8.3, 44
// and 14.7 us for both; with a branch around each of the loads 10.5, 73 and 25.)  And the mean is known before the heads are
// taken apart, so that pass centres them: 5.8 / 79 / 16.1 us for both, where a copy (6.7 / 91 / 15.7) and a pass over it (12 /
// 77 / 16) were needed.
// ------------------------------------------------------------------------------------
#define MEAN_DEEP 64
#define MEAN_MAX_C 256

// Longer prompts and more heads than the order has been compared for are not taken (false).
static bool mean_order(int H, int N, int* Y, int* C) {
  if (H <= 0 || H > 32 || N <= 0 || N > 262144 || (int64_t)H * N * RI_DIM * 2 > 0x7fffffffLL) return false;
  *Y = H == 1 ? 4 : 2;
  const int rows = (N + *Y - 1) / *Y;
  if (rows < 256) *C = 1;
  else if (H == 1) *C = rows <= 4096 ? min((rows + 15) / 16, 128) : 256;
  else for (*C = rows < 2048 ? 4 : 8; (rows + *C - 1) / *C >= 2048; *C *= 2) {}
  return true;
}

template <bool HALF>
__global__ __launch_bounds__(64) void mean_chain_kernel(const uint32_t* __restrict__ k, int64_t row, int64_t head,
                                                        float2* __restrict__ chains, int N, int H, int S) {
  const int h = blockIdx.x % H, r = blockIdx.x / H, lane = threadIdx.x;
  const int n = r < N ? (N - 1 - r) / S + 1 : 0;   // rows of the chain
  const uint32_t* at = k + h * head + r * row;
  const int64_t step = S * row;
  float s0 = 0.f, s1 = 0.f;
  uint32_t v[MEAN_DEEP];
  int left = n - 1;
  const auto fetch = [&](int e) {   // eight rows; past the last one it is repeated and not added
#pragma unroll
    for (int j = e; j < e + 8; ++j) {
      v[j] = at[lane];
      if (left > 0) at += step;
      --left;
    }
  };
  const auto add = [&](int j) { ri_add2<HALF>(v[j], s0, s1); };
  int i = 0;
  if (n >= MEAN_DEEP) {
#pragma unroll
    for (int e = 0; e < MEAN_DEEP; e += 8) fetch(e);
    // (no branch around a load here: the compiler counts the loads behind the ones it waits for, and takes those that may
    // not have been made for not made)
    for (; i + 2 * MEAN_DEEP <= n; i += MEAN_DEEP)
#pragma unroll
      for (int e = 0; e < MEAN_DEEP; e += 8) {
#pragma unroll
        for (int j = e; j < e + 8; ++j) add(j);
        fetch(e);
      }
    i += MEAN_DEEP;
#pragma unroll
    for (int e = 0; e < MEAN_DEEP; e += 8) {
#pragma unroll
      for (int j = e; j < e + 8; ++j) add(j);
      if (i + e < n) fetch(e);
    }
  } else {
#pragma unroll
    for (int e = 0; e < MEAN_DEEP; e += 8)
      if (e < n) fetch(e);
  }
#pragma unroll
  for (int e = 0; e < MEAN_DEEP; e += 8)
#pragma unroll
    for (int j = e; j < e + 8; ++j)
      if (i + j < n) add(j);
  chains[((size_t)h * S + r) * (RI_DIM / 2) + lane] = make_float2(s0, s1);
}

__device__ __forceinline__ float4 add4(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }

// grid (4, H): 32 dims each, four per thread
template <bool HALF, int Y>
__global__ __launch_bounds__(512) void mean_fold_kernel(const float4* __restrict__ chains, uint16_t* __restrict__ mean, int C,
                                                        float inv) {
  __shared__ __attribute__((aligned(16))) float sums[MEAN_MAX_C][32];
  static_assert(__alignof__(sums) == 16, "written four dims at a time");
  const int h = blockIdx.y, quad = threadIdx.x & 7;
  const float4* in = chains + (size_t)h * 4 * Y * C * (RI_DIM / 4) + blockIdx.x * 8 + quad;
  for (int c = threadIdx.x >> 3; c < C; c += 64) {
    float4 x[Y][4];
#pragma unroll
    for (int y = 0; y < Y; ++y)
#pragma unroll
      for (int j = 0; j < 4; ++j) x[y][j] = in[(size_t)(c * Y + y + Y * C * j) * (RI_DIM / 4)];
    float4 t[Y];
#pragma unroll
    for (int y = 0; y < Y; ++y) t[y] = add4(add4(add4(x[y][0], x[y][1]), x[y][2]), x[y][3]);
#pragma unroll
    for (int o = Y / 2; o > 0; o >>= 1)
#pragma unroll
      for (int y = 0; y < o; ++y) t[y] = add4(t[y], t[y + o]);
    *reinterpret_cast<float4*>(&sums[c][quad * 4]) = t[0];
  }
  __syncthreads();
  if (threadIdx.x >= 32) return;
  float t[Y];
#pragma unroll
  for (int y = 0; y < Y; ++y) t[y] = 0.f;
  int c = 0;
  for (; c + Y <= C; c += Y)
#pragma unroll
    for (int y = 0; y < Y; ++y) t[y] += sums[c + y][threadIdx.x];
#pragma unroll
  for (int y = 0; y < Y; ++y)
    if (c + y < C) t[y] += sums[c + y][threadIdx.x];
#pragma unroll
  for (int o = Y / 2; o > 0; o >>= 1)
#pragma unroll
    for (int y = 0; y < o; ++y) t[y] += t[y + o];
  // (half: the product of two 24-bit numbers is exact in 53 bits, one rounding; bfloat16: to fp32, then to the element type)
  mean[h * RI_DIM + blockIdx.x * 32 + threadIdx.x] =
      HALF ? __builtin_bit_cast(uint16_t, (_Float16)((double)t[0] * (double)inv)) : ri_f32_to_bf16(t[0] * inv);
}

extern "C" size_t ri_prefill_mean_workspace_bytes(int H, int N) {
  int Y, C;
  return mean_order(H, N, &Y, &C) ? (size_t)H * 4 * Y * C * RI_DIM * sizeof(float) : 0;
}

template <bool HALF>
static int prefill_mean(const void* key, int64_t row_stride, int64_t head_stride, int first, int N, int H, void* mean,
                        void* workspace, size_t workspace_bytes, hipStream_t s) {
  int Y, C;
  if (!key || !mean || !workspace || ri_any_misaligned16(key, mean, workspace) || first < 0 || row_stride < 0 ||
      head_stride < 0 || (row_stride | head_stride) % 8 != 0 || !mean_order(H, N, &Y, &C))
    return RI_ERR_ARG;
  if (workspace_bytes < ri_prefill_mean_workspace_bytes(H, N)) return RI_ERR_WORKSPACE;
  const int S = 4 * Y * C;
  mean_chain_kernel<HALF><<<H * S, 64, 0, s>>>((const uint32_t*)key + first * (row_stride / 2), row_stride / 2,
                                               head_stride / 2, (float2*)workspace, N, H, S);
  RI_HIP_CHECK_LAUNCH();
  auto* fold = Y == 4 ? mean_fold_kernel<HALF, 4> : mean_fold_kernel<HALF, 2>;
  fold<<<dim3(4, H), 512, 0, s>>>((const float4*)workspace, (uint16_t*)mean, C, 1.0f / (float)N);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_prefill_mean(const void* key, int64_t key_row_stride, int64_t key_head_stride, int first, int N, int H,
                               void* mean, void* workspace, size_t workspace_bytes, ri_stream_t stream) {
  return prefill_mean<false>(key, key_row_stride, key_head_stride, first, N, H, mean, workspace, workspace_bytes,
                             (hipStream_t)stream);
}

extern "C" int ri_prefill_mean_f16(const void* key, int64_t key_row_stride, int64_t key_head_stride, int first, int N, int H,
                                   void* mean, void* workspace, size_t workspace_bytes, ri_stream_t stream) {
  return prefill_mean<true>(key, key_row_stride, key_head_stride, first, N, H, mean, workspace, workspace_bytes,
                            (hipStream_t)stream);
}

// ------------------------------------------------------------------------------------
// split: keys[h, i] = K[first + i, h], less mean[h] where there is one, for the clustered range, and the steady rows of K
// and V.  16 lanes per row, a workgroup moves 16 rows of one head: occupancy keeps more loads in flight than several rows
// per thread do (8 heads of 8K / 128K tokens: 6.7 / 93 us; two or four rows per thread 19 / 105).  Heads vary fastest over
// the workgroups, so those in flight together read whole tokens.  Workgroups behind the clustered range move the steady
// rows, and those behind them the rows that a clustering starts from, which is a launch less in front of it, most of which the split
// takes longer where they are many (split + that launch / as it is: 8 heads x 8192 tokens 6.1 + 2.9 / 6.3 us, 8 x 131072 81.6 + 8.5 / 87.4;
// prefills 219 / 216, 4 x 50021 in half 575 / 574, 8 x 16384 377 / 372).
// ------------------------------------------------------------------------------------
struct SplitParams {
  const uint4* k;
  const uint4* v;
  const uint4* mean;   // [H, 16]
  uint4* keys;      // [H, N, 16] pieces
  uint4* zone_k;    // [H, zone_stride, 16]
  uint4* zone_v;
  int64_t k_row, k_head, v_row, v_head;   // pieces between tokens and between heads
  int64_t zone_stride;                    // rows between heads
  int first, N, start0, end0, n_start, n_end, H, blocks;   // blocks: of 16 clustered rows
  uint4* cent;      // [H, nc, 16] initial centroids (nc 0: none)
  int nc;
  float ratio, half;   // as ri_kmeans_first_row takes them
};

template <bool HALF>
__device__ __forceinline__ uint4 sub8(uint4 x, uint4 m) {
  return make_uint4(ri_sub2<HALF>(x.x, m.x), ri_sub2<HALF>(x.y, m.y), ri_sub2<HALF>(x.z, m.z), ri_sub2<HALF>(x.w, m.w));
}

template <bool CENTRE, bool HALF>
__global__ __launch_bounds__(256) void split_kernel(SplitParams P) {
  const int h = blockIdx.x % P.H, blk = blockIdx.x / P.H;
  const int piece = threadIdx.x & 15, sub = threadIdx.x >> 4;
  if (blk < P.blocks) {
    const int i = blk * 16 + sub;
    if (i >= P.N) return;
    const uint4 x = P.k[h * P.k_head + (P.first + (int64_t)i) * P.k_row + piece];
    P.keys[((int64_t)h * P.N + i) * 16 + piece] = CENTRE ? sub8<HALF>(x, P.mean[h * 16 + piece]) : x;
    return;
  }
  const int steady = (P.n_start + P.n_end + 15) / 16;
  if (blk >= P.blocks + steady) {
    const int c = (blk - P.blocks - steady) * 16 + sub;
    if (c >= P.nc) return;
    const int64_t i = ri_kmeans_first_row(c, P.ratio, P.half, P.N);
    const uint4 x = P.k[h * P.k_head + (P.first + i) * P.k_row + piece];
    P.cent[((int64_t)h * P.nc + c) * 16 + piece] = CENTRE ? sub8<HALF>(x, P.mean[h * 16 + piece]) : x;
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

template <bool CENTRE, bool HALF>
static int prefill_split(const void* key, const void* value, int64_t key_row_stride, int64_t key_head_stride,
                         int64_t value_row_stride, int64_t value_head_stride, int first, int N, int start0, int n_start,
                         int end0, int n_end, int H, const void* mean, void* keys, void* steady_k, void* steady_v,
                         int64_t steady_stride, void* cent, int nc, ri_stream_t stream) {
  if (!key || !value || !keys || !steady_k || !steady_v || (CENTRE && !mean)) return RI_ERR_ARG;
  if (ri_any_misaligned16(key, value, mean, keys, steady_k, steady_v) || ri_any_misaligned16(cent)) return RI_ERR_ARG;
  if (nc < 0 || (nc > 0 && !cent)) return RI_ERR_ARG;
  if (N <= 0 || H <= 0 || first < 0 || start0 < 0 || end0 < 0 || n_start < 0 || n_end < 0 ||
      steady_stride < n_start + n_end || key_row_stride < 0 || key_head_stride < 0 || value_row_stride < 0 ||
      value_head_stride < 0 || (key_row_stride | key_head_stride | value_row_stride | value_head_stride) % 8 != 0)
    return RI_ERR_ARG;
  const int blocks = N / 16 + (N % 16 != 0);
  const int64_t wgs = ((int64_t)blocks + ((int64_t)n_start + n_end + 15) / 16 + ((int64_t)nc + 15) / 16) * H;
  const double ratio = nc > 0 ? (double)N / nc : 0;
  if (wgs > 0x7fffffffLL) return RI_ERR_ARG;
  const SplitParams P = {(const uint4*)key, (const uint4*)value, (const uint4*)mean, (uint4*)keys, (uint4*)steady_k,
                         (uint4*)steady_v, key_row_stride / 8, key_head_stride / 8, value_row_stride / 8,
                         value_head_stride / 8, steady_stride, first, N, start0, end0, n_start, n_end, H, blocks,
                         (uint4*)cent, nc, (float)ratio, (float)(ratio / 2)};
  split_kernel<CENTRE, HALF><<<dim3((unsigned)wgs), 256, 0, (hipStream_t)stream>>>(P);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_prefill_split(const void* key, const void* value, int64_t key_row_stride, int64_t key_head_stride,
                                int64_t value_row_stride, int64_t value_head_stride, int first, int N, int start0,
                                int n_start, int end0, int n_end, int H, void* keys, void* steady_k, void* steady_v,
                                int64_t steady_stride, ri_stream_t stream) {
  return prefill_split<false, false>(key, value, key_row_stride, key_head_stride, value_row_stride, value_head_stride, first,
                                     N, start0, n_start, end0, n_end, H, nullptr, keys, steady_k, steady_v, steady_stride,
                                     nullptr, 0, stream);
}

extern "C" int ri_prefill_split_centred(const void* key, const void* value, int64_t key_row_stride, int64_t key_head_stride,
                                        int64_t value_row_stride, int64_t value_head_stride, int first, int N, int start0,
                                        int n_start, int end0, int n_end, int H, const void* mean, void* keys,
                                        void* steady_k, void* steady_v, int64_t steady_stride, ri_stream_t stream) {
  return prefill_split<true, false>(key, value, key_row_stride, key_head_stride, value_row_stride, value_head_stride, first,
                                    N, start0, n_start, end0, n_end, H, mean, keys, steady_k, steady_v, steady_stride,
                                    nullptr, 0, stream);
}

extern "C" int ri_prefill_split_centred_f16(const void* key, const void* value, int64_t key_row_stride,
                                            int64_t key_head_stride, int64_t value_row_stride, int64_t value_head_stride,
                                            int first, int N, int start0, int n_start, int end0, int n_end, int H,
                                            const void* mean, void* keys, void* steady_k, void* steady_v,
                                            int64_t steady_stride, ri_stream_t stream) {
  return prefill_split<true, true>(key, value, key_row_stride, key_head_stride, value_row_stride, value_head_stride, first, N,
                                   start0, n_start, end0, n_end, H, mean, keys, steady_k, steady_v, steady_stride, nullptr, 0,
                                   stream);
}

extern "C" int ri_prefill_split_init(const void* key, const void* value, int64_t key_row_stride, int64_t key_head_stride,
                                     int64_t value_row_stride, int64_t value_head_stride, int first, int N, int start0,
                                     int n_start, int end0, int n_end, int H, const void* mean, void* keys, void* steady_k,
                                     void* steady_v, int64_t steady_stride, void* centroids, int nc, ri_stream_t stream) {
  return prefill_split<true, false>(key, value, key_row_stride, key_head_stride, value_row_stride, value_head_stride, first,
                                    N, start0, n_start, end0, n_end, H, mean, keys, steady_k, steady_v, steady_stride,
                                    centroids, nc, stream);
}

extern "C" int ri_prefill_split_init_f16(const void* key, const void* value, int64_t key_row_stride, int64_t key_head_stride,
                                         int64_t value_row_stride, int64_t value_head_stride, int first, int N, int start0,
                                         int n_start, int end0, int n_end, int H, const void* mean, void* keys,
                                         void* steady_k, void* steady_v, int64_t steady_stride, void* centroids, int nc,
                                         ri_stream_t stream) {
  return prefill_split<true, true>(key, value, key_row_stride, key_head_stride, value_row_stride, value_head_stride, first, N,
                                   start0, n_start, end0, n_end, H, mean, keys, steady_k, steady_v, steady_stride, centroids,
                                   nc, stream);
}

// ------------------------------------------------------------------------------------
// center: keys[h, i] -= mean[h] (16-bit arithmetic: both operands widened, the difference rounded), in place.
// grid (ceil(rows / 16), H), 16 lanes per row.  For keys whose mean is taken after the split (mean_order's limits).
// ------------------------------------------------------------------------------------
template <bool HALF>
__global__ __launch_bounds__(256) void center_kernel(uint4* __restrict__ keys, const uint4* __restrict__ mean, int N) {
  const int i = blockIdx.x * 16 + (threadIdx.x >> 4), piece = threadIdx.x & 15;
  if (i >= N) return;
  uint4* kp = keys + ((size_t)blockIdx.y * N + i) * 16 + piece;
  const uint4 x = *kp, m = mean[(size_t)blockIdx.y * 16 + piece];
  *kp = sub8<HALF>(x, m);
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
// index: the cache's entries of a finished clustering, one launch for all of them, where they are not made with the stores
// (km_store_kernel).
// grid (ceil(nc / 16), H), 16 lanes per cluster.
// ------------------------------------------------------------------------------------
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
  out[at * 16 + piece] =
      make_uint4(ri_sum2<HALF>(x.x, m.x), ri_sum2<HALF>(x.y, m.y), ri_sum2<HALF>(x.z, m.z), ri_sum2<HALF>(x.w, m.w));
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
