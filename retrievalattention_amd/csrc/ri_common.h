// Shared device/host helpers for the gfx950 wave-index kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/retro_mi355.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define RI_DIM 128  // head dimension every kernel is specialised for

// ---- bf16 <-> fp32 (round-to-nearest-even, NaN preserved as quiet NaN) ----
__host__ __device__ __forceinline__ float ri_bf16_to_f32(uint16_t v) {
  union { uint32_t u; float f; } x;
  x.u = (uint32_t)v << 16;
  return x.f;
}
__host__ __device__ __forceinline__ uint16_t ri_f32_to_bf16(float f) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(uint16_t, (__bf16)f);   // one conversion instruction; the code below is three and a branch
#endif
  union { uint32_t u; float f; } x;
  x.f = f;
  if ((x.u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((x.u >> 16) | 0x40u);
  uint32_t r = ((x.u >> 16) & 1u) + 0x7fffu;
  return (uint16_t)((x.u + r) >> 16);
}
// fp32 value of the bf16 rounding of f
__host__ __device__ __forceinline__ float ri_round_bf16(float f) {
  return ri_bf16_to_f32(ri_f32_to_bf16(f));
}

// ---- the two 16-bit element types: bfloat16 (HALF = false) and IEEE half (HALF = true) ----
// The fused decode path, the k-means and the operators take either (the reference's operators and cache are
// generic over Half and BFloat16: batch_gemm_softmax.cu:185-197, gather_copy.cu:63-67); a kernel is
// instantiated per type and the entry points come in pairs (name, name_f16).
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));

template <bool HALF>
__host__ __device__ __forceinline__ float ri_e16_to_f32(uint16_t v) {
  if (HALF) {
#if defined(__HIP_DEVICE_COMPILE__)
    return (float)__builtin_bit_cast(_Float16, v);
#else
    // host side: plain bit arithmetic (normal, subnormal, inf/nan)
    const uint32_t s = (uint32_t)(v & 0x8000u) << 16, e = (v >> 10) & 31u, m = v & 0x3ffu;
    union { uint32_t u; float f; } x;
    if (e == 0) {
      x.f = (float)m * 5.9604644775390625e-08f;   // m * 2^-24
      x.u |= s;
    } else {
      x.u = s | (e == 31 ? 0x7f800000u : (e + 112u) << 23) | (m << 13);
    }
    return x.f;
#endif
  }
  return ri_bf16_to_f32(v);
}
// round to nearest even
template <bool HALF>
__device__ __forceinline__ uint16_t ri_f32_to_e16(float f) {
  if (HALF) return __builtin_bit_cast(uint16_t, (_Float16)f);
  return ri_f32_to_bf16(f);
}
// fp32 value of the 16-bit rounding of f
template <bool HALF>
__device__ __forceinline__ float ri_round_e16(float f) {
  return ri_e16_to_f32<HALF>(ri_f32_to_e16<HALF>(f));
}
// the two elements packed in a 32-bit word, as fp32
template <bool HALF>
__device__ __forceinline__ void ri_unpack2(uint32_t w, float& lo, float& hi) {
  if (HALF) {
    lo = (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xffffu));
    hi = (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
  } else {
    lo = __uint_as_float(w << 16);
    hi = __uint_as_float(w & 0xffff0000u);
  }
}
// s0 += the low element, s1 += the high one, each rounded once.  Halves as x * 1 + s, the same number: one instruction
// where a conversion and an addition are two (the compiler makes the two of it).
template <bool HALF>
__device__ __forceinline__ void ri_add_lo(uint32_t w, float& s) {
  if (HALF) asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel_hi:[1,0,0]" : "+v"(s) : "v"(w));
  else s += __uint_as_float(w << 16);
}
template <bool HALF>
__device__ __forceinline__ void ri_add2(uint32_t w, float& s0, float& s1) {
  ri_add_lo<HALF>(w, s0);
  if (HALF) asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(s1) : "v"(w));
  else s1 += __uint_as_float(w & 0xffff0000u);
}
// the row that centroid c of a clustering of N rows starts from: trunc(c * ratio + half) in fp32, ratio and half of N / nc
// (two roundings: built without fp contraction)
__device__ __forceinline__ int ri_kmeans_first_row(int c, float ratio, float half, int N) {
  const float x = (float)c * ratio;
  return min((int)(x + half), N - 1);
}
// a - b on packed pairs: both operands widened, the differences rounded
template <bool HALF>
__device__ __forceinline__ uint32_t ri_sub2(uint32_t a, uint32_t b) {
  float a0, a1, b0, b1;
  ri_unpack2<HALF>(a, a0, a1);
  ri_unpack2<HALF>(b, b0, b1);
  return (uint32_t)ri_f32_to_e16<HALF>(a0 - b0) | ((uint32_t)ri_f32_to_e16<HALF>(a1 - b1) << 16);
}
// a + b, as ri_sub2
template <bool HALF>
__device__ __forceinline__ uint32_t ri_sum2(uint32_t a, uint32_t b) {
  float a0, a1, b0, b1;
  ri_unpack2<HALF>(a, a0, a1);
  ri_unpack2<HALF>(b, b0, b1);
  return (uint32_t)ri_f32_to_e16<HALF>(a0 + b0) | ((uint32_t)ri_f32_to_e16<HALF>(a1 + b1) << 16);
}
// finfo(type).min as a bit pattern: the score of a masked (empty) cluster
template <bool HALF>
__host__ __device__ __forceinline__ uint16_t ri_e16_lowest() { return HALF ? 0xfbff : 0xff7f; }

__device__ __forceinline__ bf16x8_t ri_as_bf16x8(uint4 v) {
  return __builtin_bit_cast(bf16x8_t, v);
}
__device__ __forceinline__ uint4 ri_ld16(const void* p) {
  return *reinterpret_cast<const uint4*>(p);
}
__device__ __forceinline__ uint4 ri_zero16() { return make_uint4(0u, 0u, 0u, 0u); }

// unpack 8 bf16 packed in a uint4 into fp32
__device__ __forceinline__ void ri_unpack8(uint4 v, float* f) {
  f[0] = __uint_as_float(v.x << 16); f[1] = __uint_as_float(v.x & 0xffff0000u);
  f[2] = __uint_as_float(v.y << 16); f[3] = __uint_as_float(v.y & 0xffff0000u);
  f[4] = __uint_as_float(v.z << 16); f[5] = __uint_as_float(v.z & 0xffff0000u);
  f[6] = __uint_as_float(v.w << 16); f[7] = __uint_as_float(v.w & 0xffff0000u);
}

// bf16 bit pattern -> key whose unsigned order equals the float order
__host__ __device__ __forceinline__ uint32_t ri_bf16_sort_key(uint16_t b) {
  return (b & 0x8000u) ? (uint32_t)(~b & 0xffffu) : (uint32_t)(b | 0x8000u);
}

__device__ __forceinline__ void ri_wave_sync() {   // LDS written by this wave is read by this wave
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sixteen rows of 128 elements as operands of MFMA 16x16x32 (lane l: row l % 16, dims 32 kk + 8 (l / 16) ..).  They are
// loaded four whole rows per instruction (lane l: piece l % 16 of row 4 i + l / 16) and turned in 4 KiB of the wave's LDS,
// because a compute unit takes a cycle and more per row that sixteen neighbouring lanes of a load touch: rows per lane
// stream 14.5 bytes per cycle from the L2, whole rows 43 to 56 (one workgroup, 128 .. 512 KB).  Scoring and selection of 8
// groups of 4 heads and 512 clusters 10.2 -> 8.0 us, of 16 and 1024 11.6 -> 10.8, of 12 of 7 heads and 1856 13.5 -> 13.0;
// where all compute units stream, memory bounds it (32 of 8192: 26).  The attention, whose rows are few per wave and in a
// chain, gains nothing by it and loads its keys by lanes.  Piece p of row r lies at place p ^ r of its row: both accesses
// hit all banks once.
__device__ __forceinline__ void ri_rows_put(uint4* sh, const uint4 (&v)[4]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 4 * i + (lane >> 4);
    sh[row * 16 + ((lane & 15) ^ row)] = v[i];
  }
}
__device__ __forceinline__ void ri_rows_get(const uint4* sh, uint4 (&o)[4]) {
  const int r = threadIdx.x & 15, h = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) o[kk] = sh[r * 16 + ((h + 4 * kk) ^ r)];
}

// Rows of bf16 matrices are read and written 16 bytes at a time: their base pointers must be
// 16-byte aligned (a null pointer counts as aligned: optional arguments are checked elsewhere).
static inline bool ri_misaligned16(const void* p) { return ((uintptr_t)p & 15u) != 0; }
template <typename... P>
static inline bool ri_any_misaligned16(P... p) {
  return (ri_misaligned16((const void*)p) || ...);
}

#define RI_HIP_CHECK_LAUNCH()                         \
  do {                                                \
    hipError_t e__ = hipGetLastError();               \
    if (e__ != hipSuccess) {                          \
      ri_set_last_hip_error((int)e__);                \
      return RI_ERR_LAUNCH;                           \
    }                                                 \
  } while (0)

void ri_set_last_hip_error(int e);

// {a, b} = this lane's value and that of lane (lane ^ D), in either order; register moves only
template <int D>
__device__ __forceinline__ void ri_lane_pair(uint32_t v, uint32_t& a, uint32_t& b) {
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

// x combined with that of lane (lane ^ D) (commutative, so every lane of a pair gets the same bits), and over the whole
// wave from the far lanes to the near ones.  (A shuffle through the LDS crossbar takes about a hundred cycles, and in these
// chains each waits for the one before: with register moves scoring + selection of 12 groups of 7 heads, 1856 clusters 12.9
// -> 12.6 us, of 16 of 16, 2048 18.8 -> 17.8, nine updates of 8 x 8192 tokens 104.3 -> 101.4.)
template <int D>
__device__ __forceinline__ float ri_xor_max(float x) {
  uint32_t a, b;
  ri_lane_pair<D>(__float_as_uint(x), a, b);
  return fmaxf(__uint_as_float(a), __uint_as_float(b));
}
template <int D>
__device__ __forceinline__ float ri_xor_sum(float x) {
  uint32_t a, b;
  ri_lane_pair<D>(__float_as_uint(x), a, b);
  return __uint_as_float(a) + __uint_as_float(b);
}
__device__ __forceinline__ float ri_wave_max(float x) {
  return ri_xor_max<1>(ri_xor_max<2>(ri_xor_max<4>(ri_xor_max<8>(ri_xor_max<16>(ri_xor_max<32>(x))))));
}
__device__ __forceinline__ float ri_wave_sum(float x) {
  return ri_xor_sum<1>(ri_xor_sum<2>(ri_xor_sum<4>(ri_xor_sum<8>(ri_xor_sum<16>(ri_xor_sum<32>(x))))));
}

// Kernel arguments that are wanted at once: the first fourteen words are in registers when a wave starts, but none of a struct;
// as vectors they are few arguments for the host to lay out (about 20 ns each).
typedef uint64_t ri_ptr4 __attribute__((ext_vector_type(4)));
typedef int ri_int4 __attribute__((ext_vector_type(4)));
typedef int ri_int2 __attribute__((ext_vector_type(2)));
// (through a global pointer: from an integer alone the compiler makes loads that ask where the address lies)
template <typename T>
__device__ __forceinline__ T* ri_global(uint64_t p) {
  return (T*)(__attribute__((address_space(1))) T*)p;
}
static inline ri_ptr4 ri_pack_ptrs(const void* a, const void* b, const void* c, const void* d) {
  return (ri_ptr4){(uint64_t)a, (uint64_t)b, (uint64_t)c, (uint64_t)d};
}

// ---- shared between score.hip and select.hip ----
#define RI_SCORE_TILE 256          // centroids per scoring workgroup and softmax partial
#define RI_SCORE_TILE_FEW 64       // where that is few workgroups (score_tile in select.hip)
// tile: RI_SCORE_TILE or RI_SCORE_TILE_FEW
int ri_launch_score(const void* q, const void* centroids, float* logits, float* tile_max, float* tile_sum,
                    int BG, int gs, int nc, int tile, float scale, bool half, hipStream_t s);

// Row statistics from the partials of a row's tiles [ntiles, gs]: one wave per row, lanes over
// tiles, xor-butterfly reductions (fixed order, so the result is reproducible).
__device__ __forceinline__ void ri_wave_reduce_partials(const float* pm, const float* ps, int ntiles, int gs,
                                                        int j, int lane, float* m_out, float* invz_out) {
  // the first 64 tiles' partials are loaded together, ahead of the reductions
  const bool has0 = lane < ntiles;
  const float pm0 = has0 ? pm[(size_t)lane * gs + j] : -INFINITY;
  const float ps0 = has0 ? ps[(size_t)lane * gs + j] : 0.f;
  float m = pm0;
  for (int t = lane + 64; t < ntiles; t += 64) m = fmaxf(m, pm[(size_t)t * gs + j]);
  m = ri_wave_max(m);
  float z = has0 ? ps0 * __expf(pm0 - m) : 0.f;
  for (int t = lane + 64; t < ntiles; t += 64) z += ps[(size_t)t * gs + j] * __expf(pm[(size_t)t * gs + j] - m);
  *m_out = m;
  *invz_out = 1.0f / ri_wave_sum(z);
}

// The same from at most 64 partials, a lane's own (-inf, 0 past the last).
__device__ __forceinline__ void ri_wave_reduce_partials(float pm, float ps, float* m_out, float* invz_out) {
  const float m = ri_wave_max(pm);
  *m_out = m;
  *invz_out = 1.0f / ri_wave_sum(ps * __expf(pm - m));
}

// Inclusive prefix sum over the 64 lanes of a wave with DPP row shifts and row broadcasts
// (no LDS traffic): shifts by 1, 2, 3 build sums of four neighbours, shifts by 4 and 8 finish the
// 16-lane rows, the two broadcasts carry row totals into the rows behind.
__device__ __forceinline__ uint32_t ri_wave_incl_scan(uint32_t v) {
  uint32_t r = v;
  r += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);   // row_shr:1
  r += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);   // row_shr:2
  r += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x113, 0xf, 0xf, true);   // row_shr:3
  r += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)r, 0x114, 0xf, 0xe, false);  // row_shr:4, banks 1-3
  r += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)r, 0x118, 0xf, 0xc, false);  // row_shr:8, banks 2-3
  r += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)r, 0x142, 0xa, 0xf, false);  // row_bcast:15 -> rows 1, 3
  r += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)r, 0x143, 0xc, 0xf, false);  // row_bcast:31 -> rows 2, 3
  return r;
}

