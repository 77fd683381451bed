// Prefill k-means kernels (gfx950): inner-product assignment on bf16 MFMA, deterministic
// inverted lists, and list-ordered segmented reductions for centroid and value sums.
// Restates cache_hub/kmeans.py (assign :6-49, update :52-80, reverse index :128-173,
// index add :176-221) with a fixed summation order instead of fp32 atomics.
#include "ri_common.h"

typedef __attribute__((address_space(3))) void* km_lds_ptr;
typedef const __attribute__((address_space(1))) void* km_glb_ptr;

// 16 bytes per lane from global memory straight into LDS: lane l lands at lds_base + 16 l
// (lds_base: byte address inside the workgroup's LDS, the same in every lane, as `base` is; `at`: the lane's byte offset).
// The wait for the data is the caller's (s_waitcnt vmcnt): issued as inline assembly so that LDS reads of other
// buffers are not made to wait for it.
__device__ __forceinline__ void km_lds_dma16(const void* base, uint32_t at, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(at), "s"(base), "s"(lds_base) : "memory", "m0");
}

// first data row of problem p: problems are `seg` consecutive N-row slices of each head
__device__ __forceinline__ size_t km_row0(int p, int seg, int64_t head_rows, int N) {
  return (size_t)(p / seg) * (size_t)head_rows + (size_t)(p % seg) * (size_t)N;
}

// Workgroups go to the eight chiplets in turn, each with an L2 of its own.  A launch over P problems of T workgroups each
// has the grid (T << sh, P >> sh), problem p = (y << sh) + x % (1 << sh), with 1 << sh the largest power of two up to eight
// that divides P: up to eight problems run beside each other, each on its own chiplets, and what the workgroups of a
// problem share (its centroids, its assignment) is fetched by as few of them as can be.  Nine iterations of 8 x 8192
// tokens, 512 centroids: 244 -> 216 us (with eight heads of 8192 tokens the keys, too, stay in the L2 of their chiplet from
// pass to pass), of 24 x 8119 420 -> 404, of 128 x 8192 1552 -> 1516, of 4 x 8120 184 -> 177; 17 x 7000 314 and 313 (an odd
// P runs as before).
static int km_together(int P) { return P % 8 == 0 ? 3 : P % 4 == 0 ? 2 : P % 2 == 0 ? 1 : 0; }
static dim3 km_grid(int T, int P) { return dim3((unsigned)T << km_together(P), P >> km_together(P)); }

// ------------------------------------------------------------------------------------
// assign: grid km_grid(ceil(N / (W * 32 * TT)), P), W waves; a wave keeps TT columns of 32
// tokens in registers for the whole kernel.  Centroid
// tiles of CT rows go through NB LDS buffers shared by all waves of the workgroup: a tile
// is requested from global memory straight into its buffer (no registers, no LDS
// stores) NB - 1 tiles ahead, one wait and one barrier per tile.
// MFMA 16x16x32: A = centroid rows, B = token columns; accumulator i of lane l is
// row (l/16)*4 + i, column l%16.  nc is a multiple of 32; the last tile may hold
// fewer sub-tiles.  (Which tiling serves which shape: km_assign_launch below.)
// Long passes are bound by what the card's power lets the matrix cores do, and a product of sixteen rows reads and writes
// half the sums per multiplication that one of 32 does: loops over registers alone hold 2.05 - 2.12 PFLOP/s against 1.75 -
// 1.86 with 32x32x16, and 8 x 131072 tokens, 8192 centroids take 1378 us against 1504 (1.60 and 1.46 PFLOP/s; the matrix
// cores were busy 73 % of the time, at a clock that fell with it).
// HALF: keys and centroids are IEEE half instead of bfloat16.
// ------------------------------------------------------------------------------------
template <int V>
__device__ __forceinline__ void km_wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(V) : "memory"); }

// (the compiler would quiet a NaN in front of its own maximum; these have none)
__device__ __forceinline__ float km_max(float a, float b) {
  float m;
  asm("v_max_f32_e32 %0, %1, %2" : "=v"(m) : "v"(a), "v"(b));
  return m;
}

typedef uint32_t km_pair __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
// o[u] (+)= a b[u]: sixteen rows with twice sixteen tokens, 32 dims.  Written out so that the sums stay where they are: left to
// the compiler every product gets another register for its sum, 64 more than there are.  Hazards are its own: two slots from a
// register move to a product that reads it (in the shadow of the product before), and, behind the last one, km_products_wait.
template <bool HALF, bool TIED, bool FIRST>
__device__ __forceinline__ void km_products(f32x4_t& o0, f32x4_t& o1, const uint4& a, const uint4& b0, const uint4& b1) {
  if (!TIED) {
    const f32x4_t c0 = FIRST ? f32x4_t{0.f, 0.f, 0.f, 0.f} : o0, c1 = FIRST ? f32x4_t{0.f, 0.f, 0.f, 0.f} : o1;
    if (HALF) {
      o0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b0), c0, 0, 0, 0);
      o1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b1), c1, 0, 0, 0);
    } else {
      o0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ri_as_bf16x8(a), ri_as_bf16x8(b0), c0, 0, 0, 0);
      o1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ri_as_bf16x8(a), ri_as_bf16x8(b1), c1, 0, 0, 0);
    }
    return;
  }
  typedef uint32_t op_t __attribute__((ext_vector_type(4)));
  const op_t x = __builtin_bit_cast(op_t, a), y0 = __builtin_bit_cast(op_t, b0), y1 = __builtin_bit_cast(op_t, b1);
#define KM_TWO(TYPE, C0, C1)                                                                                            \
  "s_nop 1\n\tv_mfma_f32_16x16x32_" TYPE " %0, %2, %3, " C0 "\n\tv_mfma_f32_16x16x32_" TYPE " %1, %2, %4, " C1
  if (FIRST) {
    if (HALF) asm volatile(KM_TWO("f16", "0", "0") : "=&v"(o0), "=&v"(o1) : "v"(x), "v"(y0), "v"(y1));
    else asm volatile(KM_TWO("bf16", "0", "0") : "=&v"(o0), "=&v"(o1) : "v"(x), "v"(y0), "v"(y1));
  } else {
    if (HALF) asm volatile(KM_TWO("f16", "%0", "%1") : "+v"(o0), "+v"(o1) : "v"(x), "v"(y0), "v"(y1));
    else asm volatile(KM_TWO("bf16", "%0", "%1") : "+v"(o0), "+v"(o1) : "v"(x), "v"(y0), "v"(y1));
  }
#undef KM_TWO
}
// eight slots from a product to whoever reads its sum: nobody does in front of this
template <int TT>
__device__ __forceinline__ void km_products_wait(f32x4_t (&o)[TT][2][2]) {
  asm volatile("s_nop 7\n\ts_nop 1");
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) asm volatile("" : "+v"(o[tt][0][0]), "+v"(o[tt][0][1]), "+v"(o[tt][1][0]), "+v"(o[tt][1][1]));
}

// base + the row, past the lane's first one in a sub-tile, of the first of a lane's eight scores (x: rows 0 .. 3, y: 16 .. 19)
// that equals m: the half that holds m is selected, then its half, down to one score.  low4 is the maximum of best and x; m is
// above best in every lane whose answer counts.  Written out because the compiler turns a select between two scores into a
// search by index.  (The hardware wants two slots between a comparison and a select that reads it.  The scores have been read
// by the maxima before: no matrix result is outstanding when this runs.)
__device__ __forceinline__ int km_first_of(const f32x4_t& x, const f32x4_t& y, float m, float low4, int base) {
  float z0, z1, z2, z3, t;
  uint64_t e, e4;
  int row;
  asm volatile(
      "v_cmp_eq_f32_e64 %6, %16, %17\n\t"
      "s_nop 1\n\t"
      "v_cndmask_b32_e64 %0, %12, %8, %6\n\t"
      "v_cndmask_b32_e64 %1, %13, %9, %6\n\t"
      "v_cndmask_b32_e64 %2, %14, %10, %6\n\t"
      "v_cndmask_b32_e64 %3, %15, %11, %6\n\t"
      "v_max_f32_e32 %4, %0, %1\n\t"
      "v_cmp_eq_f32_e64 %7, %4, %17\n\t"
      "v_cndmask_b32_e64 %5, 16, 0, %6\n\t"
      "v_add_u32_e32 %5, %18, %5\n\t"
      "v_cndmask_b32_e64 %0, %2, %0, %7\n\t"
      "v_cmp_eq_f32_e64 %6, %0, %17\n\t"
      "v_cndmask_b32_e64 %1, 2, 0, %7\n\t"
      "s_nop 0\n\t"
      "v_cndmask_b32_e64 %2, 1, 0, %6\n\t"
      "v_add3_u32 %5, %5, %1, %2"
      : "=&v"(z0), "=&v"(z1), "=&v"(z2), "=&v"(z3), "=&v"(t), "=&v"(row), "=&s"(e4), "=&s"(e)
      : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]), "v"(low4), "v"(m),
        "v"(base));
  return row;
}

// The same with the largest of the other seven scores and of what low4 and high4 started from, in `second`: what each halving
// leaves behind.
__device__ __forceinline__ int km_first_two(const f32x4_t& x, const f32x4_t& y, float m, float low4, float high4, int base,
                                            float& second) {
  float z0, z1, z2, z3, t, u;
  uint64_t e, e4;
  int row;
  asm volatile(
      "v_cmp_eq_f32_e64 %8, %18, %20\n\t"
      "s_nop 1\n\t"
      "v_cndmask_b32_e64 %0, %14, %10, %8\n\t"
      "v_cndmask_b32_e64 %1, %15, %11, %8\n\t"
      "v_cndmask_b32_e64 %2, %16, %12, %8\n\t"
      "v_cndmask_b32_e64 %3, %17, %13, %8\n\t"
      "v_cndmask_b32_e64 %6, %18, %19, %8\n\t"
      "v_max_f32_e32 %4, %0, %1\n\t"
      "v_cmp_eq_f32_e64 %9, %4, %20\n\t"
      "v_cndmask_b32_e64 %7, 16, 0, %8\n\t"
      "v_max_f32_e32 %5, %2, %3\n\t"
      "v_cndmask_b32_e64 %0, %2, %0, %9\n\t"
      "v_cmp_eq_f32_e64 %8, %0, %20\n\t"
      "v_cndmask_b32_e64 %1, %3, %1, %9\n\t"
      "v_cndmask_b32_e64 %4, %4, %5, %9\n\t"
      "v_cndmask_b32_e64 %1, %0, %1, %8\n\t"
      "v_cndmask_b32_e64 %5, 2, 0, %9\n\t"
      "v_max3_f32 %6, %6, %4, %1\n\t"
      "v_cndmask_b32_e64 %4, 1, 0, %8\n\t"
      "v_add3_u32 %7, %7, %5, %4\n\t"
      "v_add_u32_e32 %7, %21, %7"
      : "=&v"(z0), "=&v"(z1), "=&v"(z2), "=&v"(z3), "=&v"(t), "=&v"(u), "=&v"(second), "=&v"(row), "=&s"(e4), "=&s"(e)
      : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]), "v"(low4), "v"(high4), "v"(m),
        "v"(base));
  return row;
}

// ------------------------------------------------------------------------------------
// What the passes of one clustering know of each other (ri_kmeans_iterate): a pass looks only where a token's centroid can
// have changed since the one before.  A word per cluster, as the last update left it: KM_MOVED: it wrote the centroid; KM_UNIT:
// some update did, so that the centroid's norm is one; KM_FRESH: this was the first; above them the tokens of the cluster.
// ------------------------------------------------------------------------------------
#define KM_MOVED 1
#define KM_UNIT 2
#define KM_FRESH 4
#define KM_SIZE_SHIFT 3
#define KM_OPEN_WGS 768     // three to a compute unit
#define KM_OPEN_PARTS 8
#define KM_OTHERS 0x7fffffff   // in place of a centroid: another quarter's score
// How a pass goes about a problem.  KM_ALL: every centroid is scored.  KM_KEYS: most tokens came to a centroid that no update
// had written before, a key as it is, with a norm far above one; those that are left of them are scored first, and no unit
// vector scores above a token's norm.  KM_NEW: the centroids that the last update wrote are scored; of the others none but a
// token's own scores above its bound.
enum { KM_ALL, KM_KEYS, KM_NEW };
struct KmBounds {
  float* best;            // [P, N] the score of the token's centroid
  float* bound;           // [P, N] no other centroid scores above it
  const int32_t* state;   // [P, nc]
  uint8_t* touched;       // [P, nc] a token has come or gone since the last update
  const uint16_t* order;  // [P, nc] the centroids that are scored first, then the others, each ascending
  const ri_int2* plan;    // [P] KM_ALL .. KM_NEW, how many are scored first
  int32_t* open;          // [P, N] tokens of this pass that have to look at all centroids
  int32_t* open_count;    // [P]
  int32_t* partial;       // [KM_OPEN_WGS, 3, tokens of a block]
  int32_t* arrived;       // [KM_OPEN_WGS] zero between launches
  const int32_t* odd;     // [P] a centroid that an update wrote has no norm of one (see km_finish)
  int P;
};
__device__ __forceinline__ void km_settle(const KmBounds& B, int32_t* assign, size_t t, size_t first_centroid, int id, int old,
                                          float best, float bound) {
  assign[t] = id;
  B.best[t] = best;
  B.bound[t] = bound;
  if (id != old) B.touched[first_centroid + old] = B.touched[first_centroid + id] = 1;
}

// the value of the lane 32 on
__device__ __forceinline__ float km_other(float x, int hh) {
  uint32_t a, b;
  ri_lane_pair<32>(__float_as_uint(x), a, b);
  return __uint_as_float(hh ? a : b);
}

// One workgroup's turn over centroids for its tokens: W waves of TT columns of 32 tokens, which stay in registers.
// LISTED: the centroids are those at `list` (LDS), else consecutive rows.
template <int TT, int CT, int W, int NB, bool HALF, bool LISTED>
struct KmScan {
  static_assert(CT % (4 * W) == 0 && CT % 32 == 0, "a tile is whole 1 KiB wave loads and whole sub-tiles");
  static_assert(W % 4 == 0, "an instruction's first row modulo 16 is the wave's");
  static constexpr int TOKENS = W * 32 * TT;
  static constexpr int L = CT / 4 / W;   // loads of a wave per tile
  // Tokens as operands: lane: token c, dims 32 kk + 8 g.  A load whose lanes touch sixteen tokens keeps the compute unit's address
  // path busy longer than one of four whole tokens; where waves start together that is in front of the first product.  Their
  // tokens are loaded whole and turned in the wave's part of the last tile buffer, which no tile is on
  // its way to yet, 16 at a time, piece k of token t at place k ^ t of its row.  Tiles of 32 rows leave no room for sixteen
  // tokens, and other workgroups run beside: as operands.
  static constexpr int WR = CT / W;
  static constexpr bool TURN = WR == 16;
  // Operands from LDS: each is requested AHEAD steps before its own, into the register that a product has just read, across
  // sub-tiles where a tile has several.  Us with none / 2 or 4 / 3, 6 or 7 ahead: 8 x 8192 tokens, 512 centroids 8.7 / 8.2 / 8.5,
  // 4 x 8192, 512 7.5 / 7.2 / 6.9, 28 x 8192 28.2 / 27.4 / 27.5, 8 x 131072, 8192 1405 / 1378 / 1378 (and 1410 with four, where a
  // register too many leaves three workgroups to a compute unit).
  static constexpr int AHEAD = TT == 2 ? 2 : CT == 64 ? 6 : 4;

  static constexpr bool TIED = TT > 1;   // (registers are short)

  uint16_t (*sh)[CT][RI_DIM];   // [NB] tile buffers
  const uint16_t* cp;           // the problem's centroids
  const uint16_t* list;
  int nc, lane, wave, r, hh;    // r, hh: this lane's token of a column's 32, and which half's answer (merged)
  int c, g;                     // its token of sixteen, and its quarter of the products' dims and rows
  uint32_t next[L];             // LISTED: this lane's rows of the tile that is requested next
  uint4 b[TT][2][4];            // [column][sixteen tokens of it][products of 32 dims]
  float best[TT][2], second[TT][2];
  int at[TT][2];                // where best was scored: the centroid, or its place in the list

  __device__ __forceinline__ KmScan(uint16_t (*sh_c)[CT][RI_DIM], const uint16_t* centroids, int n)
      : sh(sh_c), cp(centroids), list(nullptr), nc(n), lane(threadIdx.x & 63),
        wave(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)), r(lane & 31), hh(lane >> 5), c(lane & 15), g(lane >> 4) {}

  // A tile goes from global memory straight into LDS, 16 bytes per lane and 1 KiB (four rows)
  // per wave instruction: lane l lands at byte l * 16 of the instruction's LDS window, and which
  // global piece it fetches is free, so the 16-byte pieces of row w are stored at piece ^ (w & 15):
  // the 16 lanes of a ds_read_b128 phase then hit 16 different piece positions (all 64 banks once).
  // (A wave's rows start at the same place of sixteen in every instruction, so a lane's offset never changes and the rest
  // of the address is scalar; the rows of a list are the lane's own.)
  __device__ __forceinline__ void tile_rows(int ct, int end) {
#pragma unroll
    for (int u = 0; u < L; ++u) next[u] = list[min(ct + (wave + u * W) * 4 + (lane >> 4), end - 1)];
  }
  __device__ __forceinline__ void tile_load(int ct, int buf) {
    const uint32_t piece = ((lane & 15) ^ ((wave * 4 + (lane >> 4)) & 15)) * 16;
    const uint32_t sh_base = (uint32_t)(uintptr_t)(km_lds_ptr)&sh[0][0][0];
#pragma unroll
    for (int u = 0; u < L; ++u) {
      const int row4 = (wave + u * W) * 4;      // first of the four rows of this instruction
      const uint32_t to = sh_base + (uint32_t)((buf * CT + row4) * RI_DIM * 2);
      if (LISTED) {
        km_lds_dma16(cp, next[u] * (RI_DIM * 2) + piece, to);
      } else {
        const int row = min(ct + row4, nc - 4);      // (rows past the last repeat it: the count of loads is fixed)
        km_lds_dma16(cp + (size_t)row * RI_DIM, (lane >> 4) * (RI_DIM * 2) + piece, to);
      }
    }
  }
  __device__ __forceinline__ void start(int from, int end) {
    if (LISTED) tile_rows(from, end);
#pragma unroll
    for (int t = 0; t < NB - 1; ++t) {
      tile_load(from + t * CT, t);
      if (LISTED) tile_rows(from + (t + 1) * CT, end);
    }
  }
  __device__ __forceinline__ void nothing_yet() {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        best[tt][u] = second[tt][u] = -INFINITY;
        at[tt][u] = 0;
      }
  }
  // rows t0 .. of dp, the last one `last` (open: the rows named there)
  __device__ __forceinline__ void request_tokens(const uint16_t* dp, int t0, int last, const int32_t* open = nullptr) {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int tok = min(t0 + tt * 32 + u * 16 + c, last);
        const uint16_t* q = dp + (size_t)(open ? open[tok] : tok) * RI_DIM + g * 8;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          b[tt][u][i] = TURN ? ri_ld16(dp + (size_t)min(t0 + tt * 32 + u * 16 + 4 * i + g, last) * RI_DIM + c * 8)
                             : ri_ld16(q + i * 32);
      }
  }
  // (The token registers are consumed here so that the compiler's own wait for their loads sits in front of the loop and not
  // inside it, where it would also wait for the tile in flight.)
  __device__ __forceinline__ void take_tokens() {
    uint4* const turn = reinterpret_cast<uint4*>(&sh[NB - 1][wave * WR][0]);
    km_wait_vm<(NB - 1) * L>();
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (TURN) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int row = 4 * i + g;
            turn[row * 16 + (c ^ row)] = b[tt][u][i];
          }
          ri_wave_sync();
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) b[tt][u][kk] = turn[c * 16 + ((kk * 4 + g) ^ c)];
          ri_wave_sync();   // (a wave's LDS accesses happen in order)
        }
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          asm volatile("" : "+v"(b[tt][u][kk].x), "+v"(b[tt][u][kk].y), "+v"(b[tt][u][kk].z), "+v"(b[tt][u][kk].w));
      }
  }
  // The quarters' bests so far to all of them: what is not above the best of all need not be looked for (a quarter alone finds
  // something better in about half of its sub-tiles).  Every 512 centroids, us without / with: 8 x 131072 tokens, 8192
  // centroids 1451 / 1414, 4 x 48719, 3072 116.7 / 113.0, 1 x 65536, 4096 54.9 / 52.6; every 256: 8 x 8192, 512 9.1 -> 9.4.
  __device__ __forceinline__ void share(bool track) {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float all = ri_xor_max<16>(ri_xor_max<32>(best[tt][u]));
        const bool other = all > best[tt][u];
        if (track) second[tt][u] = other ? fmaxf(second[tt][u], best[tt][u]) : second[tt][u];
        at[tt][u] = other ? KM_OTHERS : at[tt][u];
        best[tt][u] = all;
      }
  }
  // centroids (or places of the list) from .. end-1 against the tokens; track: with the second best
  __device__ __forceinline__ void score(int from, int end, bool track) {
    const uint16_t* row_at[8];   // this lane's pieces of its two rows of a sub-tile
#pragma unroll
    for (int k = 0; k < 8; ++k) row_at[k] = &sh[0][k % 2 * 16 + c][((k / 2 * 4 + g) ^ c) * 8];
    for (int ct0 = from; ct0 < end; ct0 += NB * CT) {
#pragma unroll
      for (int buf = 0; buf < NB; ++buf) {   // (unrolled: the buffer is in the offset of every LDS read)
        const int ct = ct0 + buf * CT;
        if (ct >= end) break;
        km_wait_vm<(NB - 2) * L>();   // this tile's loads of this wave have landed ...
        asm volatile("s_barrier" ::: "memory");   // ... and every wave's; and every wave is done with the tile before
        tile_load(ct + (NB - 1) * CT, buf == 0 ? NB - 1 : buf - 1);
        if (LISTED) tile_rows(ct + NB * CT, end);
        uint4 rows[AHEAD ? AHEAD : 1];
        const auto operand = [&](int k) {
          return *reinterpret_cast<const uint4*>(row_at[k % 8] + (buf * CT + k / 8 * 32) * RI_DIM);
        };
        if (AHEAD) {
#pragma unroll
          for (int kk = 0; kk < AHEAD; ++kk) rows[kk] = operand(kk);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int half = 0; half < CT / 32; ++half) {
          if (ct + half * 32 < end) {  // uniform: only the last tile can lack sub-tiles
            f32x4_t acc[TT][2][2];
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) {
              const int k = half * 8 + kk;
              const uint4 a = AHEAD ? rows[k % (AHEAD ? AHEAD : 1)] : operand(k);
#pragma unroll
              for (int tt = 0; tt < TT; ++tt) {
                if (kk < 2)
                  km_products<HALF, TIED, true>(acc[tt][0][kk % 2], acc[tt][1][kk % 2], a, b[tt][0][kk / 2], b[tt][1][kk / 2]);
                else
                  km_products<HALF, TIED, false>(acc[tt][0][kk % 2], acc[tt][1][kk % 2], a, b[tt][0][kk / 2], b[tt][1][kk / 2]);
              }
              if (AHEAD) {
                if (k + AHEAD < CT / 4) rows[k % (AHEAD ? AHEAD : 1)] = operand(k + AHEAD);
                __builtin_amdgcn_sched_barrier(0);
              }
            }
            if (TIED) km_products_wait<TT>(acc);
            if (LISTED && ct + half * 32 + 32 > end) {   // uniform: rows past the last score nothing
              const int left = end - (ct + half * 32) - g * 4;
#pragma unroll
              for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                  for (int i = 0; i < 8; ++i)
                    acc[tt][u][i / 4][i % 4] = i / 4 * 16 + i % 4 < left ? acc[tt][u][i / 4][i % 4] : -INFINITY;
            }
            // argmax epilogue: the lane's eight scores are in ascending row order, so the first score
            // equal to their maximum is the lowest row; the index search only runs when some lane
            // of the wave improves on its best (about half of the sub-tiles of a full-size pass)
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
              for (int u = 0; u < 2; ++u) {
                // (from a score seen before, which is no NaN.  From the second best where that is wanted: it then is the larger
                // of the two wherever the best stays.)
                const f32x4_t &x = acc[tt][u][0], &y = acc[tt][u][1];
                float &top = best[tt][u], &next_best = second[tt][u];
                const float seen = track ? next_best : top;
                const float low4 = fmaxf(fmaxf(fmaxf(fmaxf(seen, x[0]), x[1]), x[2]), x[3]);
                if (!track) {
                  const float m = fmaxf(fmaxf(fmaxf(fmaxf(low4, y[0]), y[1]), y[2]), y[3]);
                  const bool upd = m > top;
                  if (__builtin_amdgcn_ballot_w64(upd) != 0ull) {
                    const int k = km_first_of(x, y, m, low4, g * 4 + ct + half * 32);
                    at[tt][u] = upd ? k : at[tt][u];
                  }
                  top = m;   // (the same where no lane improves)
                } else {
                  const float high4 = fmaxf(fmaxf(fmaxf(fmaxf(seen, y[0]), y[1]), y[2]), y[3]);
                  const float m = km_max(low4, high4);
                  const bool upd = m > top;
                  if (__builtin_amdgcn_ballot_w64(upd) != 0ull) {
                    float s;
                    const int k = km_first_two(x, y, m, low4, high4, g * 4 + ct + half * 32, s);
                    s = km_max(s, top);
                    next_best = upd ? s : m;
                    at[tt][u] = upd ? k : at[tt][u];
                    top = upd ? m : top;
                  } else {
                    next_best = m;
                  }
                }
              }
          }
        }
        if (((ct + CT - from) & 511) == 0 && ct + CT < end) share(track);   // (a second turn starts anywhere in the list)
      }
    }
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
      for (int u = 0; u < 2; ++u) asm volatile("" : "+v"(best[tt][u]), "+v"(at[tt][u]));   // (one register each, whichever way out)
    km_wait_vm<0>();   // (no load may land in LDS that is no longer this workgroup's, or that another turn fills)
  }
  // The quarters of a wave have scored every other four rows for the same tokens: best, its place and second best of all of them
  // for token r of a column, in both halves.  (The first exchange brings each row of lanes two quarters' answers for the
  // sixteen tokens that are its own.)
  __device__ __forceinline__ void merged(int tt, float& top, int& place, float& next_best) {
    const auto pair = [](uint32_t x, uint32_t y) { return __builtin_bit_cast(km_pair, __builtin_amdgcn_permlane16_swap(x, y, false, false)); };
    const km_pair pb = pair(__float_as_uint(best[tt][0]), __float_as_uint(best[tt][1])), pa = pair(at[tt][0], at[tt][1]),
                  ps = pair(__float_as_uint(second[tt][0]), __float_as_uint(second[tt][1]));
    const auto own = [](uint32_t x, uint32_t i) { return i == KM_OTHERS ? -INFINITY : __uint_as_float(x); };
    const auto first = [](float x, int i, float y, int j) { return y > x || (y == x && j < i); };   // the other one's
    const float x0 = own(pb.x, pa.x), x1 = own(pb.y, pa.y);
    const bool o = first(x0, (int)pa.x, x1, (int)pa.y);
    const float b = o ? x1 : x0, s = fmaxf(fminf(x0, x1), fmaxf(__uint_as_float(ps.x), __uint_as_float(ps.y)));
    const int a = o ? (int)pa.y : (int)pa.x;
    const float ob = km_other(b, hh);
    const int oa = __float_as_int(km_other(__int_as_float(a), hh));
    const bool other = first(b, a, ob, oa);
    next_best = fmaxf(fminf(ob, b), ri_xor_max<32>(s));
    top = other ? ob : b;
    place = other ? oa : a;
  }
};

// Between the passes of ri_kmeans_iterate a problem's assignment lies as 16-bit words in the first half of its row of `assign`,
// where km_direct_kernel takes it from (narrow; figures there).
#define KM_NARROW 4   // beside the shift of km_grid in the kernels' `shape`
__device__ __forceinline__ void km_put_place(int32_t* row, int tok, int place, int narrow) {
  if (narrow) reinterpret_cast<uint16_t*>(row)[tok] = (uint16_t)place;
  else row[tok] = place;
}

template <int TT, int CT, int W, int NB, bool HALF>
__global__ __launch_bounds__(W * 64) void km_assign_kernel(const uint16_t* __restrict__ data, const uint16_t* __restrict__ cent,
                                                           int32_t* __restrict__ assign, int N, int nc, int seg,
                                                           int64_t head_rows, int shape) {
  typedef KmScan<TT, CT, W, NB, HALF, false> Scan;
  __shared__ __attribute__((aligned(1024))) uint16_t sh_c[NB][CT][RI_DIM];
  const int sh = shape & 3;
  const int p = (blockIdx.y << sh) + (blockIdx.x & ((1 << sh) - 1));
  Scan s(sh_c, cent + (size_t)p * nc * RI_DIM, nc);
  const int t0 = (blockIdx.x >> sh) * Scan::TOKENS + s.wave * (32 * TT);
  s.request_tokens(data + km_row0(p, seg, head_rows, N) * RI_DIM, t0, N - 1);
  s.start(0, nc);
  s.take_tokens();
  s.nothing_yet();
  s.score(0, nc, false);
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) {
    float top, second;
    int place;
    s.merged(tt, top, place, second);
    const int tok = t0 + tt * 32 + s.r;
    if (s.hh == 0 && tok < N) km_put_place(assign + (size_t)p * N, tok, place, shape & KM_NARROW);
  }
}

// base + the row, past the lane's first one in a sub-tile, of the first of a lane's sixteen scores that equals m, found as
// km_first_of finds one of eight.  low8 and low4 are the maxima of best and the first eight and four scores, high4 of best and
// scores 8 .. 11.
__device__ __forceinline__ int km_first_of16(const f32x16_t& x, float m, float best, float low8, float low4, float high4,
                                             int base) {
  float y0, y1, y2, y3, y4, y5, y6, y7, t;
  uint64_t e, e8;
  int row;
  asm volatile(
      "v_cmp_eq_f32_e64 %8, %25, %26\n\t"
      "s_nop 1\n\t"
      "v_cndmask_b32_e64 %0, %17, %9, %8\n\t"
      "v_cndmask_b32_e64 %1, %18, %10, %8\n\t"
      "v_cndmask_b32_e64 %2, %19, %11, %8\n\t"
      "v_cndmask_b32_e64 %3, %20, %12, %8\n\t"
      "v_cndmask_b32_e64 %4, %21, %13, %8\n\t"
      "v_cndmask_b32_e64 %5, %22, %14, %8\n\t"
      "v_cndmask_b32_e64 %6, %23, %15, %8\n\t"
      "v_cndmask_b32_e64 %7, %24, %16, %8"
      : "=&v"(y0), "=&v"(y1), "=&v"(y2), "=&v"(y3), "=&v"(y4), "=&v"(y5), "=&v"(y6), "=&v"(y7), "=&s"(e8)
      : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]), "v"(x[8]), "v"(x[9]),
        "v"(x[10]), "v"(x[11]), "v"(x[12]), "v"(x[13]), "v"(x[14]), "v"(x[15]), "v"(low8), "v"(m));
  // (sum i is row (i / 4) * 8 + i % 4)
  asm volatile(
      "v_cndmask_b32_e64 %8, %13, %12, %10\n\t"
      "v_cmp_eq_f32_e64 %11, %8, %15\n\t"
      "v_cndmask_b32_e64 %9, 16, 0, %10\n\t"
      "s_nop 0\n\t"
      "v_cndmask_b32_e64 %0, %4, %0, %11\n\t"
      "v_cndmask_b32_e64 %1, %5, %1, %11\n\t"
      "v_cndmask_b32_e64 %2, %6, %2, %11\n\t"
      "v_cndmask_b32_e64 %3, %7, %3, %11\n\t"
      "v_max3_f32 %8, %14, %0, %1\n\t"
      "v_cmp_eq_f32_e64 %10, %8, %15\n\t"
      "v_cndmask_b32_e64 %4, 8, 0, %11\n\t"
      "s_nop 0\n\t"
      "v_cndmask_b32_e64 %0, %2, %0, %10\n\t"
      "v_cmp_eq_f32_e64 %11, %0, %15\n\t"
      "v_cndmask_b32_e64 %5, 2, 0, %10\n\t"
      "v_add3_u32 %9, %9, %4, %5\n\t"
      "v_cndmask_b32_e64 %6, 1, 0, %11\n\t"
      "v_add3_u32 %9, %9, %6, %16"
      : "+v"(y0), "+v"(y1), "+v"(y2), "+v"(y3), "+v"(y4), "+v"(y5), "+v"(y6), "+v"(y7), "=&v"(t), "=&v"(row), "+s"(e8),
        "=&s"(e)
      : "v"(low4), "v"(high4), "v"(best), "v"(m), "v"(base));
  return row;
}

// The same pass for launches that leave many compute units without work: there power bounds nothing, and half as many products,
// each of 32 rows with 32 tokens, and one search of sixteen scores are fewer instructions than two of each with eight.  (Figures
// at km_assign_launch.)  Eight waves of 32 tokens, tiles of 128 rows in two buffers; a lane has token r, dims 16 kk + 8 hh.
template <bool HALF>
__global__ __launch_bounds__(512) void km_assign_few_kernel(const uint16_t* __restrict__ data, const uint16_t* __restrict__ cent,
                                                            int32_t* __restrict__ assign, int N, int nc, int seg,
                                                            int64_t head_rows, int shape) {
  constexpr int CT = 128, AHEAD = 8;
  typedef KmScan<1, CT, 8, 2, HALF, false> Scan;
  static_assert(Scan::TURN && Scan::WR == 16, "room for sixteen tokens of a wave");
  __shared__ __attribute__((aligned(1024))) uint16_t sh_c[2][CT][RI_DIM];
  const int sh = shape & 3;
  const int p = (blockIdx.y << sh) + (blockIdx.x & ((1 << sh) - 1));
  Scan s(sh_c, cent + (size_t)p * nc * RI_DIM, nc);
  const int t0 = (blockIdx.x >> sh) * Scan::TOKENS + s.wave * 32, r = s.r, hh = s.hh;
  const uint16_t* dp = data + km_row0(p, seg, head_rows, N) * RI_DIM;
  uint4 in[8], b[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) in[i] = ri_ld16(dp + (size_t)min(t0 + 4 * i + s.g, N - 1) * RI_DIM + s.c * 8);
  s.start(0, nc);
  uint4* const turn = reinterpret_cast<uint4*>(&sh_c[1][s.wave * Scan::WR][0]);
  km_wait_vm<Scan::L>();
#pragma unroll
  for (int w = 0; w < 2; ++w) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * i + s.g;
      turn[row * 16 + (s.c ^ row)] = in[w * 4 + i];
    }
    ri_wave_sync();
    if (r >> 4 == w) {
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) b[kk] = turn[s.c * 16 + ((kk * 2 + hh) ^ s.c)];
    }
    ri_wave_sync();   // (a wave's LDS accesses happen in order)
  }
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) asm volatile("" : "+v"(b[kk].x), "+v"(b[kk].y), "+v"(b[kk].z), "+v"(b[kk].w));
  float best = -INFINITY;
  int at = 0;
  const uint16_t* row_at[8];   // this lane's pieces of its row of a sub-tile
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) row_at[kk] = &sh_c[0][r][((kk * 2 + hh) ^ s.c) * 8];
  for (int ct0 = 0; ct0 < nc; ct0 += 2 * CT) {
#pragma unroll
    for (int buf = 0; buf < 2; ++buf) {   // (unrolled: the buffer is in the offset of every LDS read)
      const int ct = ct0 + buf * CT;
      if (ct >= nc) break;
      km_wait_vm<0>();   // this tile's loads of this wave have landed ...
      asm volatile("s_barrier" ::: "memory");   // ... and every wave's; and every wave is done with the tile before
      s.tile_load(ct + CT, 1 - buf);
      uint4 rows[AHEAD];
      const auto operand = [&](int k) {
        return *reinterpret_cast<const uint4*>(row_at[k % 8] + (buf * CT + k / 8 * 32) * RI_DIM);
      };
#pragma unroll
      for (int kk = 0; kk < AHEAD; ++kk) rows[kk] = operand(kk);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int half = 0; half < CT / 32; ++half) {
        if (ct + half * 32 < nc) {  // uniform: only the last tile can lack sub-tiles
          f32x16_t acc;
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
          for (int kk = 0; kk < 8; ++kk) {
            const int k = half * 8 + kk;
            const uint4 a = rows[k % AHEAD];
            acc = HALF ? __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                                __builtin_bit_cast(f16x8_t, b[kk]), acc, 0, 0, 0)
                       : __builtin_amdgcn_mfma_f32_32x32x16_bf16(ri_as_bf16x8(a), ri_as_bf16x8(b[kk]), acc, 0, 0, 0);
            if (k + AHEAD < CT / 4) rows[k % AHEAD] = operand(k + AHEAD);
            __builtin_amdgcn_sched_barrier(0);
          }
          float low8 = best, high8 = best, low4 = best, high4 = best;   // (from the best so far, which is no NaN)
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            low8 = fmaxf(low8, acc[i]);
            high8 = fmaxf(high8, acc[8 + i]);
            if (i == 3) low4 = low8, high4 = high8;
          }
          const float m = km_max(low8, high8);
          const bool upd = m > best;
          if (__builtin_amdgcn_ballot_w64(upd) != 0ull) {
            const int k = km_first_of16(acc, m, best, low8, low4, high4, hh * 4 + ct + half * 32);
            at = upd ? k : at;
            best = m;
          }
        }
      }
    }
  }
  km_wait_vm<0>();   // (no load may land in LDS that is no longer this workgroup's)
  const float other = km_other(best, hh);
  const int other_at = __float_as_int(km_other(__int_as_float(at), hh));
  if (other > best || (other == best && other_at < at)) at = other_at;
  const int tok = t0 + r;
  if (hh == 0 && tok < N) km_put_place(assign + (size_t)p * N, tok, at, shape & KM_NARROW);
}

// A pass of a clustering that knows the pass before (KmBounds), grid (ceil(N / TOKENS), P).  The clusters that no token has
// joined or left keep their centroids, most keys win against unit vectors by their norm, and a token whose second best score
// is known needs no more than the centroids that were written since: the same scores, hence the same assignment, of far fewer
// products.  8 x 131072 tokens, 8192 centroids, us of ten passes: 10 x 1383 -> 1383 (all), 1252, 569, 103 and 69 + 400 (keys
// left: 81, 38, 4 and 0.1 %; a fifth of the tokens is left open by the last), 1684 (all, with the second best: its search is
// what a full pass loses by it), 1395 + 69, 678 + 62, 438 + 55 and 313 + 43 (90, 46, 28 and 19 % of the centroids written, 3 to
// 1.6 % of the tokens open).  Two columns of tokens and small tiles: with a short list the load of the tokens is the launch, and
// three workgroups per compute unit overlap it (19 % of 8192, with products of 32 rows: 324, of which 55 are the bytes; four
// columns, 8 waves: 393; one column: 450).  The problems' workgroups are dealt over all chiplets, unlike those of a plain pass: problems take unequal
// time (12943 -> 14059 with a problem to a chiplet).
template <int TT, int CT, int W, int NB, bool HALF>
__global__ __launch_bounds__(W * 64, TT == 2 ? 3 : 2) void km_assign_again_kernel(
    const uint16_t* __restrict__ data, const uint16_t* __restrict__ cent, int32_t* __restrict__ assign, int N, int nc, int seg,
    int64_t head_rows, KmBounds B) {
  typedef KmScan<TT, CT, W, NB, HALF, true> Scan;
  __shared__ __attribute__((aligned(1024))) uint16_t sh_c[NB][CT][RI_DIM];
  __shared__ int sh_open[W + 1];   // uncertain tokens of every wave, then where the workgroup's go
  extern __shared__ __attribute__((aligned(16))) uint16_t list[];   // the centroids in the order they are scored
  const int p = blockIdx.y, wg0 = blockIdx.x * Scan::TOKENS;
  const size_t first_token = (size_t)p * N, first_centroid = (size_t)p * nc;
  Scan s(sh_c, cent + first_centroid * RI_DIM, nc);
  s.list = list;
  const int t0 = wg0 + s.wave * (32 * TT);
  s.request_tokens(data + km_row0(p, seg, head_rows, N) * RI_DIM, t0, N - 1);
  const int mode = B.plan[p].x, n1 = B.plan[p].y;
  const uint4* const order = reinterpret_cast<const uint4*>(B.order + first_centroid);
#pragma unroll 4
  for (int i = threadIdx.x; i < nc / 8; i += W * 64) reinterpret_cast<uint4*>(list)[i] = order[i];
  s.nothing_yet();
  if (mode == KM_NEW) {   // (scores up to the bound are of no interest)
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        s.best[tt][u] = s.second[tt][u] = B.bound[first_token + min(t0 + tt * 32 + u * 16 + s.c, N - 1)];
        s.at[tt][u] = nc - 1;   // (unless one does: uncertain below)
      }
  }
  __syncthreads();
  s.start(0, max(n1, 1));
  s.take_tokens();
  bool track = mode != KM_KEYS;
  for (int part = 0, from = 0, end = n1;; part = 1, from = mode == KM_KEYS ? n1 : 0, end = nc) {
    s.score(from, end, track);
    const bool whole = part == 1 || mode == KM_ALL;
    int rr = s.r;
    asm volatile("" : "+v"(rr));   // (what follows from it is computed here and not kept through the loop)
    int id[TT], old[TT];
    float top[TT], bound[TT];
    uint32_t sure = 0;
    int uncertain = 0;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      int place;
      s.merged(tt, top[tt], place, bound[tt]);
      const int tok = t0 + tt * 32 + rr;
      const size_t t = first_token + min(tok, N - 1);
      old[tt] = assign[t];
      id[tt] = top[tt] > -INFINITY ? list[place] : 0;
      bool ok = true;
      if (part == 1) {
        ok = !(top[tt] == bound[tt]) || top[tt] == -INFINITY;   // (a tie across the two turns: not in the order of ids)
      } else if (mode == KM_NEW) {
        // its own centroid, where that was not written, scores what it did
        const float limit = B.bound[t], own = B.best[t];
        if (!(B.state[first_centroid + old[tt]] & KM_MOVED)) {
          const bool stay = own > top[tt] || (own == top[tt] && old[tt] < id[tt]);
          bound[tt] = fmaxf(bound[tt], fminf(own, top[tt]));
          id[tt] = stay ? old[tt] : id[tt];
          top[tt] = stay ? own : top[tt];
        }
        ok = top[tt] > limit;
      } else if (mode == KM_KEYS) {
        // |x c| <= |x| |c|, and a centroid that an update has written is a unit vector rounded to 16 bits (and this sum,
        // like the scores, to 32: far inside the hundredth)
        float part_sq[2] = {0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int kk = 0; kk < 16; ++kk) {
            float lo, hi;
            uint32_t word = (&s.b[tt][u][kk / 4].x)[kk % 4];
            asm volatile("" : "+v"(word));   // (here, and not ahead of the loop: the registers are full)
            ri_unpack2<HALF>(word, lo, hi);
            part_sq[u] = fmaf(lo, lo, fmaf(hi, hi, part_sq[u]));
          }
        const km_pair sq = __builtin_bit_cast(km_pair, __builtin_amdgcn_permlane16_swap(   // (as in `merged`)
                               __float_as_uint(part_sq[0]), __float_as_uint(part_sq[1]), false, false));
        ok = top[tt] > 1.01f * sqrtf(ri_xor_sum<32>(__uint_as_float(sq.x) + __uint_as_float(sq.y))) + 1e-17f && !B.odd[p];   // (1e-17: squares too small for a float)
      }
      __builtin_amdgcn_sched_barrier(0);
      if (ok) sure |= 1u << tt;
      uncertain += __popcll(__builtin_amdgcn_ballot_w64(!ok && s.hh == 0 && tok < N));
    }
    // Where most of a workgroup's tokens are uncertain it looks at the other centroids itself; else one addition in memory
    // reserves the places of all of its open tokens (one address takes an addition every 40 ns or so: one per wave and column
    // was 20 us of 8 x 20000 tokens).
    if (s.lane == 0) sh_open[s.wave] = uncertain;
    __syncthreads();
    int all = 0, at = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      if (w < s.wave) at += sh_open[w];
      all += sh_open[w];
    }
    all = __builtin_amdgcn_readfirstlane(all);
    if (!whole) {
      if (4 * all > 3 * min(Scan::TOKENS, N - wg0)) {
        __syncthreads();
        track = true;
        if (mode == KM_NEW) s.nothing_yet();
        s.start(mode == KM_KEYS ? n1 : 0, nc);
        continue;
      }
    }
    if (all) {
      if (threadIdx.x == 0) sh_open[W] = atomicAdd(&B.open_count[p], all);
      __syncthreads();
      at += sh_open[W];
    }
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      const int tok = t0 + tt * 32 + rr;
      const bool mine = s.hh == 0 && tok < N, ok = sure >> tt & 1;
      if (mine && ok) km_settle(B, assign, first_token + tok, first_centroid, id[tt], old[tt], top[tt], bound[tt]);
      const uint64_t left = __builtin_amdgcn_ballot_w64(mine && !ok);
      if (mine && !ok) B.open[first_token + at + __popcll(left & ((1ull << s.lane) - 1ull))] = tok;
      at += __popcll(left);
    }
    return;
  }
}

template <bool HALF>
using KmOpenScan = KmScan<2, 32, 4, 4, HALF, false>;

// The tokens that a pass left open (a few in a hundred), against all centroids, grid KM_OPEN_WGS: blocks of a problem's open tokens, each cut into
// as many parts of the centroids as there are workgroups for; the last of a block's parts to arrive puts them together.
// (What the others wrote reaches it by write-through stores that are complete before they arrive.)  Bound by the matrix cores
// where there are many (210000 of 8 x 131072, 8192 centroids: 400 us), else by its chain: 400 tokens of
// eight problems, 640 centroids: 10.5 us, 17 while the parts were put together one after the other.
template <bool HALF>
__global__ __launch_bounds__(256) void km_assign_open_kernel(const uint16_t* __restrict__ data,
                                                                const uint16_t* __restrict__ cent, int32_t* __restrict__ assign,
                                                                int N, int nc, int seg, int64_t head_rows, KmBounds B) {
  typedef KmOpenScan<HALF> Scan;
  constexpr int TT = 2;
  static_assert(!Scan::TURN && Scan::TOKENS == 4 * 32 * TT, "tokens by name");
  __shared__ __attribute__((aligned(1024))) uint16_t sh_c[4][32][RI_DIM];
  __shared__ int sh_last;
  const int lane = threadIdx.x & 63;
  // blocks of every problem, a lane per problem
  const int blocks = lane < B.P ? (B.open_count[lane] + Scan::TOKENS - 1) / Scan::TOKENS : 0;
  const int incl = (int)ri_wave_incl_scan((uint32_t)blocks), items = __builtin_amdgcn_readlane(incl, 63);
  if (items == 0) return;
  const int parts = min(max((int)gridDim.x / items, 1), min(KM_OPEN_PARTS, nc / 32));
  for (int w = blockIdx.x; w < items * parts; w += gridDim.x) {
    const int item = w / parts, part = w % parts;
    const int p = __ffsll((long long)__builtin_amdgcn_ballot_w64(incl > item)) - 1;
    const int block = item - (__builtin_amdgcn_readlane(incl, p) - __builtin_amdgcn_readlane(blocks, p));
    const size_t first_token = (size_t)p * N, first_centroid = (size_t)p * nc;
    const int32_t* const open = B.open + first_token;
    const int n = __builtin_amdgcn_readfirstlane(B.open_count[p]);
    const int from = (int)((int64_t)(nc / 32) * part / parts) * 32, end = (int)((int64_t)(nc / 32) * (part + 1) / parts) * 32;
    Scan s(sh_c, cent + first_centroid * RI_DIM, nc);
    const int t0 = block * Scan::TOKENS + s.wave * (32 * TT);
    s.request_tokens(data + km_row0(p, seg, head_rows, N) * RI_DIM, t0, n - 1, open);
    s.start(from, end);
    s.take_tokens();
    s.nothing_yet();
    s.score(from, end, true);
    int last = 1;
    int32_t* const mine = B.partial + (size_t)w * 3 * Scan::TOKENS + s.wave * (32 * TT) + s.r;
    if (parts > 1) {
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        float top, second;
        int place;
        s.merged(tt, top, place, second);
        if (s.hh == 0) {
          __hip_atomic_store(mine + tt * 32, __float_as_int(top), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(mine + tt * 32 + Scan::TOKENS, __float_as_int(second), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(mine + tt * 32 + 2 * Scan::TOKENS, place, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      km_wait_vm<0>();
      __syncthreads();
      if (threadIdx.x == 0) {
        int32_t* const arrived = B.arrived + item;
        last = __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == parts - 1;
        if (last) __hip_atomic_store(arrived, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sh_last = last;
      }
      __syncthreads();
      last = __builtin_amdgcn_readfirstlane(sh_last);
    }
    if (last) {
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        float top, second;
        int place;
        s.merged(tt, top, place, second);
        const int at = t0 + tt * 32 + s.r;
        if (s.hh == 0 && at < n) {
          if (parts > 1) {
            top = second = -INFINITY;
            place = 0;
            int32_t v[KM_OPEN_PARTS][3];   // (all on their way before the first is looked at)
#pragma unroll
            for (int q = 0; q < KM_OPEN_PARTS; ++q)
#pragma unroll
              for (int k = 0; k < 3; ++k)
                v[q][k] = __hip_atomic_load(mine + ((ptrdiff_t)(min(q, parts - 1) - part) * 3 + k) * Scan::TOKENS + tt * 32,
                                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int q = 0; q < KM_OPEN_PARTS; ++q) {   // (ascending centroids: a tie stays where it is)
              if (q >= parts) break;
              const float a = __int_as_float(v[q][0]);
              second = fmaxf(fmaxf(second, __int_as_float(v[q][1])), fminf(top, a));
              place = a > top ? v[q][2] : place;
              top = fmaxf(top, a);
            }
          }
          const int tok = open[at];
          km_settle(B, assign, first_token + tok, first_centroid, place, assign[first_token + tok], top, second);
        }
      }
    }
    __syncthreads();   // (the tile buffers, and sh_last)
  }
}

// ------------------------------------------------------------------------------------
// inverted lists
// ------------------------------------------------------------------------------------
// Inverted lists are a stable sort of the token ids by cluster id.  Ids of at most 9 bits take one counting pass, two
// launches, three with a large table: per-chunk digit histograms (KM_SORT_CHUNK tokens, LDS counters), an exclusive scan of the
// [digit][chunk] table per problem, and a scatter in which every wave walks its part of a chunk in token order, ranks equal digits
// inside each 64-token round with ballots and keeps running positions in LDS.  Longer ids take that pass over their upper
// digit and one launch that sorts every bucket of it by the lower digit in a workgroup and writes offsets and counts on
// the way.  Stability makes every list ascending without any per-list sort, and no global atomics are involved, so the
// result does not depend on scheduling.  Every launch is a short serial chain, so chunks are shared by four waves and
// tables are read in one round trip (all launches of 4 x 48787 tokens, 3040 clusters: 16.0 us; two passes of three
// launches with a wave per chunk, a search of the bounds and their differences: 38.5; 8 x 131072, 8192: 25.2 and 62.8).
#define KM_SORT_CHUNK 1024
#define KM_SORT_ROUNDS (KM_SORT_CHUNK / 256)   // 64-token rounds of each of the four waves of a chunk
#define KM_SORT_MAX_BINS 512

__device__ __forceinline__ void km_wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// chunk_hist[p][digit][chunk] (by_chunk: [p][chunk][digit]) = tokens of the chunk whose key has that digit; a workgroup per chunk
__global__ __launch_bounds__(256) void km_sort_hist_kernel(const int32_t* __restrict__ keys,
                                                           int32_t* __restrict__ chunk_hist, int N, int nchunks,
                                                           int shift, int bits, bool by_chunk) {
  __shared__ int32_t h[KM_SORT_MAX_BINS];
  const int p = blockIdx.y, chunk = blockIdx.x, bins = 1 << bits;
  const int i0 = chunk * KM_SORT_CHUNK + threadIdx.x;
  int32_t k[KM_SORT_ROUNDS];
#pragma unroll
  for (int r = 0; r < KM_SORT_ROUNDS; ++r) k[r] = keys[(size_t)p * N + min(i0 + r * 256, N - 1)];
  for (int b = threadIdx.x; b < bins; b += 256) h[b] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < KM_SORT_ROUNDS; ++r)
    if (i0 + r * 256 < N) atomicAdd(&h[(k[r] >> shift) & (bins - 1)], 1);
  __syncthreads();
  for (int b = threadIdx.x; b < bins; b += 256)
    chunk_hist[by_chunk ? ((size_t)p * nchunks + chunk) * bins + b : ((size_t)p * bins + b) * nchunks + chunk] = h[b];
}

// in-place exclusive prefix sum over the n = bins * nchunks entries of each problem.
// When the digit of this pass is the whole cluster id (offsets != nullptr), the scanned entry of
// (digit c, chunk 0) is where list c starts: the CSR offsets and the counts are written here.
__global__ __launch_bounds__(1024) void km_sort_scan_kernel(int32_t* __restrict__ chunk_hist, int n,
                                                            int32_t* __restrict__ offsets,
                                                            int32_t* __restrict__ counts, int nchunks, int nc,
                                                            int N) {
  __shared__ int32_t sh_w[16];
  __shared__ int32_t sh_carry;
  int32_t* a = chunk_hist + (size_t)blockIdx.x * n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) sh_carry = 0;
  __syncthreads();
  // sixteen rows of 64 entries per wave and round: a table of 128 digits and 128 chunks is one round trip
  for (int base = 0; base < n; base += 16 * 1024) {
    const int i0 = base + wave * 1024 + lane;
    int32_t v[16], x[16], run = 0;
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = a[min(i0 + u * 64, n - 1)];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      if (i0 + u * 64 >= n) v[u] = 0;
      const int32_t inc = (int32_t)ri_wave_incl_scan((uint32_t)v[u]);
      x[u] = run + inc - v[u];
      run += __builtin_amdgcn_readlane(inc, 63);
    }
    if (lane == 0) sh_w[wave] = run;
    __syncthreads();
    int32_t ex = sh_carry, tot = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int32_t y = sh_w[w];
      if (w < wave) ex += y;
      tot += y;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u)
      if (i0 + u * 64 < n) a[i0 + u * 64] = ex + x[u];
    __syncthreads();
    if (threadIdx.x == 0) sh_carry += tot;
    __syncthreads();
  }
  if (!offsets) return;
  // (the barrier above made the scanned table visible to the whole workgroup)
  int32_t* off = offsets + (size_t)blockIdx.x * (nc + 1);
  for (int c = threadIdx.x; c <= nc; c += 1024) {
    const int32_t lo = (c < nc) ? a[(size_t)c * nchunks] : N;
    off[c] = lo;
    if (c < nc) {
      const int32_t hi = (c + 1 < nc) ? a[(size_t)(c + 1) * nchunks] : N;
      counts[(size_t)blockIdx.x * nc + c] = hi - lo;
    }
  }
}

// What a scatter without a scan in front of it writes besides: where every digit starts (starts), or, of whole ids, offsets and
// counts.
struct KmFirsts {
  int32_t *starts, *offsets, *counts;
  int nc;
};
// Up to KM_SORT_TABLE counts the scatter's workgroups add up the table themselves, which is one round trip more for each
// where the scan is a launch of one workgroup per problem; the first chunk's writes where the digits start.
// at: [bins] where this chunk's tokens of each digit go.  16 <= bins / 4 <= 128 pieces to a row of the table, sixteen per thread.
#define KM_SORT_TABLE 16384
__device__ __forceinline__ void km_sort_places(const int32_t* __restrict__ table, int32_t* at, int p, int chunk, int nchunks,
                                               int bits, int N, const KmFirsts& F) {
  __shared__ __attribute__((aligned(16))) int32_t sh_all[KM_SORT_TABLE / 16], sh_before[KM_SORT_TABLE / 16];
  __shared__ int32_t sh_w[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, bins = 1 << bits;
  const int row0 = tid >> (bits - 2), quad = tid & ((bins >> 2) - 1), rows = 1024 >> bits;   // rows that the workgroup reads at a time
  const int4* const in = reinterpret_cast<const int4*>(table + (size_t)p * nchunks * bins) + quad;
  int4 v[16], all = make_int4(0, 0, 0, 0), before = all;
#pragma unroll
  for (int u = 0; u < 16; ++u) v[u] = in[(size_t)min(row0 + u * rows, nchunks - 1) << (bits - 2)];
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int row = row0 + u * rows, there = row < nchunks ? -1 : 0, ahead = row < chunk ? -1 : 0;
    all.x += v[u].x & there; all.y += v[u].y & there; all.z += v[u].z & there; all.w += v[u].w & there;
    before.x += v[u].x & ahead; before.y += v[u].y & ahead; before.z += v[u].z & ahead; before.w += v[u].w & ahead;
  }
  *reinterpret_cast<int4*>(&sh_all[tid * 4]) = all;   // [row0][digit]
  *reinterpret_cast<int4*>(&sh_before[tid * 4]) = before;
  __syncthreads();
  // a thread's digits: tid, or with 512 of them 2 tid and the next
  const int each = bits == 9 ? 2 : 1, b0 = tid * each;
  int32_t n[2] = {0, 0}, ex[2] = {0, 0};
  for (int e = 0; e < each; ++e)
    if (b0 + e < bins)
      for (int r = 0; r < rows; ++r) {
        n[e] += sh_all[(r << bits) + b0 + e];
        ex[e] += sh_before[(r << bits) + b0 + e];
      }
  const int inc = (int)ri_wave_incl_scan((uint32_t)(n[0] + n[1]));
  if (lane == 63) sh_w[wave] = inc;
  __syncthreads();
  int start = inc - n[0] - n[1];
#pragma unroll
  for (int w = 0; w < 4; ++w) start += w < wave ? sh_w[w] : 0;
  for (int e = 0; e < each; ++e) {
    const int b = b0 + e;
    if (b < bins) at[b] = start + ex[e];
    if (chunk == 0) {
      if (F.starts && b < bins) F.starts[p * bins + b] = start;
      if (F.offsets && b < F.nc) {
        F.offsets[(size_t)p * (F.nc + 1) + b] = start;
        F.counts[(size_t)p * F.nc + b] = n[e];
      }
    }
    start += n[e];
  }
  if (chunk == 0 && F.offsets && tid == 0) F.offsets[(size_t)p * (F.nc + 1) + F.nc] = N;
  __syncthreads();
}

// A workgroup per chunk; its four waves take 256 consecutive tokens each and count their digits first, so that each knows
// where it starts.  low >= 0: token << low | the id's low bits, else the token.  SCANNED: chunk_hist is, else by chunks.
template <bool SCANNED>
__global__ __launch_bounds__(256) void km_sort_scatter_kernel(const int32_t* __restrict__ keys,
                                                              const int32_t* __restrict__ chunk_hist,
                                                              int32_t* __restrict__ out_toks, int N, int nchunks,
                                                              int shift, int bits, int low, KmFirsts F) {
  __shared__ int32_t sh_at[SCANNED ? 1 : KM_SORT_MAX_BINS];
  __shared__ int32_t sh[4][KM_SORT_MAX_BINS];
  const int p = blockIdx.y, chunk = blockIdx.x, bins = 1 << bits;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i0 = chunk * KM_SORT_CHUNK + wave * (KM_SORT_CHUNK / 4) + lane;
  int32_t* run = sh[wave];
  int32_t k[KM_SORT_ROUNDS];
#pragma unroll
  for (int r = 0; r < KM_SORT_ROUNDS; ++r) k[r] = keys[(size_t)p * N + min(i0 + r * 64, N - 1)];
  for (int b = lane; b < bins; b += 64) run[b] = 0;
  int32_t first[KM_SORT_MAX_BINS / 256];
  if (!SCANNED) km_sort_places(chunk_hist, sh_at, p, chunk, nchunks, bits, N, F);
#pragma unroll
  for (int u = 0; u < KM_SORT_MAX_BINS / 256; ++u) {
    const int b = min((int)threadIdx.x + u * 256, bins - 1);
    first[u] = SCANNED ? chunk_hist[((size_t)p * bins + b) * nchunks + chunk] : sh_at[b];
  }
  km_wave_lds_sync();
#pragma unroll
  for (int r = 0; r < KM_SORT_ROUNDS; ++r)
    if (i0 + r * 64 < N) atomicAdd(&run[(k[r] >> shift) & (bins - 1)], 1);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < KM_SORT_MAX_BINS / 256; ++u) {
    const int b = threadIdx.x + u * 256;
    if (b < bins) {
      int32_t at = first[u];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int32_t n = sh[w][b];
        sh[w][b] = at;
        at += n;
      }
    }
  }
  __syncthreads();
  const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
  for (int r = 0; r < KM_SORT_ROUNDS; ++r) {
    const int i = i0 + r * 64;
    const bool valid = i < N;
    const int bin = (k[r] >> shift) & (bins - 1);
    uint64_t peers = __builtin_amdgcn_ballot_w64(valid);  // lanes of this round with the same digit
    for (int b = 1; b < bins; b <<= 1) {
      const uint64_t m = __builtin_amdgcn_ballot_w64(valid && (bin & b));
      peers &= (bin & b) ? m : ~m;
    }
    const int start = run[bin];
    km_wave_lds_sync();  // every lane has read the running position before the leader advances it
    if (valid) {
      if (lane == 63 - __clzll((long long)peers)) run[bin] = start + __popcll(peers);
      out_toks[(size_t)p * N + start + __popcll(peers & below)] =
          low < 0 ? i : (int32_t)((uint32_t)i << low | (uint32_t)(k[r] & ((1 << low) - 1)));
    }
    km_wave_lds_sync();
  }
}

// The three launches above in one, for problems that fit one workgroup (at most KM_SMALL_MAX tokens,
// cluster ids of at most 9 bits: a segment of the segmented iterations): sixteen waves take
// consecutive chunks of the problem's tokens, count their digits into wave-private LDS rows, the
// workgroup scans the [digit][wave] table in LDS, and every wave scatters its chunk as
// km_sort_scatter_kernel does.  Same stable order, hence the same lists; the digit table never
// leaves LDS.  Writes offsets and counts like the one-pass scan.
#define KM_SMALL_WAVES 16
#define KM_SMALL_MAX (KM_SMALL_WAVES * KM_SORT_CHUNK)

__global__ __launch_bounds__(KM_SMALL_WAVES * 64) void km_sort_small_kernel(const int32_t* __restrict__ keys,
                                                                           int32_t* __restrict__ offsets,
                                                                           int32_t* __restrict__ counts,
                                                                           int32_t* __restrict__ members, int N,
                                                                           int nc, int bits) {
  __shared__ int32_t sh[KM_SMALL_WAVES][KM_SORT_MAX_BINS];
  __shared__ int32_t sh_w[KM_SMALL_WAVES];
  const int p = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int bins = 1 << bits;
  const int rounds = (N + KM_SMALL_WAVES * 64 - 1) / (KM_SMALL_WAVES * 64);   // 64-token rounds per wave
  const int base = wave * rounds * 64;
  int32_t* run = sh[wave];
  for (int b = lane; b < bins; b += 64) run[b] = 0;
  km_wave_lds_sync();
  int32_t k[KM_SORT_CHUNK / 64];
#pragma unroll
  for (int r = 0; r < KM_SORT_CHUNK / 64; ++r) {
    const int i = base + r * 64 + lane;
    k[r] = (r < rounds && i < N) ? (keys[(size_t)p * N + i] & (bins - 1)) : -1;
  }
#pragma unroll
  for (int r = 0; r < KM_SORT_CHUNK / 64; ++r)
    if (k[r] >= 0) atomicAdd(&run[k[r]], 1);
  __syncthreads();
  // exclusive scan in (digit, wave) order: thread t owns digit t / 2, waves 8 (t % 2) .. + 7
  {
    const int t = threadIdx.x, bin = t >> 1, w0 = (t & 1) * 8;
    int32_t v[8], tot = 0;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      v[u] = (bin < bins) ? sh[w0 + u][bin] : 0;
      tot += v[u];
    }
    int32_t inc = tot;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t o = __shfl_up(inc, d);
      if (lane >= d) inc += o;
    }
    if (lane == 63) sh_w[wave] = inc;
    const int32_t pair = tot + __shfl_down(tot, 1);   // even t: the digit's count over all waves
    __syncthreads();
    int32_t ex = inc - tot;
#pragma unroll
    for (int w = 0; w < KM_SMALL_WAVES; ++w)
      if (w < wave) ex += sh_w[w];
    if ((t & 1) == 0 && bin < nc) {
      offsets[(size_t)p * (nc + 1) + bin] = ex;
      counts[(size_t)p * nc + bin] = pair;
    }
    if (t == 0) offsets[(size_t)p * (nc + 1) + nc] = N;
    if (bin < bins) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        sh[w0 + u][bin] = ex;
        ex += v[u];
      }
    }
  }
  __syncthreads();
  const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
  for (int r = 0; r < KM_SORT_CHUNK / 64; ++r) {
    if (r < rounds) {   // uniform
      const bool valid = k[r] >= 0;
      const int bin = valid ? k[r] : 0;
      uint64_t peers = __ballot(valid);  // lanes of this round with the same digit
      for (int b = 0; b < bits; ++b) {
        const bool bit = (bin >> b) & 1;
        const uint64_t m = __ballot(valid && bit);
        peers &= bit ? m : ~m;
      }
      const int start = run[bin];
      km_wave_lds_sync();  // every lane has read the running position before the leader advances it
      if (valid) {
        const int pos = start + __popcll(peers & below);
        if (lane == 63 - __clzll((long long)peers)) run[bin] = start + __popcll(peers);
        members[(size_t)p * N + pos] = base + r * 64 + lane;
      }
      km_wave_lds_sync();
    }
  }
}

// Second half of a two-digit sort: one workgroup per bucket of 2^bits consecutive clusters.  The bucket's tokens (as the
// scatter left them: ascending) are counted per (cluster, wave), each wave over its own stretch of them, and placed in
// (cluster, wave) order by the same ballot ranking; the counters' scan is the bucket's part of offsets and counts.
// packed: the entries carry the cluster's low bits; where token and bits do not fit one word, the assignment is read again.
#define KM_BUCKET_WAVES 8
#define KM_BUCKET_HELD 4   // rounds of 64 tokens per wave kept in registers between the two walks

__global__ __launch_bounds__(KM_BUCKET_WAVES * 64) void km_bucket_kernel(
    const int32_t* __restrict__ assign, const int32_t* __restrict__ toks, const int32_t* __restrict__ starts,
    int32_t* __restrict__ counts, int32_t* __restrict__ offsets, int32_t* __restrict__ members, int N, int nc, int pitch,
    int bits, int buckets, int bins, bool packed) {
  constexpr int NW = KM_BUCKET_WAVES, HELD = KM_BUCKET_HELD;
  __shared__ int32_t sh_run[KM_SORT_MAX_BINS][NW];
  __shared__ int32_t sh_w[NW];
  const int p = blockIdx.y, bucket = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int C = 1 << bits, c0 = bucket << bits;
  const int32_t* first = starts + (size_t)p * bins * pitch;   // a digit's start every `pitch` words
  const int start = first[(size_t)bucket * pitch];
  const int end = bucket + 1 < buckets ? first[(size_t)(bucket + 1) * pitch] : N;
  const int rounds = (end - start + NW * 64 - 1) / (NW * 64);   // of 64 tokens per wave
  const int32_t* as = assign + (size_t)p * N;
  const int32_t* tk = toks + (size_t)p * N;
  const int i0 = start + wave * rounds * 64 + lane;
  for (int k = tid; k < C * NW; k += NW * 64) (&sh_run[0][0])[k] = 0;
  int32_t t[HELD], c[HELD];
  const auto fetch = [&](int r0) {   // four rounds' tokens and clusters; -1: none
#pragma unroll
    for (int u = 0; u < HELD; ++u) t[u] = tk[min(i0 + (r0 + u) * 64, N - 1)];
#pragma unroll
    for (int u = 0; u < HELD; ++u) {
      c[u] = (packed ? t[u] : as[t[u]]) & (C - 1);
      if (packed) t[u] = (int32_t)((uint32_t)t[u] >> bits);
    }
#pragma unroll
    for (int u = 0; u < HELD; ++u)
      if (r0 + u >= rounds || i0 + (r0 + u) * 64 >= end) c[u] = -1;
  };
  __syncthreads();
  for (int r0 = 0; r0 < rounds; r0 += HELD) {
    fetch(r0);
#pragma unroll
    for (int u = 0; u < HELD; ++u)
      if (c[u] >= 0) atomicAdd(&sh_run[c[u]][wave], 1);
  }
  __syncthreads();
  int carry = start;
  for (int k0 = 0; k0 < C * NW; k0 += NW * 64) {   // exclusive scan in (cluster, wave) order
    const int k = k0 + tid;
    const int v = k < C * NW ? (&sh_run[0][0])[k] : 0;
    const int inc = (int)ri_wave_incl_scan((uint32_t)v);
    if (lane == 63) sh_w[wave] = inc;
    __syncthreads();
    int ex = carry + inc - v;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      if (w < wave) ex += sh_w[w];
      carry += sh_w[w];
    }
    const int cl = c0 + k / NW;
    // a cluster's count: from its first wave's position to its last wave's end, eight lanes on
    const int past = __shfl_down(ex + v, NW - 1);
    if (k < C * NW) {
      (&sh_run[0][0])[k] = ex;
      if (k % NW == 0 && cl < nc) {
        offsets[(size_t)p * (nc + 1) + cl] = ex;
        counts[(size_t)p * nc + cl] = past - ex;
      }
    }
    __syncthreads();
  }
  if (bucket == buckets - 1 && tid == 0) offsets[(size_t)p * (nc + 1) + nc] = N;
  const uint64_t below = (1ull << lane) - 1ull;
  for (int r0 = 0; r0 < rounds; r0 += HELD) {
    if (rounds > HELD) fetch(r0);
#pragma unroll
    for (int u = 0; u < HELD; ++u) {
      if (r0 + u < rounds) {
        const bool ok = c[u] >= 0;
        const int cl = ok ? c[u] : 0;
        uint64_t peers = __builtin_amdgcn_ballot_w64(ok);   // lanes of this round with the same cluster
        for (int b = 1; b < C; b <<= 1) {
          const uint64_t m = __builtin_amdgcn_ballot_w64(ok && (cl & b));
          peers &= (cl & b) ? m : ~m;
        }
        const int at = sh_run[cl][wave];
        km_wave_lds_sync();   // every lane has read the running position before the leader advances it
        if (ok) {
          members[(size_t)p * N + at + __popcll(peers & below)] = t[u];
          if (lane == 63 - __clzll((long long)peers)) sh_run[cl][wave] = at + __popcll(peers);
        }
        km_wave_lds_sync();
      }
    }
  }
}

// ------------------------------------------------------------------------------------
// list-ordered reductions.  A list is summed in blocks of KM_BLK rows: inside a block one fp32
// add per row in list order starting from +0, then the block sums are added in block order
// starting from block 0's.  One wave per block, lane l owns dims 2l and 2l+1.  Lists of at
// most KM_BLK rows (nearly all of them) are finished by their own wave.  A longer list (the first
// Lloyd iterations produce a few huge ones) is split into its blocks, which other waves of the same
// launch sum in parallel; who adds the block sums in order is a second, small launch, or, in a clustering's
// later updates whose passes know nothing of each other, the wave whose block is the last to arrive.
//
// Which wave sums which block needs no queue and no counter: block j of a long list that starts at
// list offset o owns slot 2 * (o / KM_BLK) + j of its problem.  Two long lists never share a slot (a
// list of more than KM_BLK rows ends at least as many whole blocks later as it has blocks beyond its
// first), slots stay below km_item_cap(N), and the owner of a slot, if it has one, is the last
// cluster whose offset is below KM_BLK * (slot / 2 + 1): every later list starts at or after the
// owner's end, which is not.  A wave given a slot finds that cluster by a 64-way search of the
// offsets and leaves when the cluster is short or has fewer blocks.
// ------------------------------------------------------------------------------------
#define KM_BLK 256

// Rows k0 .. k1-1 of a list added in list order, U per round: the lanes fetch the round's member ids with one load and
// make row addresses of them, which are broadcast from the lanes as scalar bases; the row loads (in eights; a short last
// eight repeats its last row, and adds +0 for it, which changes no sum) are all in flight before the first add.  The
// wave's instructions bound this as much as the bytes: three fetch a row (address arithmetic per row took seven, and a
// select per row is left to the last eight: 8 x 131072 tokens, 8192 clusters 71.3 -> 57.0 us, with 64 rows in flight 67.4;
// half the tokens in seven clusters of 4 x 20000 tokens 27.7 -> 19.7).
// pitch: words between rows.  With wp the rows are also copied: row k of the list to wp + k * 64, with stores that do not stay in
// the caches, which nobody reads them from soon.  Copies take sixteen rows a round: the addresses of the stores are registers
// too, and of 84 a SIMD holds five waves where of 58 it holds eight.  Keys and values of 8 x 131072 tokens, us with 32 / 24 / 16 / 8
// rows 214.5 / 222 / 199.5 / 211.5, a prefill 3240 / - / 3225, with sixteen and such stores 204.4 and 3196; 4 x 50021 half 37.4 / 43.0 / 36.5 /
// 37.6, 34.8 with such stores, 8 x 8192 17.5 / 20.2 / 17.7 / 19.9, 16.7.  (Loads past the caches as well: 38.3 and 19.8 in these two.)
// CENTER: the sum is of the rows minus `mean` (this lane's two dims), as ri_prefill_center leaves them.
template <bool HALF, int U, bool COPY = false, bool CENTER = false>
__device__ __forceinline__ void km_sum_rows(const uint32_t* __restrict__ rp, const int32_t* mem, int k0, int k1, float& s0,
                                            float& s1, size_t pitch = RI_DIM / 2, uint32_t* __restrict__ wp = nullptr,
                                            uint32_t mean = 0u) {
  static_assert(U <= 64 && U % 8 == 0, "an id per lane, rows in eights");
  const int lane = threadIdx.x & 63;
  const auto add = [&](uint32_t w) { ri_add2<HALF>(w, s0, s1); };
  const auto term = [&](uint32_t w) { return CENTER ? ri_sub2<HALF>(w, mean) : w; };
  for (int k = k0; k < k1; k += U) {
    const int n = min(U, k1 - k);
    const uint64_t at = (uint64_t)(rp + (size_t)mem[k + min(lane, n - 1)] * pitch);
    const uint32_t lo = (uint32_t)at, hi = (uint32_t)(at >> 32);
    uint32_t v[U];
#pragma unroll
    for (int e = 0; e < U; e += 8)
      if (e < n) {
#pragma unroll
        for (int j = e; j < e + 8; ++j) {
          const uint64_t row = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, j) << 32 |
                               (uint32_t)__builtin_amdgcn_readlane(lo, j);
          v[j] = reinterpret_cast<const uint32_t*>(row)[(uint32_t)lane];
        }
      }
#pragma unroll
    for (int e = 0; e < U; e += 8) {
      if (e + 8 <= n) {
#pragma unroll
        for (int j = e; j < e + 8; ++j) {
          add(term(v[j]));
          if (COPY) __builtin_nontemporal_store(v[j], wp + (size_t)(k + j) * (RI_DIM / 2));
        }
      } else if (e < n) {
#pragma unroll
        for (int j = e; j < e + 8; ++j) {
          add(j < n ? term(v[j]) : 0u);   // the word 0 is (+0, +0) in either type
          if (COPY && j < n) __builtin_nontemporal_store(v[j], wp + (size_t)(k + j) * (RI_DIM / 2));
        }
      }
    }
  }
}

// The same sum without copies: sixty-four rows in flight at any time, each register
// requested again as soon as its row is added, ids a round ahead, rows by buffer offsets (bytes within 31 bits: km_reduce).  A
// round that is requested, waited for and added 32 rows at a time leaves a wave waiting for most of a block, and costs more than
// the waves that its fewer registers make room for (72 to 82; five to a SIMD where seven were).  Updates over given lists, us, rounds /
// ahead, an early and a late iteration: 1 x 22198 tokens, 800 clusters 15.1, 9.8 / 9.8, 7.7; 2 x 20124, 448 16.1, 13.6 / 10.9, 9.6; 2 x
// 44152, 1536 20.0, 15.4 / 15.0, 10.4; 4 x 65536, 2048 25.0, 24.3 / 21.8, 19.4; 4 x 131072, 8192 37.3, 34.3 / 34.4, 32.6; 8 x 131072, 4096
// 58.6, 56.2 / 55.0, 51.7; 8 x 200000, 8192 101.7, 100.8 / 98.8, 97.1.  Where the launch is at the memory's rate they are level: 8 x 131072, 8192
// 61.2, 63.5 / 57.5, 65.8, and on average over a clustering of them 56.3 / 56.7 (keys), 68.4 / 67.0 (values).
template <bool HALF>
__device__ __forceinline__ void km_sum_rows_ahead(__amdgpu_buffer_rsrc_t rows, uint32_t row_bytes, const int32_t* mem, int k0, int k1,
                                                  float& s0, float& s1) {
  constexpr int U = 64;
  const int lane = threadIdx.x & 63;
  const uint32_t byte = (uint32_t)lane * 4u;
  uint32_t v[U];
  int off, so[8];
  const auto offsets = [&](int e) {
#pragma unroll
    for (int j = 0; j < 8; ++j) so[j] = __builtin_amdgcn_readlane(off, e + j);
  };
  const auto request = [&](int e) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[e + j] = __builtin_amdgcn_raw_buffer_load_b32(rows, byte, so[j], 0);
  };
  const auto add8 = [&](int e) {
#pragma unroll
    for (int j = e; j < e + 8; ++j) ri_add2<HALF>(v[j], s0, s1);
  };
  const auto rest = [&](int k) {
#pragma unroll
    for (int e = 0; e < U; e += 8) {
      if (k + e + 8 <= k1) {
        add8(e);
      } else if (k + e < k1) {
#pragma unroll
        for (int j = e; j < e + 8; ++j) ri_add2<HALF>(k + j < k1 ? v[j] : 0u, s0, s1);   // the word 0 is (+0, +0) in either type
      }
    }
  };
  int k = k0;
  off = (int)((uint32_t)mem[min(k + lane, k1 - 1)] * row_bytes);
  if (k + U < k1) {
    int next = mem[min(k + U + lane, k1 - 1)];
#pragma unroll
    for (int e = 0; e < U; e += 8) {
      offsets(e);
      __builtin_amdgcn_sched_barrier(0);
      request(e);
    }
    do {   // (as in km_sum_listed: no branch around a load)
      k += U;
      off = (int)((uint32_t)next * row_bytes);
      next = mem[min(k + U + lane, k1 - 1)];
#pragma unroll
      for (int e = 0; e < U; e += 8) {
        offsets(e);
        __builtin_amdgcn_sched_barrier(0);
        add8(e);
        __builtin_amdgcn_sched_barrier(0);
        request(e);
        __builtin_amdgcn_sched_barrier(0);
      }
    } while (k + U < k1);
    rest(k);
  } else {
#pragma unroll
    for (int e = 0; e < U; e += 8)
      if (k + e < k1) {
        offsets(e);
        __builtin_amdgcn_sched_barrier(0);
        request(e);
      }
    rest(k);
  }
}

// odd (where it is asked for): set if the squares underflow or are no numbers, so that the result's norm need not be one
template <bool MEAN, bool HALF>
__device__ __forceinline__ uint32_t km_finish(float s0, float s1, int count, int normalize, uint32_t* op,
                                              int32_t* odd = nullptr) {
  if (MEAN) {
    const float cnt = (float)count;
    s0 = s0 / cnt;
    s1 = s1 / cnt;
    if (normalize) {
      const float nrm = sqrtf(ri_wave_sum(s0 * s0 + s1 * s1));  // two roundings: built without fp contraction
      if (odd && !(nrm >= 1e-15f)) *odd = 1;
      s0 = s0 / nrm;
      s1 = s1 / nrm;
    }
  }
  const uint32_t word = (uint32_t)ri_f32_to_e16<HALF>(s0) | ((uint32_t)ri_f32_to_e16<HALF>(s1) << 16);
  *op = word;
  return word;
}

// slots of one problem: the last list starts below N and a slot index is at most 2 (N / KM_BLK) + 1
static inline int km_item_cap(int N) { return 2 * (N / KM_BLK) + 2; }

// The long list that owns `slot`, found by the whole wave: returns its cluster (or -1), its length
// in s, its list offset in o and the block of it that the slot stands for in j.
// off[0 .. nc] ascending, off[0] = 0.
__device__ __forceinline__ int km_slot_owner(const int32_t* __restrict__ off, int nc, int slot, int& s, int& o,
                                             int& j) {
  const int lane = threadIdx.x & 63;
  const int limit = KM_BLK * (slot / 2 + 1);
  // last index in [0, nc) whose offset is below limit: narrow [lo, lo + len) 64 ways per round
  int lo = 0, len = nc;
  while (len > 1) {
    const int stride = (len + 63) / 64;
    const int i = lo + lane * stride;
    const bool below = (i < lo + len) && off[i] < limit;
    const int k = __popcll(__ballot(below));   // probes are ascending: the first k are below (k >= 1)
    const int nlo = lo + (k - 1) * stride;
    len = min(stride, lo + len - nlo);
    lo = nlo;
  }
  o = off[lo];
  s = off[lo + 1] - o;
  j = slot - 2 * (o / KM_BLK);
  if (s <= KM_BLK || j < 0 || j >= (s + KM_BLK - 1) / KM_BLK) return -1;
  return lo;
}

// What an update of a clustering reads and writes of KmBounds (state == nullptr: every cluster is summed, nothing is kept)
struct KmMoves {
  int32_t* state;
  uint8_t* touched;
  uint16_t* order;
  ri_int2* plan;
  int32_t *open_count, *odd;
  int first;   // nothing is known of the clusters yet
};
__device__ __forceinline__ int32_t km_next_state(int32_t state, int size, int touched) {
  const int moved = touched && size > 0;   // (an empty cluster keeps its centroid)
  return size << KM_SIZE_SHIFT | (state & KM_UNIT) | (moved ? KM_MOVED | KM_UNIT | (state & KM_UNIT ? 0 : KM_FRESH) : 0);
}

// How the next pass goes about problem p, by one workgroup of 256; a thread takes nc / 256 consecutive centroids (up to 64: a
// bit of a word each).
__device__ __forceinline__ void km_plan(const KmMoves& M, int p, int N, int nc) {
  __shared__ int sums[3][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int each = (nc + 1023) / 1024 * 4, c0 = min((int)threadIdx.x * each, nc), n = min(each, nc - c0);
  const int4* const state = reinterpret_cast<const int4*>(M.state + (size_t)p * nc + c0);
  const bool known = !M.first && M.plan[p].x != KM_KEYS;
  uint64_t moved = 0, keys = 0;
  int fresh = 0;
#pragma unroll 8
  for (int i = 0; i < n; i += 4) {
    const int4 e = state[i / 4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int w = (&e.x)[j];
      moved |= (uint64_t)(w & KM_MOVED ? 1 : 0) << (i + j);
      keys |= (uint64_t)(w & KM_UNIT ? 0 : 1) << (i + j);
      fresh += w & KM_FRESH ? w >> KM_SIZE_SHIFT : 0;
    }
  }
  // (both counts in one scan: at most 16384 each)
  const uint32_t both = (uint32_t)__popcll(moved) | (uint32_t)__popcll(keys) << 16, incl = ri_wave_incl_scan(both);
  const int fresh_incl = (int)ri_wave_incl_scan((uint32_t)fresh);
  if (lane == 63) {
    sums[0][wave] = (int)incl;
    sums[1][wave] = fresh_incl;
  }
  __syncthreads();
  uint32_t all = 0, before = incl - both;
  int all_fresh = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w < wave) before += (uint32_t)sums[0][w];
    all += (uint32_t)sums[0][w];
    all_fresh += sums[1][w];
  }
  const int all_keys = (int)(all >> 16);
  const int mode = 2 * (int64_t)all_fresh >= N ? all_keys > 0 ? KM_KEYS : KM_ALL : known ? KM_NEW : KM_ALL;
  const int n1 = mode == KM_ALL ? nc : mode == KM_KEYS ? all_keys : (int)(all & 0xffffu);
  const uint64_t first = mode == KM_ALL ? 0ull : mode == KM_KEYS ? keys : moved;
  int at1 = mode == KM_ALL ? 0 : mode == KM_KEYS ? (int)(before >> 16) : (int)(before & 0xffffu);
  int at2 = mode == KM_ALL ? c0 : n1 + c0 - at1;
  uint16_t* const order = M.order + (size_t)p * nc;
  for (int i = 0; i < n; ++i) order[first >> i & 1 ? at1++ : at2++] = (uint16_t)(c0 + i);
  if (threadIdx.x == 0) {
    M.plan[p] = (ri_int2){mode, n1};
    M.open_count[p] = 0;
  }
}

// A cache's entries of the clusters, made where their means are (out == nullptr: none): mean + the keys' mean, whether empty,
// sizes, first rows, as index_kernel makes them of finished means.
struct KmIndex {
  uint32_t* out;   // [P, nc, 64] words
  uint8_t* mask;
  uint16_t* size16;
  int32_t *size, *start;
};
// (behind the rows: a load's wait covers the stores in front of it)
template <bool HALF>
__device__ __forceinline__ void km_entry(const KmIndex& X, size_t at, int size, int start, uint32_t word, uint32_t mean) {
  const int lane = threadIdx.x & 63;
  X.out[at * (RI_DIM / 2) + lane] = ri_sum2<HALF>(word, mean);
  if (lane == 0) {
    X.mask[at] = size == 0;
    X.size16[at] = ri_f32_to_e16<HALF>((float)size);
    X.size[at] = size;
    X.start[at] = start;
  }
}

// grid (item workgroups + ceil(nc / 4), P), four waves each.  The first item_wgs workgroups take
// one slot per wave (blocks of long lists, their fp32 sums go to partial[p][slot]); the others one
// cluster per wave.  arrived: words that the blocks of a long list are counted in, the last of which finishes it (null: a launch does).
// COPY (sums of value rows): every row is also written where its list puts it, row off + k of problem p to
// copy + (p * copy_stride + off + k) * 128: the cluster-contiguous store, without a second pass over the rows.
// AHEAD (without copies): sums by km_sum_rows_ahead.
template <bool MEAN, bool HALF, bool COPY, bool CENTER, bool AHEAD = false>
__device__ __forceinline__ void km_reduce_rows(const uint16_t* __restrict__ rows, size_t pitch,
                                               const int32_t* __restrict__ counts, const int32_t* __restrict__ offsets,
                                               const int32_t* __restrict__ members, uint16_t* __restrict__ out,
                                               float2* __restrict__ partial, int item_wgs, int cap, int N, int nc,
                                               int seg, int64_t head_stride, int normalize,
                                               uint16_t* __restrict__ copy, int64_t copy_stride,
                                               const uint16_t* __restrict__ mean, const KmMoves& M = KmMoves{},
                                               const KmIndex& X = KmIndex{}, int32_t* arrived = nullptr) {
  const int p = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int32_t* off = offsets + (size_t)p * (nc + 1);
  // (head_stride and pitch in words: the rows of a head need not be contiguous)
  const uint32_t* rp = reinterpret_cast<const uint32_t*>(rows) + (size_t)(p / seg) * head_stride +
                       (size_t)(p % seg) * N * pitch;
  uint32_t* wp = COPY ? reinterpret_cast<uint32_t*>(copy) + (size_t)p * copy_stride * (RI_DIM / 2) + lane : nullptr;
  const uint32_t mw = CENTER ? reinterpret_cast<const uint32_t*>(mean)[p * (RI_DIM / 2) + lane] : 0u;
  static_assert(!AHEAD || (!COPY && !CENTER), "sums alone");
  const auto sum = [&](int o, int k0, int k1, float& s0, float& s1) {
    const int32_t* const list = members + (size_t)p * N + o;
    if constexpr (AHEAD) {
      const __amdgpu_buffer_rsrc_t all = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(rp), 0,
                                                                           (int)(((N - 1) * pitch + RI_DIM / 2) * 4), 0x00020000);
      km_sum_rows_ahead<HALF>(all, (uint32_t)pitch * 4u, list, k0, k1, s0, s1);
    } else {
      km_sum_rows<HALF, COPY ? 16 : 32, COPY, CENTER>(rp, list, k0, k1, s0, s1, pitch, COPY ? wp + (size_t)o * (RI_DIM / 2) : nullptr, mw);
    }
  };
  if ((int)blockIdx.x < item_wgs) {
    const int slot = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (slot >= cap) return;
    int s, o, j;
    const int c = km_slot_owner(off, nc, slot, s, o, j);
    if (c < 0 || (M.state && !M.first && !M.touched[(size_t)p * nc + c])) return;
    float s0 = 0.f, s1 = 0.f;
    sum(o, j * KM_BLK, min(s, (j + 1) * KM_BLK), s0, s1);
    float2* const mine = partial + ((size_t)p * cap + slot) * 64 + lane;
    if (!arrived) {
      *mine = make_float2(s0, s1);
      return;
    }
    // The last of a list's blocks to arrive adds them all: a launch less (clusterings of one segment, us, with it / without: 1 x 22198
    // tokens, 800 clusters 335 / 316; 2 x 44152, 1536 643 / 624; 1 x 71854, 2976 844 / 822).  (Block sums go past the chiplets' caches and
    // are complete before their wave arrives; one that has arrived waits for nobody.)
    typedef unsigned long long word;
    const auto pack = [](float x, float y) { return (word)__float_as_uint(y) << 32 | __float_as_uint(x); };
    __hip_atomic_store(reinterpret_cast<word*>(mine), pack(s0, s1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    km_wait_vm<0>();
    const int nb = (s + KM_BLK - 1) / KM_BLK;
    int32_t* const count = arrived + (size_t)p * cap + slot - j;
    int before = 0;
    if (lane == 0) before = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(before) != nb - 1) return;
    if (lane == 0) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("" ::: "memory");
    const word* const all = reinterpret_cast<const word*>(mine) - (size_t)j * 64;
    s0 = s1 = 0.f;
    for (int b = 0; b < nb; b += 8) {
      word v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        v[u] = __hip_atomic_load(all + (size_t)min(b + u, nb - 1) * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int u = 0; u < 8; ++u) {   // (in block order, from the first one's)
        const float x = __uint_as_float((uint32_t)v[u]), y = __uint_as_float((uint32_t)(v[u] >> 32));
        if (b + u == 0) s0 = x, s1 = y;
        else if (b + u < nb) s0 += x, s1 += y;
      }
    }
    km_finish<MEAN, HALF>(s0, s1, s, normalize, reinterpret_cast<uint32_t*>(out + ((size_t)p * nc + c) * RI_DIM) + lane);
    return;
  }
  const int c = ((int)blockIdx.x - item_wgs) * 4 + (threadIdx.x >> 6);
  if (c >= nc) return;
  const int s = counts[(size_t)p * nc + c];
  if (M.state) {   // (touched is cleared by the fold's launch)
    const size_t at = (size_t)p * nc + c;
    const int touched = M.first || M.touched[at];
    if (lane == 0) M.state[at] = km_next_state(M.first ? 0 : M.state[at], s, touched);
    if (!touched) return;   // the tokens of the update before, in the same order: it has their mean
  }
  uint32_t* op = reinterpret_cast<uint32_t*>(out + ((size_t)p * nc + c) * RI_DIM) + lane;
  const int o = off[c];
  if (s == 0) {
    if (!MEAN) *op = 0u;  // empty cluster: zero value sum; the centroid is left untouched
    else if (CENTER && X.out) km_entry<HALF>(X, (size_t)p * nc + c, s, o, *op, mw);
    return;
  }
  if (s > KM_BLK) return;  // summed by the slot waves, finished by the last of them (arrived) or by km_reduce_fold_kernel
  float s0 = 0.f, s1 = 0.f;
  sum(o, 0, s, s0, s1);
  const uint32_t word = km_finish<MEAN, HALF>(s0, s1, s, normalize, op, M.state ? M.odd + p : nullptr);
  if (CENTER && X.out) km_entry<HALF>(X, (size_t)p * nc + c, s, o, word, mw);
}

template <bool MEAN, bool HALF, bool COPY, bool AHEAD>
__global__ __launch_bounds__(256) void km_reduce_kernel(const uint16_t* __restrict__ rows, size_t pitch,
                                                        const int32_t* __restrict__ counts,
                                                        const int32_t* __restrict__ offsets,
                                                        const int32_t* __restrict__ members,
                                                        uint16_t* __restrict__ out, float2* __restrict__ partial,
                                                        int item_wgs, int cap, int N, int nc, int seg,
                                                        int64_t head_stride, int normalize,
                                                        uint16_t* __restrict__ copy, int64_t copy_stride, KmMoves M,
                                                        int32_t* arrived) {
  km_reduce_rows<MEAN, HALF, COPY, false, AHEAD>(rows, pitch, counts, offsets, members, out, partial, item_wgs, cap, N, nc, seg,
                                          head_stride, normalize, copy, copy_stride, nullptr, M, KmIndex{}, arrived);
}

// Value sums with the value store (z = 0) and means of the centred keys with the key store (z = 1): the last step of a
// prefill.  The keys are read raw, from where the model left them, and centred on the way to their sum, so that the
// store needs no pass of its own.  Bound by the bytes: 8 x 131072 tokens, 1.07 GB in 206 us = 5.2 TB/s, the rate of a
// copy (keys 51 us, values 102 and the copy of the keys 98 in launches of their own).
struct KmStoreArgs {
  const uint16_t* rows;
  uint16_t *out, *copy;
  float2* partial;
  size_t pitch;          // words
  int64_t head_stride;   // words
};
template <bool HALF>
__global__ __launch_bounds__(256) void km_store_kernel(KmStoreArgs V, KmStoreArgs K, const uint16_t* __restrict__ mean,
                                                       const int32_t* __restrict__ counts,
                                                       const int32_t* __restrict__ offsets,
                                                       const int32_t* __restrict__ members, int item_wgs, int cap, int N,
                                                       int nc, int64_t copy_stride, KmIndex X) {
  if (blockIdx.z == 0)
    km_reduce_rows<false, HALF, true, false>(V.rows, V.pitch, counts, offsets, members, V.out, V.partial, item_wgs, cap, N,
                                             nc, 1, V.head_stride, 0, V.copy, copy_stride, nullptr);
  else
    km_reduce_rows<true, HALF, true, true>(K.rows, K.pitch, counts, offsets, members, K.out, K.partial, item_wgs, cap, N,
                                           nc, 1, K.head_stride, 0, K.copy, copy_stride, mean, KmMoves{}, X);
}

// grid (item workgroups, P): the wave of a long list's first slot adds the block sums in block
// order and finishes the cluster
template <bool MEAN, bool HALF>
__device__ __forceinline__ void km_fold(const int32_t* __restrict__ offsets, const float2* __restrict__ partial,
                                        uint16_t* __restrict__ out, int cap, int nc, int normalize,
                                        const KmMoves& M = KmMoves{}, const uint32_t* mean = nullptr,
                                        const KmIndex& X = KmIndex{}) {
  const int p = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int slot = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (M.state)
    for (int c = blockIdx.x * 256 + threadIdx.x; c < nc; c += gridDim.x * 256) M.touched[(size_t)p * nc + c] = 0;
  if (slot >= cap) return;
  int s, o, j;
  const int c = km_slot_owner(offsets + (size_t)p * (nc + 1), nc, slot, s, o, j);
  if (c < 0 || j != 0 || (M.state && !(M.state[(size_t)p * nc + c] & KM_MOVED))) return;
  const int nb = (s + KM_BLK - 1) / KM_BLK;
  const float2* pp = partial + ((size_t)p * cap + slot) * 64 + lane;
  float2 t = pp[0];
  int b = 1;
  for (; b + 4 <= nb; b += 4) {
    float2 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = pp[(size_t)(b + u) * 64];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      t.x += v[u].x;
      t.y += v[u].y;
    }
  }
  for (; b < nb; ++b) {
    const float2 v = pp[(size_t)b * 64];
    t.x += v.x;
    t.y += v.y;
  }
  uint32_t* op = reinterpret_cast<uint32_t*>(out + ((size_t)p * nc + c) * RI_DIM) + lane;
  const uint32_t word = km_finish<MEAN, HALF>(t.x, t.y, s, normalize, op, M.state ? M.odd + p : nullptr);
  if (X.out) km_entry<HALF>(X, (size_t)p * nc + c, s, o, word, mean[p * (RI_DIM / 2) + lane]);
}

template <bool MEAN, bool HALF>
__global__ __launch_bounds__(256) void km_reduce_fold_kernel(const int32_t* __restrict__ offsets,
                                                             const float2* __restrict__ partial,
                                                             uint16_t* __restrict__ out, int cap, int nc,
                                                             int normalize, KmMoves M, int N, int32_t* arrived) {
  if (arrived && threadIdx.x < 4 && blockIdx.x * 4 + threadIdx.x < cap) arrived[(size_t)blockIdx.y * cap + blockIdx.x * 4 + threadIdx.x] = 0;
  if (M.state && blockIdx.x == gridDim.x - 1) km_plan(M, blockIdx.y, N, nc);   // (a workgroup of its own: no slot is left)
  km_fold<MEAN, HALF>(offsets, partial, out, cap, nc, normalize, M);
}

template <bool HALF>
__global__ __launch_bounds__(256) void km_store_fold_kernel(KmStoreArgs V, KmStoreArgs K,
                                                            const uint16_t* __restrict__ mean,
                                                            const int32_t* __restrict__ offsets, int cap, int nc, KmIndex X) {
  if (blockIdx.z == 0) km_fold<false, HALF>(offsets, V.partial, V.out, cap, nc, 0);
  else km_fold<true, HALF>(offsets, K.partial, K.out, cap, nc, 0, KmMoves{}, reinterpret_cast<const uint32_t*>(mean), X);
}

// ------------------------------------------------------------------------------------
// update straight from the assignment, for problems of at most KM_DIRECT_MAX tokens (the segments of the segmented
// iterations): list sort, list-ordered sums and means in one launch, no lists in memory.
// grid km_grid(ceil(nc / CPW), P), eight waves: a workgroup owns CPW consecutive clusters.  Every wave takes a contiguous run of
// the problem's tokens, compacts those of the workgroup's clusters into LDS (in token order), counts them, and after a
// scan in (cluster, wave) order scatters them to the workgroup's list in LDS, ranking equal clusters inside a round of 64
// with ballots: the stable order of the list kernels, hence the same sums.  The run is read four tokens to a lane (eight in 16 bits), up to
// 1024 requested at once; a token costs three instructions (its cluster in a byte, all others' flagged), positions come
// from one wave scan per 512 and only the few hits are looped over.  A ballot, a rank and a branch for every 64 tokens
// were most of a late update: 8 x 8192 tokens, 512 clusters 8.2 -> 7.5 us, 4 x 15000, 928 clusters 10.8 -> 9.2, 1 x 16384
// 8.5 -> 6.9, 128 x 8192 52.0 -> 49.8.  Then a wave sums whole clusters of at most
// KM_BLK rows; the blocks of longer ones are spread over the waves and folded in block order.
// Reading all assignments of the problem per workgroup is what the split costs: 32 KB at 8192 tokens in 32 bits, a third of
// a late update's time.  NARROW: an earlier pass left them as 16-bit words (km_put_place); twice eight tokens to a lane, two
// words to an instruction, one scan per 1024.  Loads are made without a condition, what they bring too much is put out
// afterwards (behind a condition each waited for the one before), and what the rows' address takes, a division and four
// arguments, is done while they are on their way (after the lists it took 400 ns).  Late updates by the two, us: 8 x 8192 tokens, 512
// clusters 7.1 -> 5.8, 24 x 8119 half 12.7 -> 11.5, 128 x 8192 49.7 -> 47.0 (50.5 in 32 bits).
// 128 x 8192 tokens, 512 clusters each: 47 us, bound by reading the keys, against 13 + 70 + 5 us of list
// sort, sums and fold; 8 x 8192: 5.8 us against 12 + 11 + 4.5.
// counts / offsets / members (CSR, as km_sort_small_kernel writes them) only when asked for, and then alone if there is
// no `cent`: the last pass of a prefill, whose means come with the stores (8 x 8192 tokens, whole prefill 367 -> 363 us).
// ------------------------------------------------------------------------------------
#define KM_DIRECT_WAVES 8
#define KM_DIRECT_MAX 16384

#define KM_DIRECT_SHORT 128   // longer lists are summed in blocks and folded, as lists of several blocks are
// Rows k0 .. k1-1 of a list in LDS added in list order, U in flight: ids come with one LDS read per U and are broadcast
// from the lanes as buffer offsets; a row's register takes the row U further on as soon as it is added (in eights; past the
// last row that is repeated, and +0 is added for it, which changes no sum).  A wave's own chain bounds a list: two
// instructions fetch a row and two per dim add it, one in half (an address per row in 64 bits, and a select per row, made
// it ten; 8 x 8192 tokens, 512 clusters: 10.6 -> 9.6 us; 128 x 8192: 67.6 -> 61.6).  Requests beside the additions instead
// of U rows at a time, nine updates of Lloyd iterations together: 128 x 8192 tokens 543 -> 517 us (half 626 -> 512, where
// 80 registers instead of 82 also make room for a third workgroup), 24 x 8119 183 -> 175 (216 -> 166), 8 x 8192 107 -> 104.
// The offsets of eight rows are read from the lanes before the additions that free their registers: a load right behind
// the readlane that makes its offset waits five issues for it (the same nine updates 101 -> 99, 128 x 8192 507 -> 503, 4 x
// 15000 tokens, 928 clusters 155 -> 145).
// WHOLE: two dims per lane, else one (two waves share the row).
template <bool HALF, int U, bool WHOLE>
__device__ __forceinline__ void km_sum_listed(__amdgpu_buffer_rsrc_t rows, uint32_t byte, const uint16_t* list, int k0, int k1,
                                              float& s0, float& s1) {
  static_assert(U <= 64 && U % 8 == 0, "an id per lane, rows in eights");
  const int lane = threadIdx.x & 63;
  const auto add = [&](uint32_t w) {
    if (WHOLE) ri_add2<HALF>(w, s0, s1);
    else ri_add_lo<HALF>(w, s0);
  };
  uint32_t v[U];
  int off, so[8];
  const auto ids = [&](int k) { off = (int)list[min(k + lane, k1 - 1)] * (RI_DIM * 2); };
  const auto offsets = [&](int e) {
#pragma unroll
    for (int j = 0; j < 8; ++j) so[j] = __builtin_amdgcn_readlane(off, e + j);
  };
  const auto request = [&](int e) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[e + j] = WHOLE ? __builtin_amdgcn_raw_buffer_load_b32(rows, byte, so[j], 0)
                       : (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rows, byte, so[j], 0);
  };
  const auto fetch = [&](int e) {
    offsets(e);
    __builtin_amdgcn_sched_barrier(0);
    request(e);
  };
  const auto add8 = [&](int e) {
#pragma unroll
    for (int j = e; j < e + 8; ++j) add(v[j]);
  };
  const auto rest = [&](int k) {
#pragma unroll
    for (int e = 0; e < U; e += 8) {
      if (k + e + 8 <= k1) {
        add8(e);
      } else if (k + e < k1) {
#pragma unroll
        for (int j = e; j < e + 8; ++j) add(k + j < k1 ? v[j] : 0u);   // the word 0 is (+0, +0) in either type
      }
    }
  };
  int k = k0;
  ids(k);
  if (k + U < k1) {
#pragma unroll
    for (int e = 0; e < U; e += 8) fetch(e);
    // (no branch around a load here: the compiler counts the loads behind the ones it waits for, and takes those that may
    // not have been made for not made)
    do {
      k += U;
      ids(k);
#pragma unroll
      for (int e = 0; e < U; e += 8) {
        offsets(e);
        __builtin_amdgcn_sched_barrier(0);   // (else each goes to the load it is for)
        add8(e);
        __builtin_amdgcn_sched_barrier(0);
        request(e);
        __builtin_amdgcn_sched_barrier(0);   // (else the next loads move up, into registers of their own)
      }
    } while (k + U < k1);
    rest(k);
  } else {
#pragma unroll
    for (int e = 0; e < U; e += 8)
      if (k + e < k1) fetch(e);
    rest(k);
  }
}

// four consecutive assignments; a problem's first one lies on four bytes only
typedef int32_t km_quad __attribute__((ext_vector_type(4), aligned(4)));
// eight consecutive ones in 16 bits (a problem's row of `assign` starts on four bytes)
typedef uint32_t km_eight __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t km_u16x2 __attribute__((ext_vector_type(2)));
// tokens of a wave's run: whole quads of 64 lanes
__host__ __device__ constexpr int km_direct_run(int N) {
  return (N + KM_DIRECT_WAVES * 256 - 1) / (KM_DIRECT_WAVES * 256) * 256;
}

// The values and keys of a list, tokens list[k0 .. k1-1], in sums and copies as km_sum_rows makes them (s: two dims of the values,
// two of the keys less their mean).  Both rows of sixteen tokens are on their way before the first is added: a load's wait covers
// the stores in front of it.  VALUES, KEYS: both or one of them.
struct KmStoreDirect {
  KmStoreArgs v, k;        // (no partials)
  const uint16_t* mean;
  int64_t stride;          // rows of the stores from problem to problem
  KmIndex X;
};
template <bool HALF, bool VALUES, bool KEYS>
__device__ __forceinline__ void km_store_listed(const uint32_t* rv, size_t pv, const uint32_t* rk, size_t pk, const uint16_t* list,
                                                int k0, int k1, float (&s)[4], uint32_t* wv, uint32_t* wk, uint32_t mean) {
  const int lane = threadIdx.x & 63;
  for (int k = k0; k < k1; k += 16) {
    const int n = min(16, k1 - k), token = list[k + min(lane & 15, n - 1)];
    uint32_t v[16], x[16];
#pragma unroll
    for (int e = 0; e < 16; e += 8)
      if (e < n) {
#pragma unroll
        for (int j = e; j < e + 8; ++j) {
          const size_t t = (uint32_t)__builtin_amdgcn_readlane(token, j);
          if (VALUES) v[j] = (rv + t * pv)[(uint32_t)lane];
          if (KEYS) x[j] = (rk + t * pk)[(uint32_t)lane];
        }
      }
#pragma unroll
    for (int e = 0; e < 16; e += 8) {
      if (e >= n) break;
#pragma unroll
      for (int j = e; j < e + 8; ++j) {
        if (VALUES) ri_add2<HALF>(j < n ? v[j] : 0u, s[0], s[1]);
        if (KEYS) ri_add2<HALF>(j < n ? ri_sub2<HALF>(x[j], mean) : 0u, s[2], s[3]);
      }
#pragma unroll
      for (int j = e; j < e + 8; ++j)
        if (j < n) {
          if (VALUES) __builtin_nontemporal_store(v[j], wv + (size_t)(k + j) * (RI_DIM / 2));
          if (KEYS) __builtin_nontemporal_store(x[j], wk + (size_t)(k + j) * (RI_DIM / 2));
        }
    }
  }
}

// STORE: the lists' values and keys are summed and stored as ri_kmeans_store_rows does it, see km_store_direct_kernel.
template <bool HALF, int CPW, bool NARROW, bool STORE>
__device__ __forceinline__ void km_direct_group(
    const uint16_t* __restrict__ rows, const int32_t* __restrict__ assign, uint16_t* __restrict__ cent, int N, int nc,
    int shape, int seg, int64_t head_rows, int32_t* __restrict__ counts, int32_t* __restrict__ offsets,
    int32_t* __restrict__ listed, const KmStoreDirect& T) {
  constexpr int NW = KM_DIRECT_WAVES, E = CPW * NW / 64;   // E: (cluster, wave) counters per lane
  static_assert((CPW & (CPW - 1)) == 0 && CPW * NW % 64 == 0 && CPW <= 64, "counters dealt to the lanes, a cluster in a byte");
  __shared__ int32_t sh_run[CPW * NW], sh_at[NW][CPW], sh_off[CPW + 1], sh_below[NW];
  extern __shared__ __attribute__((aligned(16))) uint32_t sh_buf[];   // NW * run_len words: compacted tokens, later block sums
  int32_t* const members = NARROW ? nullptr : listed;
  const int sh = shape & 3, normalize = shape >> 2 & 1;
  // (last problem first: its keys are what the assignment pass has just left in the memory-side cache)
  const int p = (((shape >> 3) - (int)blockIdx.y) << sh) + (blockIdx.x & ((1 << sh) - 1)), c0 = (blockIdx.x >> sh) * CPW;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int run_len = km_direct_run(N);
  uint32_t* const mine = sh_buf + wave * run_len;
  uint16_t* const list = reinterpret_cast<uint16_t*>(sh_buf + NW * run_len);
  if (lane < CPW) sh_run[lane * NW + wave] = 0;
  km_wave_lds_sync();
  const int32_t* as = assign + (size_t)p * N;
  const int t1 = min((wave + 1) * run_len, N);
  int cnt = 0, below = 0;   // tokens of this wave in the workgroup's clusters, (per lane) in lower ones
  const auto take = [&](uint32_t c, int token, int at) {
    mine[at] = c << 16 | (uint32_t)token;
    atomicAdd(&sh_run[c * NW + wave], 1);
  };
  size_t row0 = 0;
  const auto find_rows = [&]() {   // a division, while the assignments are on their way
    __builtin_amdgcn_sched_barrier(0);
    int problem = p, segments = seg;
    asm volatile("" : "+s"(problem), "+s"(segments));   // (else it moves ahead of them)
    row0 = km_row0(problem, segments, head_rows, N);
    asm volatile("" : "+s"(row0));
  };
  int t0 = wave * run_len;
  do {   // (once for a wave without tokens, too)
    if constexpr (NARROW) {
      // twice eight consecutive tokens per lane, without a condition: what lies past the problem's N words is still its own row
      km_eight a[2];
#pragma unroll
      for (int q = 0; q < 2; ++q)
        a[q] = *reinterpret_cast<const km_eight*>(reinterpret_cast<const uint16_t*>(as) + min(t0 + q * 512 + lane * 8, 2 * N - 8));
      find_rows();
      uint64_t loc[2], hit[2];   // a byte per token: its cluster from c0 on, CPW for all others
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        uint32_t d[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t w = a[q][j];   // (a cast of the element itself takes the first one's)
          const km_u16x2 x = __builtin_bit_cast(km_u16x2, w) - km_u16x2((uint16_t)c0);
          d[j] = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(x, km_u16x2((uint16_t)CPW)));
        }
        loc[q] = (uint64_t)__builtin_amdgcn_perm(d[3], d[2], 0x06040200) << 32 | __builtin_amdgcn_perm(d[1], d[0], 0x06040200);
        const int left = t1 - (t0 + q * 512 + lane * 8);
        if (t0 + q * 512 + 512 > t1)   // (uniform)
          loc[q] = left >= 8 ? loc[q] : loc[q] | (uint64_t)CPW * 0x0101010101010101ull << 8 * max(left, 0);
        hit[q] = ~loc[q] & (uint64_t)CPW * 0x0101010101010101ull;
      }
      // positions of a lane's first hits in both eights, in one scan (at most 512 each)
      const uint32_t n = (uint32_t)__popcll(hit[0]) | (uint32_t)__popcll(hit[1]) << 16, inc = ri_wave_incl_scan(n);
      const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
      int at[2] = {cnt + (int)((inc - n) & 0xffffu), cnt + (int)(all & 0xffffu) + (int)((inc - n) >> 16)};
      cnt += (int)(all & 0xffffu) + (int)(all >> 16);
#pragma unroll
      for (int q = 0; q < 2; ++q)
        for (uint64_t h = hit[q]; h; h &= h - 1) {
          const int j = (__ffsll((long long)h) - 1) >> 3;
          take((uint32_t)(loc[q] >> (8 * j)) & (uint32_t)(CPW - 1), t0 + q * 512 + lane * 8 + j, at[q]++);
        }
    } else {
      // four quads of consecutive tokens per lane; the one that would pass the problem's end begins at its last four tokens
      km_quad a[4];
      if (N >= 4) {
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] = *reinterpret_cast<const km_quad*>(as + min(t0 + q * 256 + lane * 4, N - 4));
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int j = 0; j < 4; ++j) a[q][j] = as[min(j, N - 1)];
      }
      if (!STORE && cent) find_rows();   // (lists alone and stores ask for no rows here: 8 x 8192 tokens' lists 5.55 -> 5.4 us)
#pragma unroll
      for (int q0 = 0; q0 < 4; q0 += 2) {
        if (t0 + q0 * 256 >= t1) break;
        uint32_t loc[2], hit[2], at[2];
        int first[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int i = t0 + (q0 + q) * 256 + lane * 4;
          first[q] = min(i, max(N - 4, 0));
          if (t0 + (q0 + q) * 256 + 256 > t1) {   // (uniform)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (first[q] + j < i || first[q] + j >= t1) a[q0 + q][j] = 0x7fffffff;
          }
          loc[q] = 0;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t d = (uint32_t)(a[q0 + q][j] - c0);
            loc[q] |= min(d, (uint32_t)CPW) << (8 * j);
            if (members) below += (int)(d >> 31);
          }
          hit[q] = ~loc[q] & (uint32_t)CPW * 0x01010101u;
        }
        // positions of a lane's first hits in both quads, in one scan (at most 256 each)
        const uint32_t n = (uint32_t)__popc(hit[0]) | (uint32_t)__popc(hit[1]) << 16, inc = ri_wave_incl_scan(n);
        const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
        at[0] = cnt + ((inc - n) & 0xffffu);
        at[1] = cnt + (int)(all & 0xffffu) + ((inc - n) >> 16);
        cnt += (int)(all & 0xffffu) + (int)(all >> 16);
#pragma unroll
        for (int q = 0; q < 2; ++q)
          for (uint32_t h = hit[q]; h; h &= h - 1) {
            const int j = (__ffs((int)h) - 1) >> 3;
            take(loc[q] >> (8 * j) & (uint32_t)(CPW - 1), first[q] + j, at[q]++);
          }
      }
    }
    t0 += 1024;
  } while (t0 < t1);
  if (members) {
    below = (int)ri_wave_incl_scan((uint32_t)below);
    if (lane == 63) sh_below[wave] = below;
  }
  __syncthreads();
  int32_t* const run = sh_at[wave];
  {   // exclusive scan in (cluster, wave) order; every wave makes it, and keeps the positions of its own tokens
    int v[E], sum = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) sum += v[e] = sh_run[lane * E + e];
    int ex = (int)ri_wave_incl_scan((uint32_t)sum) - sum;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int c = (lane * E + e) / NW, w = (lane * E + e) % NW;
      if (w == wave) run[c] = ex;
      if (w == 0 && wave == 0) sh_off[c] = ex;
      ex += v[e];
    }
    if (wave == 0 && lane == 63) sh_off[CPW] = ex;
  }
  km_wave_lds_sync();
  const uint64_t lower = (1ull << lane) - 1ull;
  for (int k = 0; k < cnt; k += 64) {
    const bool ok = k + lane < cnt;
    const uint32_t e = mine[min(k + lane, cnt - 1)];
    const int c = (int)(e >> 16);
    uint64_t peers = __builtin_amdgcn_ballot_w64(ok);   // lanes of this round with the same cluster
#pragma unroll
    for (int b = 1; b < CPW; b <<= 1) {
      const uint64_t m = __builtin_amdgcn_ballot_w64(ok && (c & b));
      peers &= (c & b) ? m : ~m;
    }
    const int start = run[c];
    km_wave_lds_sync();  // every lane has read the running position before the leader advances it
    if (ok) {
      list[start + __popcll(peers & lower)] = (uint16_t)(e & 0xffffu);
      if (lane == 63 - __clzll((long long)peers)) run[c] = start + __popcll(peers);
    }
    km_wave_lds_sync();
  }
  __syncthreads();

  int base = 0;   // tokens of lower clusters
  const auto write_lists = [&]() {
    for (int k = tid; k < sh_off[CPW]; k += NW * 64) members[(size_t)p * N + base + k] = list[k];
    if (tid < CPW && c0 + tid < nc) {
      offsets[(size_t)p * (nc + 1) + c0 + tid] = base + sh_off[tid];
      counts[(size_t)p * nc + c0 + tid] = sh_off[tid + 1] - sh_off[tid];
    }
    if (tid == 0 && c0 + CPW >= nc) offsets[(size_t)p * (nc + 1) + nc] = N;
  };
  if (members) {
#pragma unroll
    for (int w = 0; w < NW; ++w) base += sh_below[w];
  }
  if constexpr (STORE) {
    const uint32_t* const rv = reinterpret_cast<const uint32_t*>(T.v.rows) + (size_t)p * T.v.head_stride;
    const uint32_t* const rk = reinterpret_cast<const uint32_t*>(T.k.rows) + (size_t)p * T.k.head_stride;
    const size_t first = ((size_t)p * T.stride + base) * (RI_DIM / 2) + lane, clusters = (size_t)p * nc + c0;
    uint32_t* const wv = reinterpret_cast<uint32_t*>(T.v.copy) + first;
    uint32_t* const wk = reinterpret_cast<uint32_t*>(T.k.copy) + first;
    uint32_t* const sums = reinterpret_cast<uint32_t*>(T.v.out) + clusters * (RI_DIM / 2) + lane;
    uint32_t* const means = reinterpret_cast<uint32_t*>(T.k.out) + clusters * (RI_DIM / 2) + lane;
    const uint32_t mean = reinterpret_cast<const uint32_t*>(T.mean)[p * (RI_DIM / 2) + lane];
    const auto finish_keys = [&](int c, int o, int s, float s0, float s1) {
      const uint32_t word = km_finish<true, HALF>(s0, s1, s, 0, means + c * (RI_DIM / 2));
      if (T.X.out) km_entry<HALF>(T.X, clusters + c, s, base + o, word, mean);
    };
    bool longer = false;
    for (int c = wave; c < CPW && c0 + c < nc; c += NW) {
      const int o = sh_off[c], s = sh_off[c + 1] - o;
      if (s == 0) {   // zero value sum; the centroid stays
        sums[c * (RI_DIM / 2)] = 0u;
        if (T.X.out) km_entry<HALF>(T.X, clusters + c, 0, base + o, means[c * (RI_DIM / 2)], mean);
        continue;
      }
      if (s > KM_BLK) {
        longer = true;
        continue;
      }
      float x[4] = {0.f, 0.f, 0.f, 0.f};
      km_store_listed<HALF, true, true>(rv, T.v.pitch, rk, T.k.pitch, list, o, o + s, x, wv, wk, mean);
      km_finish<false, HALF>(x[0], x[1], s, 0, sums + c * (RI_DIM / 2));
      finish_keys(c, o, s, x[2], x[3]);
    }
    write_lists();
    if (!__syncthreads_or(longer)) return;
    // Lists of several blocks, values then keys: the blocks dealt to the waves, their sums (512 bytes each, at most N / 128 of
    // them) where the compacted tokens were, then added in order.
    float2* const part = reinterpret_cast<float2*>(sh_buf);
    const auto blocks = [&](auto keys) {
      constexpr bool KEYS = decltype(keys)::value;
      for (int fold = 0; fold < 2; ++fold) {
        for (int c = 0, item = 0; c < CPW; ++c) {
          const int o = sh_off[c], s = sh_off[c + 1] - o, nb = (s + KM_BLK - 1) / KM_BLK;
          if (nb < 2) continue;
          if (!fold) {
            for (int b = 0; b < nb; ++b)
              if (((item + b) & (NW - 1)) == wave) {
                float x[4] = {0.f, 0.f, 0.f, 0.f};
                km_store_listed<HALF, !KEYS, KEYS>(rv, T.v.pitch, rk, T.k.pitch, list, o + b * KM_BLK, o + min(s, (b + 1) * KM_BLK), x,
                                                   wv, wk, mean);
                part[(item + b) * 64 + lane] = KEYS ? make_float2(x[2], x[3]) : make_float2(x[0], x[1]);
              }
          } else if ((c & (NW - 1)) == wave) {
            float2 t = part[item * 64 + lane];
            for (int b = 1; b < nb; ++b) {
              t.x += part[(item + b) * 64 + lane].x;
              t.y += part[(item + b) * 64 + lane].y;
            }
            if (KEYS) finish_keys(c, o, s, t.x, t.y);
            else km_finish<false, HALF>(t.x, t.y, s, 0, sums + c * (RI_DIM / 2));
          }
          item += nb;
        }
        __syncthreads();
      }
    };
    blocks(std::false_type{});
    blocks(std::true_type{});
    return;
  }
  if (members) {
    write_lists();
    if (!cent) return;
  }
  const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(rows + row0 * RI_DIM), 0, N * RI_DIM * 2, 0x00020000);
  uint32_t* op = reinterpret_cast<uint32_t*>(cent + ((size_t)p * nc + c0) * RI_DIM) + lane;
  // Work items for the waves in turn: the blocks of the long lists first (early iterations have lists of thousands), then
  // the short lists; no barrier between them.  Block sums go to LDS: the compacted tokens are dead, and lists longer than
  // KM_DIRECT_SHORT have at most N / KM_DIRECT_SHORT blocks of 512 bytes.  A block of 256 rows is a long chain, so
  // its two halves go to two waves while every wave gets one at most (with more blocks that would only be twice the
  // loads): the four early iterations of 8 x 8192 tokens 104 -> 84 us together, three of 128 x 8192 267 -> 216.
  float* const part = reinterpret_cast<float*>(sh_buf);
  const int my_o = sh_off[min(lane, CPW - 1)], my_s = lane < CPW ? sh_off[min(lane, CPW - 1) + 1] - my_o : 0;
  const int my_nb = my_s > KM_DIRECT_SHORT ? (my_s + KM_BLK - 1) / KM_BLK : 0;
  uint64_t big = __builtin_amdgcn_ballot_w64(my_nb > 0);
  int nb_incl = 0, nblocks = 0;
  if (big) {
    nb_incl = (int)ri_wave_incl_scan((uint32_t)my_nb);
    nblocks = __builtin_amdgcn_readlane(nb_incl, 63);
  }
  const int halves = 2 * nblocks <= NW ? 2 : 1, items = halves * nblocks;
  for (int k = wave; k < items; k += NW) {
    const int blk = halves == 2 ? k >> 1 : k;
    const int c = __ffsll((long long)__builtin_amdgcn_ballot_w64(nb_incl > blk)) - 1;
    const int o = __builtin_amdgcn_readlane(my_o, c), s = __builtin_amdgcn_readlane(my_s, c);
    const int b = blk - (__builtin_amdgcn_readlane(nb_incl, c) - __builtin_amdgcn_readlane(my_nb, c));
    const int k0 = o + b * KM_BLK, k1 = o + min(s, (b + 1) * KM_BLK);
    float s0 = 0.f, s1 = 0.f;
    if (halves == 2) {
      km_sum_listed<HALF, 64, false>(rp, (k & 1) * RI_DIM + lane * 2, list, k0, k1, s0, s1);
      part[k * 64 + lane] = s0;
    } else {
      km_sum_listed<HALF, 64, true>(rp, lane * 4, list, k0, k1, s0, s1);
      reinterpret_cast<float2*>(part)[k * 64 + lane] = make_float2(s0, s1);
    }
  }
  // (the wave after the last block's takes the first short list)
  for (int c = (wave - items) & (NW - 1); c < CPW; c += NW) {   // (a cluster past the last has no tokens; an empty one keeps its centroid)
    const int o = __builtin_amdgcn_readlane(my_o, c), s = __builtin_amdgcn_readlane(my_s, c);
    if (s == 0 || s > KM_DIRECT_SHORT) continue;
    float s0 = 0.f, s1 = 0.f;
    km_sum_listed<HALF, 32, true>(rp, lane * 4, list, o, o + s, s0, s1);
    km_finish<true, HALF>(s0, s1, s, normalize, op + c * (RI_DIM / 2));
  }
  if (nblocks == 0) return;   // uniform over the workgroup
  __syncthreads();
  for (int i = 0; big; big &= big - 1, ++i) {   // a wave folds every eighth long list in block order
    if ((i & (NW - 1)) != wave) continue;
    const int c = __ffsll((long long)big) - 1;
    const int s = __builtin_amdgcn_readlane(my_s, c), nb = __builtin_amdgcn_readlane(my_nb, c);
    const float2* pp = reinterpret_cast<const float2*>(part) + (__builtin_amdgcn_readlane(nb_incl, c) - nb) * 64 + lane;
    float2 t = pp[0];
    for (int b = 1; b < nb; ++b) {
      t.x += pp[b * 64].x;
      t.y += pp[b * 64].y;
    }
    km_finish<true, HALF>(t.x, t.y, s, normalize, op + c * (RI_DIM / 2));
  }
}

template <bool HALF, int CPW, bool NARROW>
__global__ __launch_bounds__(KM_DIRECT_WAVES * 64, 6) void km_direct_kernel(
    const uint16_t* __restrict__ rows, const int32_t* __restrict__ assign, uint16_t* __restrict__ cent, int N, int nc,
    int shape, int seg, int64_t head_rows, int32_t* __restrict__ counts, int32_t* __restrict__ offsets,
    int32_t* __restrict__ listed) {
  km_direct_group<HALF, CPW, NARROW, false>(rows, assign, cent, N, nc, shape, seg, head_rows, counts, offsets, listed,
                                            KmStoreDirect{});
}

// Lists, value sums, means, stores and index entries of short problems in one launch, where lists, rows and a fold of long lists'
// blocks are three: the lists stay in LDS, and what bounds it is one chain of assignments, rows and stores instead of
// three.  Worth it while all workgroups of eight clusters are resident at once: 512 up to 12288 tokens, past them, where one's LDS is
// 87 KB and more, 256 (kernels.py).  This launch / the three, captured, us: 8 x 8192 tokens, 512 clusters 20.2 / 23.7, 4 x 12288, 768 18.0 /
// 20.6, 8 x 12288, 512 30.3 / 32.3, 2 x 16384, 1024 14.2 / 15.7; fewer workgroups 2 x 8192 14.2 / 13.8, 1 x 4000 12.2 / 11.9, which
// whole prefills do not show; more of them than fit 4 x 12300, 768 25.5 / 21.5, 4 x 16384, 1024 25.5 / 22.3, 2 x 16384, 1088 24.0 / 18.4.
// More clusters to a workgroup, prefills: 8 x 12000 350.4 -> 353.6, 8 x 16384 346.4 -> 352.4.
template <bool HALF>
__global__ __launch_bounds__(KM_DIRECT_WAVES * 64, 4) void km_store_direct_kernel(const int32_t* __restrict__ assign, int N, int nc,
                                                                                  int shape, int32_t* __restrict__ counts,
                                                                                  int32_t* __restrict__ offsets,
                                                                                  int32_t* __restrict__ members, KmStoreDirect T) {
  km_direct_group<HALF, 8, false, true>(nullptr, assign, nullptr, N, nc, shape, 1, N, counts, offsets, members, T);
}

// out[p, i, :] = in[p, members[p, i], :]; 16 lanes per row; strides in 16-byte pieces
__global__ __launch_bounds__(256) void km_permute_kernel(const uint4* __restrict__ in,
                                                         const int32_t* __restrict__ members,
                                                         uint4* __restrict__ out, int N, int64_t in_head,
                                                         int64_t in_row, int64_t out_head) {
  const int p = blockIdx.y;
  const int i = blockIdx.x * 16 + (threadIdx.x >> 4);
  const int piece = threadIdx.x & 15;
  if (i >= N) return;
  const int32_t src = members[(size_t)p * N + i];
  out[(size_t)p * out_head + (size_t)i * 16 + piece] = in[(size_t)p * in_head + (size_t)src * in_row + piece];
}

// centroids[g, c] = data[g, idx(c)], idx(c) = trunc(c * ratio + half) in fp32 (kmeans.py:234-236); 16 lanes per row
__global__ __launch_bounds__(256) void km_init_kernel(const uint4* __restrict__ data, uint4* __restrict__ cent, int N,
                                                      int nc, float ratio, float half) {
  const int c = blockIdx.x * 16 + (threadIdx.x >> 4), piece = threadIdx.x & 15;
  if (c >= nc) return;
  const int row = ri_kmeans_first_row(c, ratio, half, N);
  cent[((size_t)blockIdx.y * nc + c) * 16 + piece] = data[((size_t)blockIdx.y * N + row) * 16 + piece];
}

// ------------------------------------------------------------------------------------
// C entry points
// ------------------------------------------------------------------------------------
static int km_check(int P, int N, int nc) {
  if (P <= 0 || N <= 0 || nc <= 0 || P > 65535) return RI_ERR_ARG;
  return RI_OK;
}

static int km_sort_chunks(int N) { return (N + KM_SORT_CHUNK - 1) / KM_SORT_CHUNK; }

// Digits of the list sort: one when the cluster ids fit 9 bits, else an upper one, whose buckets are sorted by a workgroup
// each, and a lower one of 5 bits, or more where the upper one would have more than 9 or its table more than one round of
// the scan.  (131072 tokens, 8192 clusters: 128 buckets of 64 clusters.)  Of ten bits the lower one has four: six upper ones make a
// table that the scatter adds up itself, which leaves the scan's launch out (lists of 1 x 16400 tokens, 1024 clusters 12.4 -> 11.3 us, 1 x
// 22198, 800 12.5 -> 11.5, 8 x 17000, 544 13.4 -> 12.7, 1 x 131072, 1000 17.7 -> 14.4).
static void km_sort_bits(int N, int nc, int& lo_bits, int& hi_bits) {
  int total_bits = 1;
  while ((1 << total_bits) < nc) ++total_bits;
  lo_bits = 0;
  hi_bits = total_bits;
  if (total_bits <= 9) return;
  lo_bits = total_bits == 10 ? 4 : 5;
  while (total_bits - lo_bits > 9 ||
         (lo_bits < 7 && ((long long)km_sort_chunks(N) << (total_bits - lo_bits)) > 16 * 1024))
    ++lo_bits;
  hi_bits = total_bits - lo_bits;
}

static int km_assign_args(const void* data, const void* centroids, const int32_t* assign, int P, int N, int nc,
                          int seg) {
  if (!data || !centroids || !assign) return RI_ERR_ARG;
  if (ri_any_misaligned16(data, centroids)) return RI_ERR_ARG;
  int rc = km_check(P, N, nc);
  if (rc) return rc;
  if (nc % 32 != 0 || seg <= 0 || P % seg != 0) return RI_ERR_ARG;
  return RI_OK;
}

template <bool HALF>
static void km_assign_launch(const void* data, const void* centroids, int32_t* assign, int P, int N, int nc, int seg,
                             int64_t head_rows, bool narrow, hipStream_t stream) {
  const int shape = km_together(P) | (narrow ? KM_NARROW : 0);
#define KM_ASSIGN_LAUNCH(TT, CT, W, NB)                                                                                  \
  km_assign_kernel<TT, CT, W, NB, HALF><<<km_grid((N + W * 32 * TT - 1) / (W * 32 * TT), P), W * 64, 0, stream>>>( \
      (const uint16_t*)data, (const uint16_t*)centroids, assign, N, nc, seg, head_rows, shape)
  // Long launches: two columns, 128 registers and 32 KB of LDS, four workgroups to a compute unit; the load of one's tokens runs
  // under the others' products.  (8 x 131072 tokens, 8192 centroids: 1393 us, four columns in eight waves 1397; 8 x 96000, 3072:
  // 419 and 435; 128 x 8192, 512: 118 and 132.)  Short ones by how their 256-token pieces fall on 256 compute units: a last
  // round that is more than half full is best made of eight waves that share long tiles, one that is emptier of half as many
  // tokens per workgroup, with more LDS for each while there is one round.  Us by 256-token pieces, 512 centroids, <1, 64, 4, 2>
  // / <1, 32, 4, 3> / <1, 128, 8, 2> / <2, 32, 4, 4>: 128 7.2 / 8.1 / 8.6 / 12.4, 256 9.1 / 10.0 / 9.1 / 12.7, 350 12.7 / 13.9 /
  // 14.3 / 17.1, 420 15.3 / 17.1 / 14.6 / 17.1, 576 22.0 / 21.7 / 23.7 / 24.8, 768 27.1 / 26.6 / 26.0 / 26.8, 896 30.0 / 29.3 /
  // 31.0 / 31.4, 1024 34.3 / 33.3 / 32.8 / 34.5, 1100 36.1 / 35.1 / 37.8 / 37.8, 1400 43.7 / 43.6 / 44.9 / 43.0, 3000 89.7 / 85.6 /
  // 87.0 / 82.2; 4096 centroids: 128 40.9 / 45.5 / 47.6 / 71.3, 640 137.8 / 136.3 / 141.6 / 145.7, 1024 209.7 / 210.7 / 196.6 /
  // 196.0; 128 centroids, 1024 15.5 / 16.0 / 19.0 / 17.5.  (270 shapes of eight problems.)  Around the lines, on another card:
  // 136 8.9 / 10.1 / 8.5 / 13.2, 160 9.1 / 10.0 / 8.4 / 13.1, 192 9.1 / 10.1 / 8.5 / 13.1, 224 9.3 / 10.1 / 8.7 / 13.1; 1200 39.4 /
  // 38.1 / 37.6 / 38.9, 1280 40.3 / 39.0 / 38.1 / 40.0, 1344 42.7 / 41.4 / 43.1 / 43.8; 128 centroids, 1200 16.4 / 16.8 / 17.6 / 18.2.
  // One round that leaves compute units without work: products of 32 rows (km_assign_few_kernel / <1, 128, 8, 2>), the further
  // the longer the loop: 256 centroids, 136 pieces 5.63 / 5.72, 216 5.77 / 5.82; 512, 136 8.13 / 8.48, 176 8.12 / 8.45, 216 8.29 /
  // 8.49, 256 8.71 / 8.68; 1024, 136 13.3 / 13.9, 192 13.8 / 14.2, 208 13.9 / 14.2, 232 14.8 / 14.7; 2048, 136 24.4 / 24.9, 192 24.9 /
  // 24.9, 216 26.0 / 25.3; 4096, 136 45.4 / 45.7, 192 46.6 / 46.3; 128, 136 4.46 / 4.45.
  const long long pieces = (long long)P * ((N + 255) / 256);
  if (pieces > 128 && nc >= 256 && pieces + nc / 64 <= 224)
    km_assign_few_kernel<HALF><<<km_grid((N + 255) / 256, P), 512, 0, stream>>>(
        (const uint16_t*)data, (const uint16_t*)centroids, assign, N, nc, seg, head_rows, shape);
  else if (pieces > 1280) KM_ASSIGN_LAUNCH(2, 32, 4, 4);
  else if ((pieces - 1) % 256 >= 128 && (nc >= 256 || pieces <= 768)) KM_ASSIGN_LAUNCH(1, 128, 8, 2);
  else if (pieces <= 384) KM_ASSIGN_LAUNCH(1, 64, 4, 2);
  else KM_ASSIGN_LAUNCH(1, 32, 4, 3);
#undef KM_ASSIGN_LAUNCH
}

// a pass that knows the one before, and the tokens that it left open
template <bool HALF>
static void km_assign_again(const void* data, const void* centroids, int32_t* assign, int P, int N, int nc, int seg,
                            int64_t head_rows, const KmBounds& B, hipStream_t stream) {
  typedef KmScan<2, 32, 4, 4, HALF, true> Scan;
  km_assign_again_kernel<2, 32, 4, 4, HALF><<<dim3((N + Scan::TOKENS - 1) / Scan::TOKENS, P), 256, (size_t)nc * 2, stream>>>(
      (const uint16_t*)data, (const uint16_t*)centroids, assign, N, nc, seg, head_rows, B);
  km_assign_open_kernel<HALF><<<KM_OPEN_WGS, 256, 0, stream>>>((const uint16_t*)data, (const uint16_t*)centroids,
                                                                         assign, N, nc, seg, head_rows, B);
}

template <bool HALF>
static int km_assign(const void* data, const void* centroids, int32_t* assign, int P, int N, int nc, int seg,
                     int64_t head_rows, ri_stream_t stream) {
  int rc = km_assign_args(data, centroids, assign, P, N, nc, seg);
  if (rc) return rc;
  km_assign_launch<HALF>(data, centroids, assign, P, N, nc, seg, head_rows, false, (hipStream_t)stream);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_kmeans_assign(const void* data, const void* centroids, int32_t* assign, int P, int N,
                                int nc, int seg, int64_t head_rows, ri_stream_t stream) {
  return km_assign<false>(data, centroids, assign, P, N, nc, seg, head_rows, stream);
}

extern "C" int ri_kmeans_assign_f16(const void* data, const void* centroids, int32_t* assign, int P, int N,
                                    int nc, int seg, int64_t head_rows, ri_stream_t stream) {
  return km_assign<true>(data, centroids, assign, P, N, nc, seg, head_rows, stream);
}

extern "C" size_t ri_kmeans_workspace_bytes(int P, int N, int nc) {
  if (P <= 0 || N <= 0 || nc <= 0) return 0;
  // digit table [P, 512, chunks] + the tokens by bucket [P, N] for ids of two digits
  return ((size_t)P * KM_SORT_MAX_BINS * km_sort_chunks(N) + (size_t)P * N) * sizeof(int32_t);
}

static int km_build_lists(const int32_t* assign, int32_t* counts, int32_t* offsets, int32_t* members, int P, int N,
                          int nc, void* workspace, hipStream_t s) {
  const int nchunks = km_sort_chunks(N);
  int32_t* chunk_hist = (int32_t*)workspace;
  int32_t* toks = chunk_hist + (size_t)P * KM_SORT_MAX_BINS * nchunks;
  int lo_bits, hi_bits;
  km_sort_bits(N, nc, lo_bits, hi_bits);
  if (lo_bits == 0 && N <= KM_SMALL_MAX) {
    km_sort_small_kernel<<<P, KM_SMALL_WAVES * 64, 0, s>>>(assign, offsets, counts, members, N, nc, hi_bits);
    RI_HIP_CHECK_LAUNCH();
    return RI_OK;
  }
  const dim3 cgrid(nchunks, P);
  // (a single digit: its starts are offsets, and its counts theirs)
  const bool single = lo_bits == 0;
  const bool packed = (uint64_t)N << lo_bits <= 1ull << 32;
  const int low = single || !packed ? -1 : lo_bits;
  // Without the scan's launch, whole clusterings of ten lists, us: 1 x 20000 tokens, 512 centroids 349.4 -> 333.4, 1 x 40000, 2496 592.2 ->
  // 582.8, 4 x 32768, 2048 894.2 -> 884.8, 8 x 17000, 544 571.4 -> 567.7, 8 x 20000, 640 631.3 -> 630.0, 8 x 131072, 8192 (a table of 16384)
  // 10093 -> 10071, prefills (one list) the same.  Larger tables would be another round of every workgroup's loads, ids of less
  // than 6 bits more rows than threads add up.
  // (Where the buckets start lies behind the table, whose room is for 512 digits; 512 buckets leave none.)
  const bool table = hi_bits >= 6 && (single || hi_bits < 9) && (long long)nchunks << hi_bits <= KM_SORT_TABLE && !ri_misaligned16(chunk_hist);
  int32_t* const starts = table ? chunk_hist + ((size_t)P * nchunks << hi_bits) : chunk_hist;
  km_sort_hist_kernel<<<cgrid, 256, 0, s>>>(assign, chunk_hist, N, nchunks, lo_bits, hi_bits, table);
  RI_HIP_CHECK_LAUNCH();
  if (table) {
    km_sort_scatter_kernel<false><<<cgrid, 256, 0, s>>>(
        assign, chunk_hist, single ? members : toks, N, nchunks, lo_bits, hi_bits, low,
        KmFirsts{single ? nullptr : starts, single ? offsets : nullptr, counts, nc});
  } else {
    km_sort_scan_kernel<<<P, 1024, 0, s>>>(chunk_hist, nchunks << hi_bits, single ? offsets : nullptr,
                                           single ? counts : nullptr, nchunks, nc, N);
    RI_HIP_CHECK_LAUNCH();
    km_sort_scatter_kernel<true><<<cgrid, 256, 0, s>>>(assign, chunk_hist, single ? members : toks, N, nchunks, lo_bits,
                                                       hi_bits, low, KmFirsts{});
  }
  RI_HIP_CHECK_LAUNCH();
  if (!single) {
    const int buckets = ((nc - 1) >> lo_bits) + 1;
    km_bucket_kernel<<<dim3(buckets, P), KM_BUCKET_WAVES * 64, 0, s>>>(assign, toks, starts, counts, offsets, members, N, nc,
                                                                       table ? 1 : nchunks, lo_bits, buckets, 1 << hi_bits,
                                                                       packed);
    RI_HIP_CHECK_LAUNCH();
  }
  return RI_OK;
}

static int km_lists_args(const int32_t* assign, const int32_t* counts, const int32_t* offsets, const int32_t* members,
                         int P, int N, int nc, const void* workspace, size_t workspace_bytes) {
  if (!assign || !counts || !offsets || !members || !workspace) return RI_ERR_ARG;
  int rc = km_check(P, N, nc);
  if (rc) return rc;
  if (nc > (1 << 18)) return RI_ERR_ARG;  // two passes of at most 9 bits
  if (workspace_bytes < ri_kmeans_workspace_bytes(P, N, nc)) return RI_ERR_WORKSPACE;
  return RI_OK;
}

extern "C" int ri_kmeans_build_lists(const int32_t* assign, int32_t* counts, int32_t* offsets,
                                     int32_t* members, int P, int N, int nc, void* workspace,
                                     size_t workspace_bytes, ri_stream_t stream) {
  int rc = km_lists_args(assign, counts, offsets, members, P, N, nc, workspace, workspace_bytes);
  if (rc) return rc;
  return km_build_lists(assign, counts, offsets, members, P, N, nc, workspace, (hipStream_t)stream);
}

extern "C" size_t ri_kmeans_reduce_workspace_bytes(int P, int N, int nc) {
  if (P <= 0 || N <= 0 || nc <= 0) return 0;
  // partial [P, cap, 128] fp32
  return (size_t)P * (size_t)km_item_cap(N) * RI_DIM * sizeof(float) + 256;
}

// head_stride and row_stride in elements.  arrived (without M): [P, km_item_cap(N)] words for the blocks' arrivals, zero if `cleared`
// and zero behind the call: sums with cleared words need no launch that folds them.
template <bool MEAN, bool HALF, bool COPY>
static int km_reduce(const void* rows, int64_t head_stride, int64_t row_stride, const int32_t* counts,
                     const int32_t* offsets, const int32_t* members, void* out, int P, int N, int nc, int seg,
                     int normalize, void* copy, int64_t copy_stride, void* workspace, size_t workspace_bytes,
                     hipStream_t s, const KmMoves& M = KmMoves{}, int32_t* arrived = nullptr, bool cleared = false) {
  if (workspace_bytes < ri_kmeans_reduce_workspace_bytes(P, N, nc)) return RI_ERR_WORKSPACE;
  const int cap = km_item_cap(N);
  float2* partial = (float2*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  const int item_wgs = (cap + 3) / 4;
  if ((long long)item_wgs + (nc + 3) / 4 > 0x7fffffffLL) return RI_ERR_ARG;
  const bool ahead = !COPY && (int64_t)N * row_stride * 2 <= 0x7fffffffLL;   // (rows by offsets of 31 bits; others by address)
  auto* kernel = ahead ? km_reduce_kernel<MEAN, HALF, COPY, !COPY> : km_reduce_kernel<MEAN, HALF, COPY, false>;
  kernel<<<dim3(item_wgs + (nc + 3) / 4, P), 256, 0, s>>>(
      (const uint16_t*)rows, (size_t)row_stride / 2, counts, offsets, members, (uint16_t*)out, partial, item_wgs, cap, N,
      nc, seg, head_stride / 2, normalize, (uint16_t*)copy, copy_stride, M, cleared ? arrived : nullptr);
  RI_HIP_CHECK_LAUNCH();
  if (cleared) return RI_OK;
  km_reduce_fold_kernel<MEAN, HALF><<<dim3(item_wgs + (M.state ? 1 : 0), P), 256, 0, s>>>(offsets, partial, (uint16_t*)out,
                                                                                          cap, nc, normalize, M, N, arrived);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

template <bool HALF>
static int km_update(const void* data, const int32_t* counts, const int32_t* offsets, const int32_t* members,
                     void* centroids, int P, int N, int nc, int seg, int64_t head_rows, int normalize, void* workspace,
                     size_t workspace_bytes, ri_stream_t stream) {
  if (!data || !counts || !offsets || !members || !centroids || !workspace) return RI_ERR_ARG;
  if (ri_any_misaligned16(data, centroids, workspace)) return RI_ERR_ARG;
  int rc = km_check(P, N, nc);
  if (rc) return rc;
  if (seg <= 0 || P % seg != 0) return RI_ERR_ARG;
  return km_reduce<true, HALF, false>(data, head_rows * RI_DIM, RI_DIM, counts, offsets, members, centroids, P, N, nc, seg,
                                      normalize, nullptr, 0, workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" int ri_kmeans_update(const void* data, const int32_t* counts, const int32_t* offsets,
                                const int32_t* members, void* centroids, int P, int N, int nc, int seg,
                                int64_t head_rows, int normalize, void* workspace, size_t workspace_bytes,
                                ri_stream_t stream) {
  return km_update<false>(data, counts, offsets, members, centroids, P, N, nc, seg, head_rows, normalize, workspace,
                          workspace_bytes, stream);
}

extern "C" int ri_kmeans_update_f16(const void* data, const int32_t* counts, const int32_t* offsets,
                                    const int32_t* members, void* centroids, int P, int N, int nc, int seg,
                                    int64_t head_rows, int normalize, void* workspace, size_t workspace_bytes,
                                    ri_stream_t stream) {
  return km_update<true>(data, counts, offsets, members, centroids, P, N, nc, seg, head_rows, normalize, workspace,
                         workspace_bytes, stream);
}

template <bool HALF>
static int km_direct_launch(const void* data, const int32_t* assign, void* centroids, int32_t* counts, int32_t* offsets,
                            int32_t* members, int P, int N, int nc, int seg, int64_t head_rows, int normalize, bool narrow,
                            ri_stream_t stream) {
  // tokens compacted (4 bytes) and listed (2 bytes); block sums of a long cluster (512 bytes per KM_BLK rows) fit there too
  const size_t lds = (size_t)km_direct_run(N) * KM_DIRECT_WAVES * 6 + 512;
  const int shape = km_together(P) | (normalize ? 4 : 0) | ((P >> km_together(P)) - 1) << 3;
#define KM_DIRECT_LAUNCH_AS(CPW, NARROW)                                                                              \
  km_direct_kernel<HALF, CPW, NARROW>                                                                                 \
      <<<km_grid((nc + CPW - 1) / CPW, P), KM_DIRECT_WAVES * 64, lds, (hipStream_t)stream>>>(                         \
          (const uint16_t*)data, assign, (uint16_t*)centroids, N, nc, shape, seg, head_rows, counts, offsets, members)
#define KM_DIRECT_LAUNCH(CPW)                     \
  do {                                            \
    if (narrow) KM_DIRECT_LAUNCH_AS(CPW, true);   \
    else KM_DIRECT_LAUNCH_AS(CPW, false);         \
  } while (0)
  // As many workgroups as are resident at once (four of 512 threads, as many as the LDS of a compute unit holds): more
  // of them read the assignments more often and wait for a second round (24 x 8119 tokens, 512 clusters each: 8
  // clusters per workgroup 15.6 us, 16: 13.3, 32: 14.9; 8 x 8192: 7.5, 7.8, 10.3; 128 x 8192: 68.3, 53.3, 49.8).  Sixteen
  // waves for 16 clusters where eight have too few workgroups: late updates 7.5 -> 7.2, early ones 14.0 -> 17.5 (two
  // long lists in one workgroup wait for one compute unit's cache), so not taken.
  const long long resident = 256 * (long long)min((size_t)4, (160 * 1024) / (lds + 2560));
  const auto fits = [&](int cpw) { return (long long)P * ((nc + cpw - 1) / cpw) <= resident; };
  if (fits(8)) KM_DIRECT_LAUNCH(8);
  else if (fits(16)) KM_DIRECT_LAUNCH(16);
  else KM_DIRECT_LAUNCH(32);
#undef KM_DIRECT_LAUNCH
#undef KM_DIRECT_LAUNCH_AS
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

template <bool HALF>
static int km_update_direct(const void* data, const int32_t* assign, void* centroids, int32_t* counts, int32_t* offsets,
                            int32_t* members, int P, int N, int nc, int seg, int64_t head_rows, int normalize,
                            ri_stream_t stream) {
  if (!data || !assign || !centroids || (!counts != !members) || (!offsets != !members)) return RI_ERR_ARG;
  if (ri_any_misaligned16(data, centroids)) return RI_ERR_ARG;
  int rc = km_check(P, N, nc);
  if (rc) return rc;
  if (N > KM_DIRECT_MAX || seg <= 0 || P % seg != 0) return RI_ERR_ARG;
  return km_direct_launch<HALF>(data, assign, centroids, counts, offsets, members, P, N, nc, seg, head_rows, normalize,
                                false, stream);
}

extern "C" int ri_kmeans_lists_direct(const int32_t* assign, int32_t* counts, int32_t* offsets, int32_t* members, int P,
                                      int N, int nc, ri_stream_t stream) {
  if (!assign || !counts || !offsets || !members) return RI_ERR_ARG;
  int rc = km_check(P, N, nc);
  if (rc) return rc;
  if (N > KM_DIRECT_MAX) return RI_ERR_ARG;
  return km_direct_launch<false>(nullptr, assign, nullptr, counts, offsets, members, P, N, nc, 1, N, 0, false, stream);
}

extern "C" int ri_kmeans_update_direct(const void* data, const int32_t* assign, void* centroids, int32_t* counts,
                                       int32_t* offsets, int32_t* members, int P, int N, int nc, int seg,
                                       int64_t head_rows, int normalize, ri_stream_t stream) {
  return km_update_direct<false>(data, assign, centroids, counts, offsets, members, P, N, nc, seg, head_rows, normalize,
                                 stream);
}

extern "C" int ri_kmeans_update_direct_f16(const void* data, const int32_t* assign, void* centroids, int32_t* counts,
                                           int32_t* offsets, int32_t* members, int P, int N, int nc, int seg,
                                           int64_t head_rows, int normalize, ri_stream_t stream) {
  return km_update_direct<true>(data, assign, centroids, counts, offsets, members, P, N, nc, seg, head_rows, normalize,
                                stream);
}

// ------------------------------------------------------------------------------------
// the iterations of a clustering
// ------------------------------------------------------------------------------------
// Whether passes know the ones before.  They read every token again (8 x 131072: 55 us), which short passes are bound by
// anyway, and each is one launch more (5 us, 10 with a few tokens open).  Ten assignments and nine updates, us without / with,
// by problems, tokens and centroids, keys in clusters (as many as centroids) with four large dimensions | without any structure:
// 8 x 16400, 512: 473 / 586 | 419 / 530; 8 x 20000, 640: 572 / 664 | 498 / 598; 1 x 65536, 2048: 657 / 791 | 487 / 700; 8 x
// 20000, 1248: 760 / 796 | 684 / 616; 8 x 32768, 1024: 934 / 976 | 828 / 893; 2 x 65536, 2048: 901 / 898 | 756 / 807; 4 x 32768,
// 2048: 827 / 793 | 752 / 649; 1 x 131072, 2720: 1069 / 1058 | 926 / 1086; 2 x 65536, 4096: 1295 / 1097 | 1214 / 927; 8 x 65536,
// 1376: 1847 / 1648 | 1742 / 1807; 1 x 131072, 8192: 2325 / 1782 | 2135 / 1465; 8 x 131072, 8192: 14806 / 9586 | 14456 /
// 7570.  So from 2^29 scores a pass on.  (Up to 16384 tokens the lists never leave a workgroup, and a pass is
// bound by its keys.  64 problems: a lane each where the open tokens are dealt out; 16384 centroids: their order in LDS.)
// The more tokens a cluster has, the fewer clusters no token joins or leaves, the later; without structure none.  Without /
// with, by tokens to a centroid: 8 x 131072, 48: 5803 / 4703 | 5481 / 5407, 56: 5084 / 4266 | 4862 / 5110, 64: 4616 / 3960 | 4393 /
// 4868, 95: 3510 / 3309 | 3308 / 3972, 128: 3012 / 3007 | 2720 / 3352; 4 x 131072, 48: 3150 / 2673 | 2879 / 2922, 64: 2571 / 2323 |
// 2335 / 2635, 128: 1664 / 1731 | 1512 / 1880; 8 x 65536, 47: 1904 / 1741 | 1782 / 1875, 64: 1624 / 1579 | 1496 / 1744; 1 x 262144,
// 47: 3175 / 2731 | 2883 / 3114, 64: 2747 / 2508 | 2245 / 2697, 128: 1552 / 1615 | 1386 / 1808.  Up to 50 keys with structure
// gain more than others lose, and those lose little; past it they lose up to 30 %.
static bool km_bounded(int P, int N, int nc) {
  return N > KM_DIRECT_MAX && N <= 50ll * nc && P <= 64 && nc <= 16384 && (int64_t)P * N * nc >= 1ll << 29;
}

__global__ __launch_bounds__(KM_OPEN_WGS + 64) void km_clear_kernel(int32_t* p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0;
}

static size_t km_align256(size_t bytes) { return (bytes + 255) & ~(size_t)255; }
struct KmIterateSpace {
  size_t state, touched, best, bound, order, plan, open, open_count, partial, cleared, counts, offsets, members, lists, reduce, arrived, all;
};
static KmIterateSpace km_iterate_space(int P, int N, int nc) {
  KmIterateSpace w;
  size_t at = 0;
  const auto take = [&](size_t bytes) {
    const size_t here = at;
    at += km_align256(bytes);
    return here;
  };
  const size_t tokens = (size_t)P * N, clusters = (size_t)P * nc;
  const bool bounded = km_bounded(P, N, nc), lists = N > KM_DIRECT_MAX;
  w.state = take(bounded ? clusters * 4 : 0);
  w.touched = take(bounded ? clusters : 0);
  w.best = take(bounded ? tokens * 4 : 0);
  w.bound = take(bounded ? tokens * 4 : 0);
  w.order = take(bounded ? clusters * 2 : 0);
  w.plan = take(bounded ? (size_t)P * 8 : 0);
  w.open = take(bounded ? tokens * 4 : 0);
  w.open_count = take(bounded ? (size_t)P * 4 : 0);
  w.partial = take(bounded ? (size_t)KM_OPEN_WGS * 3 * KmOpenScan<false>::TOKENS * 4 : 0);
  w.cleared = take(bounded ? (size_t)(KM_OPEN_WGS + P) * 4 : 0);   // arrivals, odd
  w.counts = take(lists ? clusters * 4 : 0);
  w.offsets = take(lists ? (clusters + P) * 4 : 0);
  w.members = take(lists ? tokens * 4 : 0);
  w.lists = take(lists ? ri_kmeans_workspace_bytes(P, N, nc) : 0);
  w.reduce = take(lists ? ri_kmeans_reduce_workspace_bytes(P, N, nc) : 0);
  w.arrived = take(lists && !bounded ? (size_t)P * km_item_cap(N) * 4 : 0);
  w.all = at + 256;
  return w;
}

extern "C" size_t ri_kmeans_iterate_workspace_bytes(int P, int N, int nc) {
  if (P <= 0 || N <= 0 || nc <= 0) return 0;
  return km_iterate_space(P, N, nc).all;
}

template <bool HALF>
static int km_iterate(const void* data, void* centroids, int32_t* assign, int P, int N, int nc, int seg, int64_t head_rows,
                      int updates, int last, void* workspace, size_t workspace_bytes, ri_stream_t stream) {
  int rc = km_assign_args(data, centroids, assign, P, N, nc, seg);
  if (rc) return rc;
  if (updates < 0 || !workspace || (N > KM_DIRECT_MAX && nc > (1 << 18))) return RI_ERR_ARG;   // (lists of two digits)
  const KmIterateSpace w = km_iterate_space(P, N, nc);
  if (workspace_bytes < w.all) return RI_ERR_WORKSPACE;
  const bool bounded = km_bounded(P, N, nc);
  const bool narrows = N <= KM_DIRECT_MAX && N >= 8 && nc < 65536;   // (eight words, and ids that leave one over)
  hipStream_t s = (hipStream_t)stream;
  char* const base = (char*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  const KmBounds B = {(float*)(base + w.best), (float*)(base + w.bound), (const int32_t*)(base + w.state),
                      (uint8_t*)(base + w.touched), (const uint16_t*)(base + w.order), (const ri_int2*)(base + w.plan),
                      (int32_t*)(base + w.open), (int32_t*)(base + w.open_count), (int32_t*)(base + w.partial),
                      (int32_t*)(base + w.cleared), (const int32_t*)(base + w.cleared) + KM_OPEN_WGS, P};
  KmMoves M = {bounded ? (int32_t*)(base + w.state) : nullptr, B.touched, (uint16_t*)(base + w.order), (ri_int2*)(base + w.plan),
               B.open_count, B.arrived + KM_OPEN_WGS, 1};
  if (bounded) {
    km_clear_kernel<<<1, KM_OPEN_WGS + 64, 0, s>>>(B.arrived, KM_OPEN_WGS + P);
    RI_HIP_CHECK_LAUNCH();
  }
  for (int i = 0; i < updates + (last ? 1 : 0); ++i) {
    const bool narrow = narrows && i + (last ? 0 : 1) < updates;   // (the last assignment is the caller's)
    if (bounded && i > 0) km_assign_again<HALF>(data, centroids, assign, P, N, nc, seg, head_rows, B, s);
    else km_assign_launch<HALF>(data, centroids, assign, P, N, nc, seg, head_rows, narrow, s);
    RI_HIP_CHECK_LAUNCH();
    if (i == updates) break;
    if (N <= KM_DIRECT_MAX) {
      rc = km_direct_launch<HALF>(data, assign, centroids, nullptr, nullptr, nullptr, P, N, nc, seg, head_rows, 1, narrow, stream);
      if (rc) return rc;
      continue;
    }
    int32_t *const counts = (int32_t*)(base + w.counts), *const offsets = (int32_t*)(base + w.offsets),
            *const members = (int32_t*)(base + w.members);
    rc = km_build_lists(assign, counts, offsets, members, P, N, nc, base + w.lists, s);
    if (rc) return rc;
    M.first = i == 0;
    rc = km_reduce<true, HALF, false>(data, head_rows * RI_DIM, RI_DIM, counts, offsets, members, centroids, P, N, nc, seg, 1,
                                      nullptr, 0, base + w.reduce, ri_kmeans_reduce_workspace_bytes(P, N, nc), s, M,
                                      bounded ? nullptr : (int32_t*)(base + w.arrived), !bounded && i > 0);
    if (rc) return rc;
  }
  return RI_OK;
}

extern "C" int ri_kmeans_iterate(const void* data, void* centroids, int32_t* assign, int P, int N, int nc, int seg,
                                 int64_t head_rows, int updates, int last, void* workspace, size_t workspace_bytes,
                                 ri_stream_t stream) {
  return km_iterate<false>(data, centroids, assign, P, N, nc, seg, head_rows, updates, last, workspace, workspace_bytes, stream);
}

extern "C" int ri_kmeans_iterate_f16(const void* data, void* centroids, int32_t* assign, int P, int N, int nc, int seg,
                                     int64_t head_rows, int updates, int last, void* workspace, size_t workspace_bytes,
                                     ri_stream_t stream) {
  return km_iterate<true>(data, centroids, assign, P, N, nc, seg, head_rows, updates, last, workspace, workspace_bytes, stream);
}

template <bool HALF>
static int km_value_rows(const void* values, int64_t head_stride, int64_t row_stride, const int32_t* counts,
                         const int32_t* offsets, const int32_t* members, void* value_sum, void* store,
                         int64_t store_stride_rows, int P, int N, int nc, void* workspace, size_t workspace_bytes,
                         ri_stream_t stream) {
  if (!values || !counts || !offsets || !members || !value_sum || !workspace) return RI_ERR_ARG;
  if (ri_any_misaligned16(values, value_sum, store, workspace)) return RI_ERR_ARG;
  int rc = km_check(P, N, nc);
  if (rc) return rc;
  if (head_stride < 0 || row_stride < RI_DIM || (head_stride | row_stride) % 8 != 0) return RI_ERR_ARG;
  if (store && store_stride_rows < N) return RI_ERR_ARG;
  return store ? km_reduce<false, HALF, true>(values, head_stride, row_stride, counts, offsets, members, value_sum, P, N, nc,
                                              1, 0, store, store_stride_rows, workspace, workspace_bytes,
                                              (hipStream_t)stream)
               : km_reduce<false, HALF, false>(values, head_stride, row_stride, counts, offsets, members, value_sum, P, N,
                                               nc, 1, 0, nullptr, 0, workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" int ri_kmeans_value_rows(const void* values, int64_t head_stride, int64_t row_stride, const int32_t* counts,
                                    const int32_t* offsets, const int32_t* members, void* value_sum, void* store,
                                    int64_t store_stride_rows, int P, int N, int nc, void* workspace,
                                    size_t workspace_bytes, ri_stream_t stream) {
  return km_value_rows<false>(values, head_stride, row_stride, counts, offsets, members, value_sum, store,
                              store_stride_rows, P, N, nc, workspace, workspace_bytes, stream);
}

extern "C" int ri_kmeans_value_rows_f16(const void* values, int64_t head_stride, int64_t row_stride,
                                        const int32_t* counts, const int32_t* offsets, const int32_t* members,
                                        void* value_sum, void* store, int64_t store_stride_rows, int P, int N, int nc,
                                        void* workspace, size_t workspace_bytes, ri_stream_t stream) {
  return km_value_rows<true>(values, head_stride, row_stride, counts, offsets, members, value_sum, store,
                             store_stride_rows, P, N, nc, workspace, workspace_bytes, stream);
}

static int km_store_args(const void* values, int64_t v_head, int64_t v_row, const void* keys, int64_t k_head, int64_t k_row,
                         const void* mean, const void* counts, const void* offsets, const void* members, const void* value_sum,
                         const void* centroids, const void* value_store, const void* key_store, int64_t store_stride_rows, int P,
                         int N, int nc) {
  if (!values || !keys || !mean || !counts || !offsets || !members || !value_sum || !centroids || !value_store || !key_store)
    return RI_ERR_ARG;
  if (ri_any_misaligned16(values, value_sum, value_store) || ri_any_misaligned16(keys, centroids, key_store, mean))
    return RI_ERR_ARG;
  int rc = km_check(P, N, nc);
  if (rc) return rc;
  if (v_head < 0 || k_head < 0 || v_row < RI_DIM || k_row < RI_DIM || (v_head | v_row | k_head | k_row) % 8 != 0 ||
      store_stride_rows < N)
    return RI_ERR_ARG;
  return RI_OK;
}

template <bool HALF>
static int km_store_rows(const void* values, int64_t v_head, int64_t v_row, const void* keys, int64_t k_head, int64_t k_row,
                         const void* mean, const int32_t* counts, const int32_t* offsets, const int32_t* members,
                         void* value_sum, void* centroids, void* value_store, void* key_store, int64_t store_stride_rows,
                         int P, int N, int nc, void* workspace, size_t workspace_bytes, hipStream_t s,
                         const KmIndex& X = KmIndex{}) {
  int rc = km_store_args(values, v_head, v_row, keys, k_head, k_row, mean, counts, offsets, members, value_sum, centroids,
                         value_store, key_store, store_stride_rows, P, N, nc);
  if (rc) return rc;
  if (!workspace || ri_misaligned16(workspace)) return RI_ERR_ARG;
  const size_t each = ri_kmeans_reduce_workspace_bytes(P, N, nc);
  if (workspace_bytes < 2 * each) return RI_ERR_WORKSPACE;
  const int cap = km_item_cap(N), item_wgs = (cap + 3) / 4;
  if ((long long)item_wgs + (nc + 3) / 4 > 0x7fffffffLL) return RI_ERR_ARG;
  float2* const partial = (float2*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  const KmStoreArgs V = {(const uint16_t*)values, (uint16_t*)value_sum, (uint16_t*)value_store, partial,
                         (size_t)v_row / 2, v_head / 2};
  const KmStoreArgs K = {(const uint16_t*)keys, (uint16_t*)centroids, (uint16_t*)key_store,
                         partial + (size_t)P * cap * (RI_DIM / 2), (size_t)k_row / 2, k_head / 2};
  km_store_kernel<HALF><<<dim3(item_wgs + (nc + 3) / 4, P, 2), 256, 0, s>>>(V, K, (const uint16_t*)mean, counts, offsets,
                                                                            members, item_wgs, cap, N, nc,
                                                                            store_stride_rows, X);
  RI_HIP_CHECK_LAUNCH();
  km_store_fold_kernel<HALF><<<dim3(item_wgs, P, 2), 256, 0, s>>>(V, K, (const uint16_t*)mean, offsets, cap, nc, X);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

template <bool HALF>
static int km_store_index(const void* values, int64_t v_head, int64_t v_row, const void* keys, int64_t k_head, int64_t k_row,
                          const void* mean, const int32_t* counts, const int32_t* offsets, const int32_t* members,
                          void* value_sum, void* centroids, void* value_store, void* key_store, int64_t store_stride_rows,
                          void* out, uint8_t* mask, void* size16, int32_t* size, int32_t* start, int P, int N, int nc,
                          void* workspace, size_t workspace_bytes, hipStream_t s) {
  if (!out || !mask || !size16 || !size || !start || ri_any_misaligned16(out)) return RI_ERR_ARG;
  const KmIndex X = {(uint32_t*)out, mask, (uint16_t*)size16, size, start};
  return km_store_rows<HALF>(values, v_head, v_row, keys, k_head, k_row, mean, counts, offsets, members, value_sum, centroids,
                             value_store, key_store, store_stride_rows, P, N, nc, workspace, workspace_bytes, s, X);
}

template <bool HALF>
static int km_store_direct(const void* values, int64_t v_head, int64_t v_row, const void* keys, int64_t k_head,
                           int64_t k_row, const void* mean, const int32_t* assign, int32_t* counts, int32_t* offsets,
                           int32_t* members, void* value_sum, void* centroids, void* value_store, void* key_store,
                           int64_t store_stride_rows, void* out, uint8_t* mask, void* size16, int32_t* size,
                           int32_t* start, int P, int N, int nc, hipStream_t s) {
  int rc = km_store_args(values, v_head, v_row, keys, k_head, k_row, mean, counts, offsets, members, value_sum, centroids,
                         value_store, key_store, store_stride_rows, P, N, nc);
  if (rc) return rc;
  if (!assign || N > KM_DIRECT_MAX || (out && (!mask || !size16 || !size || !start || ri_misaligned16(out)))) return RI_ERR_ARG;
  const KmStoreDirect T = {{(const uint16_t*)values, (uint16_t*)value_sum, (uint16_t*)value_store, nullptr, (size_t)v_row / 2, v_head / 2},
                           {(const uint16_t*)keys, (uint16_t*)centroids, (uint16_t*)key_store, nullptr, (size_t)k_row / 2, k_head / 2},
                           (const uint16_t*)mean, store_stride_rows, {(uint32_t*)out, mask, (uint16_t*)size16, size, start}};
  const size_t lds = (size_t)km_direct_run(N) * KM_DIRECT_WAVES * 6 + 512;
  const int shape = km_together(P) | ((P >> km_together(P)) - 1) << 3;
  km_store_direct_kernel<HALF><<<km_grid((nc + 7) / 8, P), KM_DIRECT_WAVES * 64, lds, s>>>(assign, N, nc, shape, counts, offsets,
                                                                                            members, T);
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_kmeans_store_direct(const void* values, int64_t v_head, int64_t v_row, const void* keys, int64_t k_head,
                                      int64_t k_row, const void* mean, const int32_t* assign, int32_t* counts, int32_t* offsets,
                                      int32_t* members, void* value_sum, void* centroids, void* value_store, void* key_store,
                                      int64_t store_stride_rows, void* out, uint8_t* mask, void* size16, int32_t* size,
                                      int32_t* start, int P, int N, int nc, ri_stream_t stream) {
  return km_store_direct<false>(values, v_head, v_row, keys, k_head, k_row, mean, assign, counts, offsets, members, value_sum,
                                centroids, value_store, key_store, store_stride_rows, out, mask, size16, size, start, P, N, nc,
                                (hipStream_t)stream);
}

extern "C" int ri_kmeans_store_direct_f16(const void* values, int64_t v_head, int64_t v_row, const void* keys, int64_t k_head,
                                          int64_t k_row, const void* mean, const int32_t* assign, int32_t* counts, int32_t* offsets,
                                          int32_t* members, void* value_sum, void* centroids, void* value_store, void* key_store,
                                          int64_t store_stride_rows, void* out, uint8_t* mask, void* size16, int32_t* size,
                                          int32_t* start, int P, int N, int nc, ri_stream_t stream) {
  return km_store_direct<true>(values, v_head, v_row, keys, k_head, k_row, mean, assign, counts, offsets, members, value_sum,
                               centroids, value_store, key_store, store_stride_rows, out, mask, size16, size, start, P, N, nc,
                               (hipStream_t)stream);
}

extern "C" int ri_kmeans_store_index(const void* values, int64_t v_head, int64_t v_row, const void* keys, int64_t k_head,
                                     int64_t k_row, const void* mean, const int32_t* counts, const int32_t* offsets,
                                     const int32_t* members, void* value_sum, void* centroids, void* value_store,
                                     void* key_store, int64_t store_stride_rows, void* out, uint8_t* mask, void* size16,
                                     int32_t* size, int32_t* start, int P, int N, int nc, void* workspace,
                                     size_t workspace_bytes, ri_stream_t stream) {
  return km_store_index<false>(values, v_head, v_row, keys, k_head, k_row, mean, counts, offsets, members, value_sum,
                               centroids, value_store, key_store, store_stride_rows, out, mask, size16, size, start, P, N, nc,
                               workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" int ri_kmeans_store_index_f16(const void* values, int64_t v_head, int64_t v_row, const void* keys,
                                         int64_t k_head, int64_t k_row, const void* mean, const int32_t* counts,
                                         const int32_t* offsets, const int32_t* members, void* value_sum, void* centroids,
                                         void* value_store, void* key_store, int64_t store_stride_rows, void* out,
                                         uint8_t* mask, void* size16, int32_t* size, int32_t* start, int P, int N, int nc,
                                         void* workspace, size_t workspace_bytes, ri_stream_t stream) {
  return km_store_index<true>(values, v_head, v_row, keys, k_head, k_row, mean, counts, offsets, members, value_sum,
                              centroids, value_store, key_store, store_stride_rows, out, mask, size16, size, start, P, N, nc,
                              workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" int ri_kmeans_store_rows(const void* values, int64_t v_head, int64_t v_row, const void* keys, int64_t k_head,
                                    int64_t k_row, const void* mean, const int32_t* counts, const int32_t* offsets,
                                    const int32_t* members, void* value_sum, void* centroids, void* value_store,
                                    void* key_store, int64_t store_stride_rows, int P, int N, int nc, void* workspace,
                                    size_t workspace_bytes, ri_stream_t stream) {
  return km_store_rows<false>(values, v_head, v_row, keys, k_head, k_row, mean, counts, offsets, members, value_sum,
                              centroids, value_store, key_store, store_stride_rows, P, N, nc, workspace, workspace_bytes,
                              (hipStream_t)stream);
}

extern "C" int ri_kmeans_store_rows_f16(const void* values, int64_t v_head, int64_t v_row, const void* keys,
                                        int64_t k_head, int64_t k_row, const void* mean, const int32_t* counts,
                                        const int32_t* offsets, const int32_t* members, void* value_sum, void* centroids,
                                        void* value_store, void* key_store, int64_t store_stride_rows, int P, int N,
                                        int nc, void* workspace, size_t workspace_bytes, ri_stream_t stream) {
  return km_store_rows<true>(values, v_head, v_row, keys, k_head, k_row, mean, counts, offsets, members, value_sum,
                             centroids, value_store, key_store, store_stride_rows, P, N, nc, workspace, workspace_bytes,
                             (hipStream_t)stream);
}

extern "C" int ri_kmeans_value_sum(const void* values, const int32_t* counts, const int32_t* offsets,
                                   const int32_t* members, void* value_sum, int P, int N, int nc, void* workspace,
                                   size_t workspace_bytes, ri_stream_t stream) {
  return km_value_rows<false>(values, (int64_t)N * RI_DIM, RI_DIM, counts, offsets, members, value_sum, nullptr, 0, P, N, nc,
                              workspace, workspace_bytes, stream);
}

extern "C" int ri_kmeans_value_sum_f16(const void* values, const int32_t* counts, const int32_t* offsets,
                                       const int32_t* members, void* value_sum, int P, int N, int nc, void* workspace,
                                       size_t workspace_bytes, ri_stream_t stream) {
  return km_value_rows<true>(values, (int64_t)N * RI_DIM, RI_DIM, counts, offsets, members, value_sum, nullptr, 0, P, N, nc,
                             workspace, workspace_bytes, stream);
}

extern "C" int ri_permute_rows_strided(const void* in, int64_t in_head_stride, int64_t in_row_stride,
                                       const int32_t* members, void* out, int P, int N, int64_t out_stride_rows,
                                       ri_stream_t stream) {
  if (!in || !members || !out || P <= 0 || N <= 0 || P > 65535 || in_head_stride < 0 || in_row_stride < RI_DIM ||
      (in_head_stride | in_row_stride) % 8 != 0 || out_stride_rows < N)
    return RI_ERR_ARG;
  if (ri_any_misaligned16(in, out)) return RI_ERR_ARG;
  km_permute_kernel<<<dim3((N + 15) / 16, P), 256, 0, (hipStream_t)stream>>>(
      (const uint4*)in, members, (uint4*)out, N, in_head_stride / 8, in_row_stride / 8, out_stride_rows * (RI_DIM / 8));
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}

extern "C" int ri_permute_rows(const void* in, const int32_t* members, void* out, int P, int N,
                               int64_t in_stride_rows, int64_t out_stride_rows, ri_stream_t stream) {
  if (in_stride_rows < N) return RI_ERR_ARG;
  return ri_permute_rows_strided(in, in_stride_rows * RI_DIM, RI_DIM, members, out, P, N, out_stride_rows, stream);
}

extern "C" int ri_kmeans_init(const void* data, void* centroids, int P, int N, int nc, ri_stream_t stream) {
  if (!data || !centroids || ri_any_misaligned16(data, centroids)) return RI_ERR_ARG;
  int rc = km_check(P, N, nc);
  if (rc) return rc;
  const double ratio = (double)N / nc;
  km_init_kernel<<<dim3((nc + 15) / 16, P), 256, 0, (hipStream_t)stream>>>((const uint4*)data, (uint4*)centroids, N, nc,
                                                                           (float)ratio, (float)(ratio / 2));
  RI_HIP_CHECK_LAUNCH();
  return RI_OK;
}
