// g4_mm.hip -- many-token matmul on the gfx950 matrix cores: Q8_0, Q4_0, Q4_K, Q6_K and
// F16 weights in tiles of 128 tokens.
//
// Y[m][r] = sum_c W[r][c] X[m][c] for the tokens of a prompt (FloatTensor.matmul
// applied to M activation rows, FloatTensor.kt:18-29).
//
// k_split writes the activations once as three exact bf16 parts in the order
// the matrix cores take them (and, for the formats with minimums, the sum of
// every 32 columns).  k_mm then works like a plain tiled product: a workgroup
// owns 128 tokens x 128 rows and goes through the columns in stages of 64.  It
// brings a stage's parts into LDS with direct loads, unpacks each weight once to
// an exact bf16 integer (g4_mmfmt.hpp), and multiplies; each block's fp32 scale
// is applied to the block's product sums, as the one-token kernels do.
#include "g4_mmfmt.hpp"
#include "g4_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace g4 {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int MM_MT = 128;          // tokens per workgroup
constexpr int MM_NT = 128;          // weight rows per workgroup
constexpr int MM_THREADS = 512;     // 8 waves: 2 blocks of a stage x 2 token halves x 2 row halves
constexpr int MM_FRAG = 1024;       // one operand: 32 tokens x 16 columns of one part
constexpr int MM_STAGE_FRAGS = 12;  // a 32-token tile's stage: 4 x 16 columns x 3 parts

// ------------------------------------------------------------- activations ---
// Operand (t, s, k, p) -- tokens 32 t .. 32 t + 31, columns 64 s + 16 k .. + 15,
// part p -- is 1 KB at ((t * stages + s) * 12 + 3 k + p) * 1024: lane l's 16
// bytes hold token l % 32, columns 8 (l / 32) .. + 7.  Tokens past M and columns
// past dim1 are zeros.  sums[block][token]: the sum over 32 columns.  The second
// block of each stage holds -x: the matrix cores round every sum down, which long
// rows would add up to more than the sums' other errors; k_mm subtracts that
// block's sums.
//
// A wave splits 16 columns of 32 tokens, eight per lane, and stores three whole
// operands; a workgroup one stage of a token tile.  Bound by the latency of its
// loads and stores.  (A whole block of 32 columns per thread left two waves per CU
// at 512 x 2048: the Q4_K product 65.9-66.3 us, so 64.8-65.1.)
__global__ __launch_bounds__(256) void k_split(const float *x, int64_t x_stride, int32_t M, int32_t dim1, int32_t stages,
                                               int32_t tiles, unsigned char *planes, float *sums) {
  __shared__ float half[4][32];
  const int lane = threadIdx.x & 63, n = lane & 31, k = threadIdx.x >> 6;
  const int s = blockIdx.x, t = blockIdx.y;
  const int tok = t * 32 + n, col = 64 * s + 16 * k + 8 * (lane >> 5);
  const bool live = tok < M && col < dim1;
  const u32x4a4 *src = (const u32x4a4 *)(x + (live ? (int64_t)tok * x_stride + col : 0));
  u32x4a4 u0 = src[0], u1 = src[1];
  if (!live) u0 = u1 = u32x4a4{0u, 0u, 0u, 0u};
  if (k >= 2) u0 ^= 0x80000000u, u1 ^= 0x80000000u;  // the stage's second block
  const float v[8] = {__uint_as_float(u0.x), __uint_as_float(u0.y), __uint_as_float(u0.z), __uint_as_float(u0.w),
                      __uint_as_float(u1.x), __uint_as_float(u1.y), __uint_as_float(u1.z), __uint_as_float(u1.w)};
  // (an infinite x leaves NaN parts: the outputs it reaches are NaN and formed again by k_mm)
  bf16x8 p[3];
  split3<false>(v, p[0], p[1], p[2]);
  unsigned char *dst = planes + (((int64_t)t * stages + s) * MM_STAGE_FRAGS + 3 * k) * MM_FRAG + 16 * lane;
#pragma unroll
  for (int q = 0; q < 3; ++q) *(bf16x8 *)(dst + q * MM_FRAG) = p[q];
  if (sums) {
    const float sum = pstep<32>(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
    if (lane < 32) half[k][n] = sum;
    __syncthreads();
    const int b = lane >> 5;
    if (k == 0) sums[(int64_t)(2 * s + b) * (32 * tiles) + t * 32 + n] = half[2 * b][n] + half[2 * b + 1][n];
  }
}

// ----------------------------------------------------------------- weights ---
// 64 columns of a row (a stage): two blocks of 32, each four 8-column slices.  Four
// adjacent lanes share a row's stage; lane i reads its share of the raw bytes and
// unpacks it to exact bf16 integers (g4_mmfmt.hpp), Q4_K as Q4_0 with the offset
// 8 d sc - dmin m: lo() is slice i of the first block, hi() of the second.
// E: the row's first element; col: the stage's first column; two: its second block
// is inside the row (else the first one is read again, unused); g: the stage's
// group in its super-block.  scale() and offset() are those of block i / 2 (SPB = 2:
// of its half i % 2).  arrived() makes the compiler wait for the loads there and
// nowhere later.
typedef uint32_t u32x2a2 __attribute__((ext_vector_type(2), aligned(2)));

template <int TYPE>
struct MmStage;

template <>
struct MmStage<T_Q8_0> {
  static constexpr int PLANES = 1, SPB = 1;  // bf16 planes, scales per block (0: none)
  static constexpr bool MIN = false;
  u32x2 q0, q1;
  uint32_t d;
  G4_DEV void arrived() { asm volatile("" : "+v"(q0), "+v"(q1), "+v"(d)); }
  G4_DEV void load(const uint8_t *W, int64_t E, int col, bool two, int i) {
    const uint8_t *p = W + ((E + col) >> 5) * 34, *p1 = two ? p + 34 : p;
    q0 = *(const u32x2a2 *)(p + 2 + 8 * i);
    q1 = *(const u32x2a2 *)(p1 + 2 + 8 * i);
    d = *(const uint16_t *)(i < 2 ? p : p1);
  }
  G4_DEV bf16x8 lo(int, int, int) const { return sbytes_bf16(opaque(q0.x), opaque(q0.y)); }
  G4_DEV bf16x8 hi(int, int, int) const { return sbytes_bf16(opaque(q1.x), opaque(q1.y)); }
  G4_DEV float scale(int, int) const { return h2f(d); }
  G4_DEV float offset(int, int) const { return 0.f; }
};

template <>
struct MmStage<T_Q4_0> {
  static constexpr int PLANES = 1, SPB = 1;
  static constexpr bool MIN = false;
  u32x2 q0, q1;
  uint32_t d;
  G4_DEV void arrived() { asm volatile("" : "+v"(q0), "+v"(q1), "+v"(d)); }
  // slices 0 and 1 are the low nibbles of bytes 0..7 and 8..15, slices 2 and 3 the high ones
  G4_DEV void load(const uint8_t *W, int64_t E, int col, bool two, int i) {
    const uint8_t *p = W + ((E + col) >> 5) * 18, *p1 = two ? p + 18 : p;
    q0 = *(const u32x2a2 *)(p + 2 + 8 * (i & 1));
    q1 = *(const u32x2a2 *)(p1 + 2 + 8 * (i & 1));
    d = *(const uint16_t *)(i < 2 ? p : p1);
  }
  G4_DEV static uint32_t lo_s(uint32_t w) { return ((w << 4) & 0xF0F0F0F0u) ^ 0x80808080u; }
  G4_DEV static uint32_t hi_s(uint32_t w) { return (w & 0xF0F0F0F0u) ^ 0x80808080u; }
  G4_DEV static bf16x8 slice(const u32x2 &q, int i) {
    const int s = i < 2 ? 4 : 0;
    return sbytes_bf16(opaque(hi_s(q.x << s)), opaque(hi_s(q.y << s)));
  }
  G4_DEV bf16x8 lo(int, int i, int) const { return slice(q0, i); }
  G4_DEV bf16x8 hi(int, int i, int) const { return slice(q1, i); }
  G4_DEV float scale(int, int) const { return h2f(d) * 0.0625f; }
  G4_DEV float offset(int, int) const { return 0.f; }
};

template <>
struct MmStage<T_Q4_K> {
  static constexpr int PLANES = 1, SPB = 1;
  static constexpr bool MIN = true;
  u32x2 q;
  u32x4 H;
  G4_DEV void arrived() { asm volatile("" : "+v"(q), "+v"(H)); }
  G4_DEV void load(const uint8_t *W, int64_t E, int col, bool, int i) {
    const int64_t G = (E + col) >> 6;
    const uint8_t *sb = W + (G >> 2) * 144;
    H = *(const u32x4 *)sb;
    q = *(const u32x2 *)(sb + 16 + 32 * (int)(G & 3) + 8 * i);
  }
  G4_DEV bf16x8 lo(int, int, int) const { return sbytes_bf16(opaque(MmStage<T_Q4_0>::lo_s(q.x)), opaque(MmStage<T_Q4_0>::lo_s(q.y))); }
  G4_DEV bf16x8 hi(int, int, int) const { return sbytes_bf16(opaque(MmStage<T_Q4_0>::hi_s(q.x)), opaque(MmStage<T_Q4_0>::hi_s(q.y))); }
  G4_DEV float scale(int g, int i) const {
    float sc, m;
    k_scale_min(H, 2 * g + (i >> 1), sc, m);
    return h2f(H.x & 0xFFFFu) * 0.0625f * sc;
  }
  G4_DEV float offset(int g, int i) const {
    float sc, m;
    k_scale_min(H, 2 * g + (i >> 1), sc, m);
    return __builtin_fmaf(8.f, h2f(H.x & 0xFFFFu) * sc, -(h2f(H.x >> 16) * m));
  }
};

// quarter g = 2n + p of a super-block: block b of the stage has bits r = 2p + b
template <>
struct MmStage<T_Q6_K> {
  static constexpr int PLANES = 1, SPB = 2;
  static constexpr bool MIN = false;
  u32x2 q0, q1, h;
  uint32_t d;
  int sc;
  G4_DEV void arrived() { asm volatile("" : "+v"(q0), "+v"(q1), "+v"(h), "+v"(d), "+v"(sc)); }
  G4_DEV void load(const uint8_t *W, int64_t E, int col, bool, int i) {
    const int64_t G = (E + col) >> 6;
    const int n = (int)(G & 3) >> 1, p = (int)(G & 1);
    const uint8_t *sb = W + (G >> 2) * 210;
    q0 = *(const u32x2a2 *)(sb + 64 * n + 8 * i);
    q1 = *(const u32x2a2 *)(sb + 64 * n + 32 + 8 * i);
    h = *(const u32x2a2 *)(sb + 128 + 32 * n + 8 * i);
    sc = (int8_t)sb[192 + 8 * n + 4 * p + i];
    d = *(const uint16_t *)(sb + 208);
  }
  // byte 4 (q - 32): the nibble on bits 2..5, the bit pair r of its qh byte on top, the sign bit inverted
  G4_DEV static uint32_t s4(uint32_t ql, uint32_t qh, int p, int b) {
    const uint32_t nib = p ? ql >> 2 : ql << 2;
    return ((nib & 0x3C3C3C3Cu) | ((qh << (6 - 2 * (2 * p + b))) & 0xC0C0C0C0u)) ^ 0x80808080u;
  }
  G4_DEV bf16x8 lo(int g, int, int) const { return sbytes_bf16(opaque(s4(q0.x, h.x, g & 1, 0)), opaque(s4(q0.y, h.y, g & 1, 0))); }
  G4_DEV bf16x8 hi(int g, int, int) const { return sbytes_bf16(opaque(s4(q1.x, h.x, g & 1, 1)), opaque(s4(q1.y, h.y, g & 1, 1))); }
  G4_DEV float scale(int, int) const { return h2f(d) * 0.25f * (float)sc; }
  G4_DEV float offset(int, int) const { return 0.f; }
};

// (plane 0 the top 8 significant bits, plane 1 the other 3)
template <>
struct MmStage<T_F16> {
  static constexpr int PLANES = 2, SPB = 0;
  static constexpr bool MIN = false;
  u32x4 q0, q1;
  G4_DEV void arrived() { asm volatile("" : "+v"(q0), "+v"(q1)); }
  G4_DEV void load(const uint8_t *W, int64_t E, int col, bool, int i) {
    const uint8_t *p = W + (E + col) * 2 + 16 * i;
    q0 = *(const u32x4 *)p;
    q1 = *(const u32x4 *)(p + 64);
  }
  G4_DEV static bf16x8 plane(const u32x4 &q, int pl) {
    bf16x8 hi, lo;
    f16_parts(q, hi, lo);
    return pl ? lo : hi;
  }
  G4_DEV bf16x8 lo(int, int, int pl) const { return plane(q0, pl); }
  G4_DEV bf16x8 hi(int, int, int pl) const { return plane(q1, pl); }
  G4_DEV float scale(int, int) const { return 1.f; }
  G4_DEV float offset(int, int) const { return 0.f; }
};

// ----------------------------------------------------------------- product ---
struct MmArgs {
  const uint8_t *W;
  int64_t base;        // first element of row 0
  int64_t row_stride;  // elements
  int32_t rows;
  int32_t dim1;
  const unsigned char *planes;
  const float *sums;
  const float *x;  // the activations themselves (outputs that came out NaN)
  int64_t x_stride;
  int32_t M;
  int32_t tiles;   // 32-token tiles of the planes
  int32_t stages;  // 64-column stages of a row
  int32_t splits;  // column splits
  int32_t n_tt;    // token tiles of MM_MT
  int32_t n_rb;    // row blocks of MM_NT
  float *y;        // splits == 1: the output, else split s at y + s * M * rows
  int64_t y_stride;
};

// Every load (the direct ones, which the compiler's own waits do not count, among
// them) and LDS operation of the wave is done; then all waves meet.
G4_DEV void mm_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 1 KB from src (wave-uniform) + 16 * lane to LDS at byte offset `to` (wave-uniform).
G4_DEV void mm_direct_load(const unsigned char *src, uint32_t to, uint32_t lane16) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(lane16), "s"(src)
               : "memory", "m0");
}

template <int TYPE>
__global__ __launch_bounds__(MM_THREADS) void k_mm(MmArgs a) {
  using F = MmStage<TYPE>;
  constexpr int NSC = F::SPB ? F::SPB : 1;
  constexpr int ABYTES = (MM_MT / 32) * MM_STAGE_FRAGS * MM_FRAG;  // a stage's parts
  // 8 columns of 128 rows, padded (where LDS has the room) so that a row's four
  // slices, written by adjacent lanes, start on other banks
  constexpr int SLICE = MM_NT * 16 + (F::PLANES == 1 ? 32 : 0);
  constexpr int S0 = ABYTES + F::PLANES * 8 * SLICE;    // scales: 2 SPB per row
  constexpr int BUF = S0 + 2 * F::SPB * MM_NT * 4;
  // the rows' offsets and the tokens' column sums, per block, of the last four stages
  constexpr int MINS = F::MIN ? 2 * (MM_NT + MM_MT) : 0;
  constexpr int LDS = 2 * BUF + 4 * MINS * 4;
  static_assert(LDS <= 160 * 1024 && BUF % 16 == 0, "LDS");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[LDS];
  float *const mins_lds = (float *)(lds + 2 * BUF);
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, j = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kh = wid >> 2, wm = (wid >> 1) & 1, wn = wid & 1;
  // row blocks b, b + 8, ... of one XCD follow each other with all their token
  // tiles, so a row block's weights come from memory once per XCD
  int id = blockIdx.x;
  const int rb8 = id & 7;
  id >>= 3;
  const int tt = id % a.n_tt;
  id /= a.n_tt;
  const int sp = id % a.splits, rb = (id / a.splits) * 8 + rb8;
  if (rb >= a.n_rb) return;
  const int sps = (a.stages + a.splits - 1) / a.splits;
  const int s0 = sp * sps, s1 = min(a.stages, s0 + sps);  // not empty (mm_plan)
  const int r_base = rb * MM_NT, t_base = tt * (MM_MT / 32);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;
  const uint32_t lane16 = 16 * lane;

  // Stages past the end are the last one again, so that every stage does the same
  // loads and stores; what they bring is not used.
  // wave w brings operands w, w + 8, ... of a stage's 48 (tiles past the end: the
  // last one again, never stored)
  auto load_a = [&](int s, int buf) {
    const int c = min(s, s1 - 1);
#pragma unroll
    for (int k = 0; k < (MM_MT / 32) * MM_STAGE_FRAGS / 8; ++k) {
      const int f = wid + 8 * k, t = f / MM_STAGE_FRAGS, q = f - t * MM_STAGE_FRAGS;
      const int tile = min(t_base + t, a.tiles - 1);
      mm_direct_load(a.planes + (((int64_t)tile * a.stages + c) * MM_STAGE_FRAGS + q) * MM_FRAG,
                     lds0 + buf * BUF + f * MM_FRAG, lane16);
    }
  };
  // the weights this thread unpacks: row tid / 4, lane tid % 4 of its four; threads
  // 0..255 also bring a column sum
  struct Raw {
    F f;
    float xs;
  };
  const int br = tid >> 2, bi = tid & 3;
  const int64_t bE = a.base + (int64_t)min(r_base + br, a.rows - 1) * a.row_stride;
  const float *xsp = nullptr;
  if constexpr (F::MIN)
    xsp = a.sums + (int64_t)((tid >> 7) & 1) * (32 * a.tiles) + min(t_base * 32 + (tid & 127), 32 * a.tiles - 1);
  auto load_b = [&](int s, Raw &w) {
    const int c = min(s, s1 - 1);
    w.f.load(a.W, bE, 64 * c, 64 * c + 32 < a.dim1, bi);
    if constexpr (F::MIN) w.xs = xsp[(int64_t)(2 * c) * (32 * a.tiles)];
  };
  auto store_b = [&](int s, const Raw &w, int buf) {
    unsigned char *b = lds + buf * BUF + ABYTES + bi * SLICE + br * 16;
    const int c = min(s, s1 - 1), g = (int)(((bE >> 6) + c) & 3);
#pragma unroll
    for (int p = 0; p < F::PLANES; ++p) {
      *(bf16x8 *)(b + 8 * p * SLICE) = w.f.lo(g, bi, p);
      *(bf16x8 *)(b + (8 * p + 4) * SLICE) = w.f.hi(g, bi, p);
    }
    float *sc = (float *)(lds + buf * BUF + S0) + br;
    if constexpr (F::SPB == 2) {
      sc[bi * MM_NT] = w.f.scale(g, bi);
    } else if constexpr (F::SPB == 1) {
      // (lanes 2k and 2k + 1 store the same)  A second block past the row has scale
      // 0, its activations are zeros; rows of K-quants are whole stages.
      sc[(bi >> 1) * MM_NT] = F::MIN || 64 * c + 32 * (bi >> 1) < a.dim1 ? w.f.scale(g, bi) : 0.f;
    }
    if constexpr (F::MIN) {
      float *m = mins_lds + (s & 3) * MINS;
      m[(bi >> 1) * MM_NT + br] = w.f.offset(g, bi);
      m[2 * MM_NT + (tid & 255)] = w.xs;
    }
  };

  // this wave's operands of a stage: block kh, 64 rows, 64 tokens
  struct Bop {
    bf16x8 w[2][F::PLANES][2];
    float sc[2][NSC];
  };
  auto read_a = [&](int buf, int t, bf16x8 (&A)[2][3]) {
    const unsigned char *p = lds + buf * BUF + ((2 * wm + t) * MM_STAGE_FRAGS + 6 * kh) * MM_FRAG + lane16;
#pragma unroll
    for (int q = 2; q >= 0; --q)
#pragma unroll
      for (int k = 0; k < 2; ++k) A[k][q] = *(const bf16x8 *)(p + (3 * k + q) * MM_FRAG);
  };
  auto read_b = [&](int buf, Bop &B) {
    const unsigned char *p = lds + buf * BUF + ABYTES + (4 * kh + j) * SLICE + (64 * wn + n) * 16;
#pragma unroll
    for (int pl = 0; pl < F::PLANES; ++pl)
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int r = 0; r < 2; ++r) B.w[r][pl][k] = *(const bf16x8 *)(p + (8 * pl + 2 * k) * SLICE + 32 * 16 * r);
    const float *sc = (const float *)(lds + buf * BUF + S0) + kh * F::SPB * MM_NT + 64 * wn + n;
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int q = 0; q < F::SPB; ++q) B.sc[r][q] = sc[q * MM_NT + 32 * r];
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[t][r][v] = 0.f;

  // token tile t's products; small parts first: the sums' rounding is that of the last products
  auto multiply = [&](const bf16x8 (&A)[2][3], const Bop &B, f32x16 (&c)[2]) {
    if constexpr (F::SPB == 2) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        f32x16 P[2] = {};
#pragma unroll
        for (int q = 2; q >= 0; --q)
#pragma unroll
          for (int r = 0; r < 2; ++r) P[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[k][q], B.w[r][0][k], P[r], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int v = 0; v < 16; ++v) c[r][v] = __builtin_fmaf(B.sc[r][k], P[r][v], c[r][v]);
      }
    } else {
      f32x16 P[2] = {};
#pragma unroll
      for (int pl = F::PLANES - 1; pl >= 0; --pl)
#pragma unroll
        for (int q = 2; q >= 0; --q)
#pragma unroll
          for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int r = 0; r < 2; ++r)
              P[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[k][q], B.w[r][pl][k], P[r], 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int v = 0; v < 16; ++v) c[r][v] = F::SPB ? __builtin_fmaf(B.sc[r][0], P[r][v], c[r][v]) : c[r][v] + P[r][v];
    }
    // here and not later: products left waiting for their scales would not fit the registers
    asm volatile("" : "+v"(c[0]), "+v"(c[1]));
  };

  // Stage s.  On entry its second token tile is in LDS and the rest of it in
  // registers (A0, B); its barrier, half way, says that everyone is done with the
  // stage's LDS and that stage s + 1 is in the other half.  So stage s + 2 has a
  // whole stage's time to arrive, and the operands of stage s + 1 are read while
  // the second half multiplies.  w holds stage s + 2's raw weights, wn receives
  // those of s + 3.
  bf16x8 A0[2][3], A1[2][3];
  auto stage = [&](int s, int buf, const Bop &B, Bop &Bn, Raw &w, Raw &wnext) {
    read_a(buf, 1, A1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(A0, B, acc[0]);
    __builtin_amdgcn_sched_barrier(0);
    mm_barrier();
    read_b(buf ^ 1, Bn);
    read_a(buf ^ 1, 0, A0);
    __builtin_amdgcn_sched_barrier(0);
    // w has arrived (the barrier waited): said before the next loads go out, so that
    // the compiler does not wait for those where it uses w
    w.f.arrived();
    if constexpr (F::MIN) asm volatile("" : "+v"(w.xs));
    load_a(s + 2, buf);
    load_b(s + 3, wnext);
    __builtin_amdgcn_sched_barrier(0);
    multiply(A1, B, acc[1]);
    store_b(s + 2, w, buf);
    __builtin_amdgcn_sched_barrier(0);
  };

  Raw wa, wb;
  Bop Ba, Bb;
  load_a(s0, 0);
  load_b(s0, wa);
  load_b(s0 + 1, wb);
  store_b(s0, wa, 0);
  store_b(s0 + 1, wb, 1);
  load_b(s0 + 2, wa);
  mm_barrier();
  load_a(s0 + 1, 1);
  read_b(0, Ba);
  read_a(0, 0, A0);
  // the offsets' terms of the wave's block of two stages in one fp32 MFMA: lanes
  // 0..31 hold the even stage's, lanes 32..63 the odd one's (zeros: there is none)
  auto mins = [&](int s, bool both) {
    const float *m = mins_lds + ((s + j) & 3) * MINS;
    float off[2], xs[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      off[k] = m[kh * MM_NT + 64 * wn + 32 * k + n];
      xs[k] = m[2 * MM_NT + kh * MM_MT + 64 * wm + 32 * k + n];
      if (j && !both) off[k] = xs[k] = 0.f;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 2; ++r) acc[t][r] = __builtin_amdgcn_mfma_f32_32x32x2f32(xs[t], off[r], acc[t][r], 0, 0, 0);
  };
  int s = s0;
  for (; s + 1 < s1; s += 2) {
    stage(s, 0, Ba, Bb, wa, wb);
    stage(s + 1, 1, Bb, Ba, wb, wa);
    if constexpr (F::MIN) mins(s, true);
  }
  if (s < s1) {
    stage(s, 0, Ba, Bb, wa, wb);
    if constexpr (F::MIN) mins(s, false);
  }
  mm_barrier();  // the last stage's loads and stores are done: the LDS is free

  // The two blocks' sums of a tile meet through LDS: wave (kh, wm, wn) keeps row
  // tile kh and hands the other one over.
  {
    float *o = (float *)lds + (size_t)wid * 32 * 64 + lane;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[(t * 16 + v) * 64] = kh ? acc[t][0][v] : acc[t][1][v];
  }
  __syncthreads();
  float *out = a.y + (int64_t)sp * (a.splits > 1 ? (int64_t)a.M * a.rows : 0);
  const float *in = (const float *)lds + (size_t)(wid ^ 4) * 32 * 64 + lane;
  const int row = r_base + 64 * wn + 32 * kh + n;
  float got[2][16];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) got[t][v] = in[(t * 16 + v) * 64];
  RedoAny bad;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float sum = kh ? got[t][v] - acc[t][1][v] : acc[t][0][v] - got[t][v];
      const int tok = (t_base + 2 * wm + t) * 32 + 8 * (v >> 2) + 4 * j + (v & 3);
      if (tok < a.M && row < a.rows) out[(int64_t)tok * a.y_stride + row] = sum;
      bad.add(sum);  // (those past the end are zeros or a copy of the last row's)
    }
  if (__builtin_amdgcn_ballot_w64(bad.any()) == 0) return;
  // each lane reads its own outputs back, and the wave forms these again
#pragma clang loop unroll(disable)
  for (int q = 0; q < 32; ++q) {
    const int v = q & 15, tok_j = (t_base + 2 * wm + (q >> 4)) * 32 + 8 * (v >> 2) + (v & 3);  // of lane half 0
    const int tok = tok_j + 4 * j;
    const bool mine = tok < a.M && row < a.rows;
    volatile float *o = out + (int64_t)(mine ? tok : 0) * a.y_stride + (mine ? row : 0);
    float s = mine ? *o : 0.f;
    const bool again = mine && redo(s);
    const uint64_t todo = __builtin_amdgcn_ballot_w64(again);
    for (int half = 0; half < 2; ++half) {
      const uint64_t lanes = todo & (0xFFFFFFFFull << (32 * half));
      if (lanes)
        form_again<TYPE>(a.W, a.base + (int64_t)(row - n) * a.row_stride, a.row_stride, 32 * half, lanes,
                         a.x + (int64_t)(tok_j + 4 * half) * a.x_stride, 64 * s0, min(64 * s1, a.dim1), a.dim1, s);
    }
    if (again) *o = s;
  }
}

// -------------------------------------------------------------------- launch ---

namespace {

struct MmPlan {
  int splits, tiles, stages, n_tt, n_rb;
  double us;  // estimated, k_split and the sum of the splits included
};

// The column splits with the least estimated time: rounds of one workgroup per
// CU, each its stages (1.5 us: 8192 x 2048, 512 tokens) plus a start and an end,
// for splits the partial sums' way through the caches and their launch, and
// k_split.  Within 10% of the measured times from 65 to 512 tokens of 16 M weights.
MmPlan mm_plan(int type, int32_t M, int32_t rows, int32_t dim1, const DevInfo &dev) {
  MmPlan p{};
  p.stages = (dim1 + 63) / 64;
  p.tiles = (M + 31) / 32;
  p.n_tt = (M + MM_MT - 1) / MM_MT;
  p.n_rb = (rows + MM_NT - 1) / MM_NT;
  // Block sums follow one another in each accumulator, one per stage.  Up to 32
  // keep the error of the K-quants below that of the one-token kernels, up to 16
  // that of the other formats, whose kernels start from a smaller one (against 64
  // bits, 2048 columns: Q4_K 1.5e-7 here, 2.0e-7 there; Q8_0 0.9e-7 and 1.2e-7).
  const int chain = type == T_Q4_K || type == T_Q6_K ? 32 : 16;
  const int smin = (p.stages + chain - 1) / chain, smax = std::min(std::max(smin, 16), p.stages);
  double best_us = 0;
  for (int sp = smin; sp <= smax; ++sp) {
    const int sps = (p.stages + sp - 1) / sp;
    if (sps * (sp - 1) >= p.stages) continue;  // an empty split
    const int64_t wgs = (int64_t)p.n_tt * p.n_rb * sp;
    double us = (double)((wgs + dev.cu_count - 1) / dev.cu_count) * (sps * 1.5 + 5.0);
    if (sp > 1) us += 3.0 + (double)sp * M * rows * 8.0 / 8e6;
    if (p.splits == 0 || us < best_us) best_us = us, p.splits = sp;
  }
  p.us = best_us + 7.0 + (double)M * dim1 * 10.0 / 4e6;
  return p;
}

constexpr int MM_TOKENS = 1024;                       // tokens per pass over the weights
constexpr int64_t MM_PART_FLOATS = int64_t(16) << 20;  // column-split partial sums held at a time

// Rows per pass: all of them, or as many as MM_PART_FLOATS holds the splits of.
int32_t mm_rows(const MmPlan &p, int32_t M, int32_t rows) {
  if (p.splits == 1 || (int64_t)p.splits * M * rows <= MM_PART_FLOATS) return rows;
  return (int32_t)std::max<int64_t>(MM_NT, MM_PART_FLOATS / ((int64_t)p.splits * M) / MM_NT * MM_NT);
}

size_t mm_align(size_t n) { return (n + 255) & ~size_t(255); }

template <int TYPE>
hipError_t mm_launch(const MmArgs &a, hipStream_t s) {
  const dim3 grid((unsigned)((a.n_rb + 7) / 8 * 8 * a.splits * a.n_tt));
  hipLaunchKernelGGL((k_mm<TYPE>), grid, dim3(MM_THREADS), 0, s, a);
  return hipGetLastError();
}

}  // namespace

// Where the tiles of 16 tokens (k_mat, for Q4_K k_tok_q4k) take longer.  Theirs
// is about 5 us before the first row tile and, per tile of 16 waves, the time
// below (16 M weights, 512 tokens).  Measured, us, 16-token tiles / here:
//                          100 tokens    201         320         512
//   Q8_0  8192 x 2048     37.9 / 30.0  65 / 42.5   95 / 72.4  142 / 79.9
//   Q4_0  8192 x 2048     27.5 / 31.6  51 / 40.9   77 / 76.8  113 / 78.1
//   Q4_0  2048 x 8192     32.8 / 32.4  62 / 42.4   83 / 68.6  119 / 89.0
//   Q4_K  8192 x 2048     21.4 / 32.3  36 / 42.9   52 / 59.4   77 / 65.9
//   Q6_K  8192 x 2048     56.6 / 31.9  99 / 45.4  147 / 66.1  216 / 71.3
//   F16   8192 x 2048     39.9 / 36.2  70 / 54.3  103 / 94.2  151 / 107
//   Q8_0  2048 x 2048     13.0 / 22.7  20 / 24.8   27 / 29.2   38 / 31.4
// Q4_K over 408 shapes of 65 to 1024 tokens, 512 to 16384 rows and 512 to 8192
// columns: never more than 3% slower than k_tok_q4k (4096 x 512, 256 tokens 17.6 /
// 24.5; 5000 x 1024, 320 tokens 26.6 / 31.7; 16384 x 512, 512 tokens 106 / 42.8).
static bool mm_faster(int type, const TokArgs &a, const DevInfo &dev) {
  if (a.M <= 64) return false;
  const int32_t M = std::min<int32_t>(a.M, 1024);
  double tile;
  switch (type) {
    case T_Q8_0: tile = 1.95; break;
    case T_Q4_0: tile = 1.5; break;
    // (of 1024 columns and fewer, half of the waves or more have none)
    case T_Q4_K: tile = a.dim1 <= 1024 ? 0.78 : 1.1; break;
    case T_F16: tile = 2.3; break;
    default: tile = 3.1; break;  // Q6_K
  }
  const int n_sl = (a.dim1 + 127) / 128, splits = (n_sl + 15) / 16, sps = (n_sl + splits - 1) / splits;
  const int wpb = type == T_Q4_K ? 16 : sps <= 4 ? 4 : sps <= 8 ? 8 : 16, n_rt = (a.rows + 15) / 16;
  const int64_t slots = (int64_t)dev.cu_count * (16 / wpb), rest = (int64_t)splits * ((M + 15) / 16);
  const int64_t gx = std::max<int64_t>(1, std::min<int64_t>(slots / rest, n_rt));
  double us = (double)((gx * rest + slots - 1) / slots) * (5.0 + (double)((n_rt + gx - 1) / gx) * tile);
  if (splits > 1) us += 4.0 + (double)splits * M * a.rows * 8.0 / 8e6;
  return mm_plan(type, M, a.rows, a.dim1, dev).us < us;
}

bool mm_ok(int type, const TokArgs &a, const DevInfo &dev) {
  if (a.M < 1 || a.rows < 1 || a.dim1 < 1) return false;
  // whole blocks of 32 (Q8_0, Q4_0), else whole 64-column stages
  const int64_t unit = type == T_Q8_0 || type == T_Q4_0 ? 32 : 64;
  if (a.dim1 % unit != 0 || a.base % unit != 0 || a.row_stride % unit != 0) return false;
  switch (type) {
    case T_Q8_0: case T_Q4_0: case T_Q4_K: case T_Q6_K: return mm_faster(type, a, dev);
    // F16 where its error is known to stay below the one-token kernels' (0.9e-7, 1.2e-7
    // there); BF16 gains little (512 tokens 97 / 76 us)
    case T_F16: return a.dim1 <= 2048 && mm_faster(type, a, dev);
    default: return false;
  }
}

size_t mm_ws_bytes(int type, const TokArgs &a, const DevInfo &dev) {
  const int32_t mc = std::min<int32_t>(a.M, MM_TOKENS);
  const MmPlan p = mm_plan(type, mc, a.rows, a.dim1, dev);
  size_t n = mm_align((size_t)p.tiles * p.stages * MM_STAGE_FRAGS * MM_FRAG);
  n += mm_align(sizeof(float) * (size_t)2 * p.stages * 32 * p.tiles);
  if (p.splits > 1) n += mm_align(sizeof(float) * (size_t)p.splits * mc * mm_rows(p, mc, a.rows));
  return n;
}

hipError_t launch_mm(int type, const TokArgs &t, void *ws, const DevInfo &dev, hipStream_t s) {
  if (!mm_ok(type, t, dev) || !ws) return hipErrorInvalidValue;
  const int32_t mc0 = std::min<int32_t>(t.M, MM_TOKENS);
  // one plan (that of a full pass) for every pass: the workspace is laid out for it
  const MmPlan full = mm_plan(type, mc0, t.rows, t.dim1, dev);
  const int32_t rc0 = mm_rows(full, mc0, t.rows);
  unsigned char *planes = (unsigned char *)ws;
  float *sums = (float *)(planes + mm_align((size_t)full.tiles * full.stages * MM_STAGE_FRAGS * MM_FRAG));
  float *part = (float *)((unsigned char *)sums + mm_align(sizeof(float) * (size_t)2 * full.stages * 32 * full.tiles));
  const bool mins = type == T_Q4_K;
  for (int32_t m0 = 0; m0 < t.M; m0 += mc0) {
    MmPlan p = full;
    const int32_t M = std::min(mc0, t.M - m0);
    p.tiles = (M + 31) / 32;
    p.n_tt = (M + MM_MT - 1) / MM_MT;
    const float *x = t.x + (int64_t)m0 * t.x_stride;
    hipLaunchKernelGGL(k_split, dim3((unsigned)p.stages, (unsigned)p.tiles), dim3(256), 0, s, x, t.x_stride, M,
                       t.dim1, p.stages, p.tiles, planes, mins ? sums : (float *)nullptr);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    for (int32_t r0 = 0; r0 < t.rows; r0 += rc0) {
      MmArgs a{};
      a.W = t.W;
      a.base = t.base + (int64_t)r0 * t.row_stride;
      a.row_stride = t.row_stride;
      a.rows = std::min(rc0, t.rows - r0);
      a.dim1 = t.dim1;
      a.planes = planes;
      a.sums = sums;
      a.x = x;
      a.x_stride = t.x_stride;
      a.M = M;
      a.tiles = p.tiles;
      a.stages = p.stages;
      a.splits = p.splits;
      a.n_tt = p.n_tt;
      a.n_rb = (a.rows + MM_NT - 1) / MM_NT;
      float *y = t.y + (int64_t)m0 * t.y_stride + r0;
      a.y = p.splits > 1 ? part : y;
      a.y_stride = p.splits > 1 ? a.rows : t.y_stride;
      switch (type) {
        case T_Q8_0: e = mm_launch<T_Q8_0>(a, s); break;
        case T_Q4_0: e = mm_launch<T_Q4_0>(a, s); break;
        case T_Q4_K: e = mm_launch<T_Q4_K>(a, s); break;
        case T_Q6_K: e = mm_launch<T_Q6_K>(a, s); break;
        default: e = mm_launch<T_F16>(a, s); break;
      }
      if (e != hipSuccess) return e;
      if (p.splits > 1) {
        e = launch_tok_reduce(part, p.splits, M, a.rows, y, t.y_stride, s);
        if (e != hipSuccess) return e;
      }
    }
  }
  return hipSuccess;
}

}  // namespace g4
