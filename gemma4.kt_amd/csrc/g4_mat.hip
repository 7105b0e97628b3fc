// g4_mat.hip -- several-token matmul on the gfx950 matrix cores for Q8_0, Q4_0,
// Q5_K, Q6_K, BF16 and F16 weights (Q4_K: g4_tok.hip).
//
// Y[m][r] = sum_c W[r][c] X[m][c] for M tokens (FloatTensor.matmul applied to M
// activation rows, FloatTensor.kt:18-29).  Products are exact: an fp32 activation
// splits into three bf16 parts, a weight is an exact bf16 integer times its
// block's scale (g4_mmfmt.hpp).
//
// Work split, as k_tok_q4k's: a wave keeps 16 tokens x 128 columns of x split in
// registers and walks the workgroup's 16-row tiles; the waves of a workgroup take
// adjacent columns, and their partial tiles are summed through LDS in a fixed order
// (deterministic).  More tokens are further workgroups, which share a row block's
// weights through the L2.  Rows of more than 2048 columns split over workgroups,
// whose partial sums launch_tok_reduce adds in order.
//
// Weights: a wave reads a tile's 16 rows x 128 columns with adjacent lanes on
// adjacent bytes, unpacks each weight once and passes it through its own LDS into
// the MFMA layout (no barrier: a wave reads only what it wrote).
//
// Bound by the latency of a tile's loads and the barrier after it, then by the
// cache lines its load instructions touch; neither the unpacking nor the products
// show (timing variants without them: 1-4% faster).  Measured at 8192 x 2048, us per
// launch (one segment of the row engine per token -> here):
//              8 tokens       19            64             512
//   Q8_0     15.1 -> 10.0  46.5 -> 14.2   81.9 -> 23.6   623 -> 142
//   Q4_0     12.0 ->  7.7  24.9 -> 10.8   71.6 -> 17.0   548 -> 113
//   Q5_K     17.2 ->  9.8  39.7 -> 13.4  108.1 -> 21.3   833 -> 124
//   Q6_K     23.1 -> 14.0  53.1 -> 20.4  140.5 -> 34.7   999 -> 216
//   BF16     34.0 -> 10.8  90.5 -> 12.5  233.2 -> 19.2  1791 -> 98.9
//   F16      40.2 -> 12.2 101.0 -> 15.6  247.9 -> 24.5  1898 -> 151
// and against 64 bits the error falls from 1.2e-7..3.0e-7 to 0.7e-7..1.5e-7 (512 to
// 32768 columns).
#include "g4_mmfmt.hpp"
#include "g4_internal.hpp"

#include <algorithm>

namespace g4 {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int MAT_COLS = 128;  // columns per wave

template <int TYPE>
constexpr bool mat_half = TYPE == T_BF16 || TYPE == T_F16;

// What a lane holds of a tile on its way from memory
template <int TYPE, bool HALF = mat_half<TYPE>>
struct MatRaw {
  static constexpr int SPB = MmFmt<TYPE>::SPB;
  static constexpr bool MIN = MmFmt<TYPE>::MIN;
  MmFmt<TYPE> f;  // quarter lane % 4 of row lane / 4
};
template <int TYPE>
struct MatRaw<TYPE, true> {
  static constexpr int SPB = 0;
  static constexpr bool MIN = false;
  u32x4 q[4];  // columns 8 (lane % 16) .. + 7 of rows 4 k + lane / 16
};

// Workgroup (row block x, column split y, 16-token tile z), sps slices of
// MAT_COLS columns per split, one per wave.
template <int TYPE, int WPB>
__global__ __launch_bounds__(WPB * 64) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_mat(TokArgs a, int sps) {
  constexpr bool HALF = mat_half<TYPE>;
  using Raw = MatRaw<TYPE>;
  constexpr int SPB = Raw::SPB;
  constexpr bool MIN = Raw::MIN;
  // LDS of a wave: first its x (16 tokens x 128 columns, rows padded so that the
  // reads are conflict-free); then, after a barrier, the partial tiles of the
  // workgroup (two, alternating) and each wave's weights: [block][piece][row] of
  // 16 bytes, padded so that what adjacent lanes write is on other banks, and the
  // rows' scales and offsets (and for MIN [block][token] the sums of x)
  constexpr int XROW = 132, PIECE = 16 * 16 + 16;
  constexpr int RED = 2 * WPB * 1024, WB = 16 * PIECE, WS = 16 * 4 * SPB * 4, WO = MIN ? 2 * 16 * 4 * 4 : 0;
  static_assert(2048 + WB + WS + WO <= 16 * XROW * 4, "the weights' LDS is the x's");
  __shared__ __attribute__((aligned(16))) unsigned char lds[WPB * 16 * XROW * 4];
  f32x4(*red)[WPB][64] = (f32x4(*)[WPB][64])lds;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, j = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sl0 = (int)blockIdx.y * sps, n_sl = (a.dim1 + MAT_COLS - 1) / MAT_COLS;
  const int nw = min(sps, n_sl - sl0);  // slices of this split (wave-uniform, as everything here)
  const int col0 = (sl0 + wid) * MAT_COLS;
  const int ng = wid < nw ? min(2, (a.dim1 - col0 + 63) >> 6) : 0;  // the wave's stages
  const int tok0 = (int)blockIdx.z * 16, mt = min(16, a.M - tok0);
  const int n_rt = (a.rows + 15) >> 4;
  const int rpb = (n_rt + gridDim.x - 1) / gridDim.x;
  const int rt0 = min(n_rt, (int)blockIdx.x * rpb), rt1 = min(n_rt, rt0 + rpb);
  if (rt0 >= rt1) return;  // the whole workgroup

  // x: adjacent lanes on adjacent 16-byte pieces, an instruction two tokens' 512 bytes
  u32x4a4 xg[8];
  {
    const int c = lane & 31;
    const bool live = col0 + 4 * c < a.dim1 && ng > 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (8 * h < mt) {
#pragma unroll
        for (int q = 4 * h; q < 4 * h + 4; ++q) {
          const int t = 2 * q + (lane >> 5);  // tokens past M: the tile's first (never stored)
          xg[q] = *(const u32x4a4 *)(a.x + (int64_t)(tok0 + (t < mt ? t : 0)) * a.x_stride + (live ? col0 + 4 * c : 0));
        }
      } else {
#pragma unroll
        for (int q = 4 * h; q < 4 * h + 4; ++q) xg[q] = u32x4a4{0u, 0u, 0u, 0u};
      }
    }
    // columns past the end are zeros
    if (ng > 0 && col0 + MAT_COLS > a.dim1)
#pragma unroll
      for (int q = 0; q < 8; ++q) xg[q] = live ? xg[q] : u32x4a4{0u, 0u, 0u, 0u};
  }

  // The weights of row tile rt.  16 rows are whole super-blocks, so a lane's place in
  // its row's bytes is the same in every tile.  Rows past the end, and waves past the
  // columns, read the matrix's first row (never used).
  const int lr = lane >> 2, li = lane & 3;
  const int left = min(4, (a.dim1 - col0 + 31) >> 5);  // blocks of the wave's slice inside the row
  const int64_t e0 = a.base + (int64_t)(rt0 * 16) * a.row_stride;
  auto load = [&](int rt, Raw &w) {
    const int64_t et = e0 + (int64_t)((rt - rt0) * 16) * a.row_stride;  // the tile's first row
    if constexpr (HALF) {
      const int c = ng > 0 && 8 * (lane & 15) < 64 * ng ? col0 + 8 * (lane & 15) : 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int r = 4 * k + (lane >> 4);
        const int64_t e = rt * 16 + r < a.rows ? et + (int64_t)r * a.row_stride : a.base;
        w.q[k] = *(const u32x4 *)(a.W + 2 * (e + c));
      }
    } else {
      const int64_t e = (rt * 16 + lr < a.rows ? et + (int64_t)lr * a.row_stride : a.base) + (ng > 0 ? col0 : 0);
      w.f.load(MmFmt<TYPE>::at(a.W, e), (int)(e >> 7) & 1, ng > 0 ? left : 1, li);
    }
  };
  const int h = (int)((a.base + (int64_t)lr * a.row_stride + col0) >> 7) & 1;
  unsigned char *const wl = lds + RED + wid * (WB + WS + WO);
  float *const ws = (float *)(wl + WB), *const wo = (float *)(wl + WB + WS), *const wx = wo + 64;
  auto put = [&](const Raw &w) {
    if constexpr (HALF) {
#pragma unroll
      for (int k = 0; k < 4; ++k) *(u32x4 *)(wl + (lane & 15) * PIECE + (4 * k + (lane >> 4)) * 16) = w.q[k];
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int at = MmFmt<TYPE>::at(k, li);
        const bf16x8 v = w.f.piece(k, h, li);
        if constexpr (SPB == 2) {
          // columns in the order of two 16-column products: piece j holds columns
          // 4j .. 4j + 3 of the block's first half and of its second
          const u32x4 u = __builtin_bit_cast(u32x4, v);
          unsigned char *c = wl + ((at & ~3) + 2 * (at & 1)) * PIECE + lr * 16 + 8 * ((at >> 1) & 1);
          *(u32x2 *)c = u32x2{u.x, u.y};
          *(u32x2 *)(c + PIECE) = u32x2{u.z, u.w};
        } else {
          *(bf16x8 *)(wl + at * PIECE + lr * 16) = v;
        }
      }
      // a block past the columns has scale 0 (its x is zeros)
#pragma unroll
      for (int k = 0; k < SPB; ++k) ws[(lr * 4 + li) * SPB + k] = li < left ? w.f.scale(k, h, li) : 0.f;
      if constexpr (MIN) wo[lr * 4 + li] = li < left ? w.f.offset(h, li) : 0.f;
    }
  };
  // the first tile's weights go out behind the x loads
  __builtin_amdgcn_sched_barrier(0);
  Raw wr;
  load(rt0, wr);
  __builtin_amdgcn_sched_barrier(0);

  // x back in the MFMA layout, lane (j, n) piece j of token n, split into its parts
  bf16x8 A[4][3];
  {
    float *xst = (float *)lds + wid * 16 * XROW;
#pragma unroll
    for (int q = 0; q < 8; ++q) *(u32x4 *)(xst + (2 * q + (lane >> 5)) * XROW + 4 * (lane & 31)) = xg[q];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float *p = xst + n * XROW + 32 * b + (SPB == 2 ? 4 * j : 8 * j);
      const u32x4 u0 = *(const u32x4 *)p, u1 = *(const u32x4 *)(p + (SPB == 2 ? 16 : 4));
      float v[8];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[k] = __uint_as_float(u0[k]), v[4 + k] = __uint_as_float(u1[k]);
        if (b & 1) v[k] = -v[k], v[4 + k] = -v[4 + k];  // (see the block sums)
      }
      split3<false>(v, A[b][0], A[b][1], A[b][2]);
    }
  }
  __syncthreads();  // every wave has its x: the LDS now holds weights and partial tiles
  put(wr);
  if constexpr (MIN) {
    // sum of x over each block, by the instructions and in the order of the products
    bf16x8 one;
#pragma unroll
    for (int e = 0; e < 8; ++e) one[e] = (__bf16)1.0f;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      f32x4 S = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = 2; p >= 0; --p) S = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[b][p], one, S, 0, 0, 0);
      if (n == 0) *(f32x4 *)(wx + 16 * b + 4 * j) = S;
    }
  }

  float *out = gridDim.y == 1 ? a.y : a.part + (int64_t)blockIdx.y * a.M * a.rows;
  const int64_t out_stride = gridDim.y == 1 ? a.y_stride : a.rows;
  RedoAny bad;
  uint64_t bad_min = 0;  // (MIN has no registers left for it: 512 tokens of Q5_K 143 us, 124 so)
  for (int rt = rt0, buf = 0; rt < rt1; ++rt, buf ^= 1) {
    bf16x8 B[4];
    f32x4 sc[SPB == 2 ? 2 : 1];
    f32x4 of = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 4; ++b) B[b] = *(const bf16x8 *)(wl + (4 * b + j) * PIECE + n * 16);
#pragma unroll
    for (int k = 0; k < SPB; ++k) sc[k] = *(const f32x4 *)(ws + n * 4 * SPB + 4 * k);
    if constexpr (MIN) of = *(const f32x4 *)(wo + n * 4);
    __builtin_amdgcn_sched_barrier(0);
    load(min(rt + 1, rt1 - 1), wr);
    __builtin_amdgcn_sched_barrier(0);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (ng > 0) {
      // small parts first: the sums' rounding is that of the last products
      f32x4 P[4][SPB == 2 ? 2 : 1];
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int k = 0; k < (SPB == 2 ? 2 : 1); ++k) P[b][k] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (TYPE == T_F16) {
        // (two blocks at a time: the parts of four would not fit the registers, 19
        // tokens of 8192 x 2048 22.0 us, 15.8 so)
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          if (g >= ng) continue;
          bf16x8 H[2], L[2];
#pragma unroll
          for (int b = 0; b < 2; ++b) f16_parts(__builtin_bit_cast(u32x4, B[2 * g + b]), H[b], L[b]);
#pragma unroll
          for (int p = 2; p >= 0; --p)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              f32x4 &c = P[2 * g + b][0];
              c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[2 * g + b][p], L[b], c, 0, 0, 0);
              c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[2 * g + b][p], H[b], c, 0, 0, 0);
            }
        }
      } else
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          if (HALF && b >= 2 * ng) continue;  // (x zero times a weight from elsewhere, perhaps infinite)
          if constexpr (SPB == 2) {
            typedef struct {
              s16x4 h[2];
            } Halves;
            const Halves x2 = __builtin_bit_cast(Halves, A[b][p]), w2 = __builtin_bit_cast(Halves, B[b]);
#pragma unroll
            for (int k = 0; k < 2; ++k)
              P[b][k] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x2.h[k], w2.h[k], P[b][k], 0, 0, 0);
          } else {
            P[b][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[b][p], B[b], P[b][0], 0, 0, 0);
          }
        }
      // Odd blocks multiply -x: the matrix cores round every sum down, which long rows
      // would add up to more than the sums' other errors.
      if constexpr (HALF)
        acc = (P[0][0] - P[1][0]) + (P[2][0] - P[3][0]);
      else
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        f32x4 S;
        if constexpr (MIN) S = *(const f32x4 *)(wx + 16 * b + 4 * j);
        const float sign = b & 1 ? -1.f : 1.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (SPB == 2) {
            acc[i] = __builtin_fmaf(sign * sc[b >> 1][2 * (b & 1)], P[b][0][i], acc[i]);
            acc[i] = __builtin_fmaf(sign * sc[b >> 1][2 * (b & 1) + 1], P[b][1][i], acc[i]);
          } else if constexpr (MIN) {
            acc[i] += sign * (rounded(sc[0][b] * P[b][0][i]) - rounded(of[b] * S[i]));
          } else if constexpr (SPB == 1) {
            acc[i] = __builtin_fmaf(sign * sc[0][b], P[b][0][i], acc[i]);
          }
        }
      }
    }
    red[buf][wid][lane] = acc;
    put(wr);
    __syncthreads();
    // the slices summed pairwise (fewer roundings than one after the other): wave c
    // takes component c of every lane's four
    if (wid < 4) {
      const float *rp = (const float *)&red[buf][0][lane] + wid;
      float v[WPB];
#pragma unroll
      for (int w = 0; w < WPB; ++w) v[w] = rp[w * 64 * 4];
#pragma unroll
      for (int d = WPB / 2; d >= 1; d >>= 1)
#pragma unroll
        for (int w = 0; w < d; ++w) v[w] = v[2 * w] + v[2 * w + 1];
      float s = v[0];
      const int r = rt * 16 + n, m = 4 * j + wid;
      const bool mine = r < a.rows && m < mt;
      if (mine) out[(int64_t)(tok0 + m) * out_stride + r] = s;
      if constexpr (MIN)
        bad_min |= __builtin_amdgcn_ballot_w64(mine && redo(s));
      else
        bad.add(mine ? s : 0.f);
    }
  }
  if ((MIN ? bad_min : __builtin_amdgcn_ballot_w64(bad.any())) == 0) return;
  // Waves 0..3: each lane reads its own outputs back, and the wave forms these again
  // (here and not where they are stored: in the loop it would cost registers, 19
  // tokens of Q8_0 14.2 -> 14.9 us, Q6_K 22.4 -> 25.3).
  for (int rt = rt0; rt < rt1; ++rt) {
    const int r = rt * 16 + n, m = 4 * j + wid;
    const bool mine = r < a.rows && m < mt;
    volatile float *o = out + (int64_t)(tok0 + (mine ? m : 0)) * out_stride + (mine ? r : 0);
    float s = mine ? *o : 0.f;
    const bool again = mine && redo(s);
    const uint64_t todo = __builtin_amdgcn_ballot_w64(again);
    for (int l0 = 0; l0 < 64; l0 += 16) {  // token 4 (l0 / 16) + wid
      const uint64_t lanes = todo & (0xFFFFull << l0);
      if (lanes)
        form_again<TYPE>(a.W, a.base + (int64_t)(rt * 16) * a.row_stride, a.row_stride, l0, lanes,
                         a.x + (int64_t)(tok0 + l0 / 4 + wid) * a.x_stride, sl0 * MAT_COLS,
                         min(a.dim1, (sl0 + nw) * MAT_COLS), a.dim1, s);
    }
    if (again) *o = s;
  }
}

namespace {

struct MatShape {
  int splits, sps, wpb, gx;
};

MatShape mat_shape(const TokArgs &a, const DevInfo &dev) {
  MatShape s;
  const int n_sl = (a.dim1 + MAT_COLS - 1) / MAT_COLS;
  s.splits = (n_sl + 15) / 16;
  s.sps = (n_sl + s.splits - 1) / s.splits;
  s.splits = (n_sl + s.sps - 1) / s.sps;
  s.wpb = s.sps <= 4 ? 4 : s.sps <= 8 ? 8 : 16;
  const int n_rt = (a.rows + 15) / 16;
  // 16 waves per CU at a time, spread over every (split, token tile)
  const int64_t gx = (int64_t)dev.cu_count * (16 / s.wpb) / ((int64_t)s.splits * ((a.M + 15) / 16));
  s.gx = (int)std::max<int64_t>(1, std::min<int64_t>(gx, n_rt));
  return s;
}

template <int TYPE>
hipError_t launch_mat_t(const TokArgs &a, const MatShape &sh, hipStream_t s) {
  const dim3 grid((unsigned)sh.gx, (unsigned)sh.splits, (unsigned)((a.M + 15) / 16));
  if (sh.wpb == 4)
    hipLaunchKernelGGL((k_mat<TYPE, 4>), grid, dim3(256), 0, s, a, sh.sps);
  else if (sh.wpb == 8)
    hipLaunchKernelGGL((k_mat<TYPE, 8>), grid, dim3(512), 0, s, a, sh.sps);
  else
    hipLaunchKernelGGL((k_mat<TYPE, 16>), grid, dim3(1024), 0, s, a, sh.sps);
  return hipGetLastError();
}

}  // namespace

bool mat_ok(int type, const TokArgs &a) {
  if (a.M < 1 || a.rows < 1 || a.dim1 < 1) return false;
  // whole blocks (Q8_0, Q4_0), whole slices (K-quants), whole 64-column groups (16 bits)
  const int64_t unit = type == T_Q8_0 || type == T_Q4_0 ? 32 : type == T_Q5_K || type == T_Q6_K ? 128 : 64;
  if (a.dim1 % unit != 0 || a.base % unit != 0 || a.row_stride % unit != 0) return false;
  switch (type) {
    case T_Q8_0: case T_Q4_0: case T_Q5_K: case T_Q6_K: case T_BF16: case T_F16: return true;
    default: return false;
  }
}

// A launch takes 4 us (512 columns) to 10 us (column splits) before its first tile;
// the row engine takes about as little for its first round of waves and jumps where
// M * rows starts the next one (16384 outputs of up to 4096 columns in the 32- and
// 256-weight blocks).  So the line is a number of outputs, and a fewest M below which
// the row engine's segments are as fast on any matrix.  Measured, us, row engine /
// here, on either side of the line:
//   Q8_0   1024 x 512,  8 tokens  3.2 / 3.7     2048 x 512,  5   4.3 / 3.8
//          1024 x 2048, 16        5.8 / 7.3     17               7.4 / 7.3
//          4096 x 2048, 4         6.1 / 6.8     5                9.5 / 6.8
//          1024 x 8192, 8         9.5 / 9.6     9               11.1 / 10.1
//   Q4_0   2048 x 2048, 12        6.3 / 6.7     14               8.2 / 6.8
//          4096 x 4096, 6         9.8 / 10.3    7               11.5 / 10.3
//   Q5_K   1024 x 2048, 16        6.8 / 8.2     17               8.7 / 8.4
//   Q6_K   1024 x 2048, 16        8.1 / 9.9     17              10.6 / 10.4
//   BF16   1024 x 2048, 4         5.6 / 5.7     5                8.0 / 5.7
//          512 x 8192, 4          7.5 / 8.3     5               11.0 / 8.3
//   F16    1024 x 2048, 4         7.1 / 8.8     5               12.3 / 8.7
// Over 760 shapes a type (256 to 16384 rows, 512 to 8192 columns, 3 to 64 tokens) the
// route taken is never more than 3.2% slower than the row engine.
int32_t mat_min_tokens(int type, const TokArgs &a) {
  int64_t outputs;
  if (type == T_BF16 || type == T_F16)
    outputs = a.dim1 <= 2048 ? 4096 : a.dim1 <= 4096 ? 4608 : 2048;
  else if (type == T_Q4_0)
    outputs = a.dim1 <= 512 ? 8192 : a.dim1 <= 1024 ? 16384 : a.dim1 <= 4096 ? 24576 : 12288;
  else
    outputs = a.dim1 <= 512 ? 8192 : a.dim1 <= 4096 ? 16384 : type == T_Q6_K ? 4608 : 8192;
  return (int32_t)std::max<int64_t>(type == T_BF16 || type == T_F16 ? 3 : 5, outputs / a.rows + 1);
}

// Tokens per pass: as many as MAT_PART_FLOATS holds the column splits' sums of.
constexpr int64_t MAT_PART_FLOATS = int64_t(16) << 20;
static int32_t mat_pass(const TokArgs &a, const MatShape &sh) {
  if (sh.splits == 1) return a.M;
  return (int32_t)std::min<int64_t>(a.M, std::max<int64_t>(16, MAT_PART_FLOATS / ((int64_t)sh.splits * a.rows) / 16 * 16));
}

int64_t mat_scratch_floats(const TokArgs &a, const DevInfo &dev) {
  const MatShape sh = mat_shape(a, dev);
  return sh.splits > 1 ? (int64_t)sh.splits * mat_pass(a, sh) * a.rows : 0;
}

hipError_t launch_mat(int type, const TokArgs &t, const DevInfo &dev, hipStream_t s) {
  if (!mat_ok(type, t)) return hipErrorInvalidValue;
  const int32_t pass = mat_pass(t, mat_shape(t, dev));
  TokArgs a = t;
  for (int32_t m0 = 0; m0 < t.M; m0 += pass) {
    a.M = std::min(pass, t.M - m0);
    a.x = t.x + (int64_t)m0 * t.x_stride;
    a.y = t.y + (int64_t)m0 * t.y_stride;
    const MatShape sh = mat_shape(a, dev);
    if (sh.splits > 1 && !a.part) return hipErrorInvalidValue;
    hipError_t e;
    switch (type) {
      case T_Q8_0: e = launch_mat_t<T_Q8_0>(a, sh, s); break;
      case T_Q4_0: e = launch_mat_t<T_Q4_0>(a, sh, s); break;
      case T_Q5_K: e = launch_mat_t<T_Q5_K>(a, sh, s); break;
      case T_Q6_K: e = launch_mat_t<T_Q6_K>(a, sh, s); break;
      case T_BF16: e = launch_mat_t<T_BF16>(a, sh, s); break;
      default: e = launch_mat_t<T_F16>(a, sh, s); break;
    }
    if (e == hipSuccess && sh.splits > 1) e = launch_tok_reduce(a.part, sh.splits, a.M, a.rows, a.y, a.y_stride, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace g4
