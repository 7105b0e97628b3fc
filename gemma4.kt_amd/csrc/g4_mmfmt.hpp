// g4_mmfmt.hpp -- weights as matrix-core operands, for the GGUF types the
// several-token kernels take.
//
// A weight is scale * integer + offset, the integer an exact bf16:
//
//   type   integer        value range   scale (per)       offset (per 32)
//   Q8_0   q              -128..127     d (32)            --
//   Q4_0   16 (q - 8)     -128..112     d / 16 (32)       --
//   Q5_K   8 q            0..248        d sc / 8 (32)     -dmin m
//   Q6_K   4 (q - 32)     -128..124     d sc / 4 (16)     --
//   BF16   the weight                   1                 --
//   F16    the weight as two bf16 (8 and 3 significant bits)
//
// (The matrix cores do not take subnormal bf16 operands exactly: the smaller parts of
// activations below about 2^-110 are.  Sums of nothing larger are formed again, see
// redo(); activations that are themselves subnormal, below 2^-126, count as 0.)
// Every integer has at most 8 significant bits, so the products with the three
// bf16 parts of an fp32 activation are exact.  Scales are exact in fp32 (11 x 8
// bits), and so are offsets.  Centred integers keep the sums' rounding at the
// size of |weight|.  A block whose weights are all exactly zero contributes
// exactly 0; for Q5_K under the conditions FmtQ5_K states (its q all one power of
// two): the sum of x is formed by the same matrix instructions as the sum of q x,
// and the two products are rounded on their own.
#pragma once

#include "g4_device.hpp"

namespace g4 {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2a4 __attribute__((ext_vector_type(2), aligned(4)));
// GGUF blocks of 18, 34 and 210 bytes start at 2 mod 4: the amdhsa targets'
// unaligned access mode takes these loads as they are
typedef uint32_t u32x4a2 __attribute__((ext_vector_type(4), aligned(2)));

// x = p1 + p2 + p3 exactly: p1 and p2 are the bf16 truncations of x and of
// x - p1 (their top 8 significant bits), x - p1 - p2 has at most 8 significant
// bits, and both differences are exact in fp32.  Truncation keeps every part of
// a finite x finite.  GUARD: an infinite x stays in p1 with zero residuals;
// without it x - p1 is NaN there, which the caller detects.  A NaN x gives NaN
// parts either way.
template <bool GUARD>
G4_DEV void split3(const float (&v)[8], bf16x8 &p1, bf16x8 &p2, bf16x8 &p3) {
  uint32_t t1[8], t2[8], t3[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    t1[e] = __float_as_uint(v[e]) & 0xFFFF0000u;
    float r1 = v[e] - __uint_as_float(t1[e]);
    if (GUARD) r1 = __builtin_isinf(v[e]) ? 0.f : r1;
    t2[e] = __float_as_uint(r1) & 0xFFFF0000u;
    t3[e] = __float_as_uint(r1 - __uint_as_float(t2[e]));
  }
  // two values' upper halves per dword (v_perm_b32)
  u32x4 a, b, c;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    a[k] = __builtin_amdgcn_perm(t1[2 * k + 1], t1[2 * k], 0x07060302u);
    b[k] = __builtin_amdgcn_perm(t2[2 * k + 1], t2[2 * k], 0x07060302u);
    c[k] = __builtin_amdgcn_perm(t3[2 * k + 1], t3[2 * k], 0x07060302u);
  }
  p1 = __builtin_bit_cast(bf16x8, a);
  p2 = __builtin_bit_cast(bf16x8, b);
  p3 = __builtin_bit_cast(bf16x8, c);
}

// bf16 of the eight signed bytes of v0 and v1
G4_DEV bf16x8 sbytes_bf16(uint32_t v0, uint32_t v1) {
  bf16x8 r;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    r[b] = (__bf16)sbyte(v0, b);
    r[4 + b] = (__bf16)sbyte(v1, b);
  }
  return r;
}

// bf16 of the eight unsigned bytes of v0 and v1
G4_DEV bf16x8 ubytes_bf16(uint32_t v0, uint32_t v1) {
  bf16x8 r;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    r[b] = (__bf16)ubyte(v0, b);
    r[4 + b] = (__bf16)ubyte(v1, b);
  }
  return r;
}

// sc and m of sub-block j of a K-quant head (q4k_scale_min on its registers,
// without a branch: j differs between lanes)
G4_DEV void k_scale_min(const u32x4 &H, int j, float &sc, float &m) {
  const uint32_t s8 = 8u * (uint32_t)(j & 3), k = (uint32_t)(j >> 2);
  const uint32_t y = H.y >> (s8 + 2 * k), z = H.z >> (s8 + 2 * k), w = H.w >> s8;
  const uint32_t mw = 15u * k, my = 63u - mw;  // j >= 4: four bits from w, two from y or z
  sc = (float)((w & mw) | (y & my));
  m = (float)(((w >> 4) & mw) | (z & my));
}

// A slice is 128 columns of a row: four blocks of 32, each four pieces of 8.
// Four adjacent lanes share a row's slice, lane i a quarter of its bytes in as
// few and wide loads as they allow (the load instructions, each over 16 rows, bound
// the kernels before the arithmetic does).
//   at(W, e): the bytes of the slice that starts at element e, a multiple of 32
//     (Q8_0, Q4_0) or 128 (Q5_K, Q6_K; h = e / 128 % 2, its half of the super-block).
//   load(): left: blocks of the slice inside the row, 1..4; later ones read the
//     last again (K-quant slices are whole).
//   piece(k), k = 0..3: 8 columns, piece at(k) % 4 of block at(k) / 4.
//   scale(), offset() (its negative): of block i (Q6_K: of its two halves).
template <int TYPE>
struct MmFmt;

template <>
struct MmFmt<T_Q8_0> {
  static constexpr int SPB = 1;  // scales per block
  static constexpr bool MIN = false;
  u32x4 q[2];
  uint32_t d;
  G4_DEV static const uint8_t *at(const uint8_t *W, int64_t e) { return W + (e >> 5) * 34; }
  G4_DEV void load(const uint8_t *p, int, int left, int i) {
    p += 34 * min(i, left - 1);
    d = *(const uint16_t *)p;
    q[0] = *(const u32x4a2 *)(p + 2);
    q[1] = *(const u32x4a2 *)(p + 18);
  }
  G4_DEV static int at(int k, int i) { return 4 * i + k; }
  G4_DEV bf16x8 piece(int k, int, int) const {
    return sbytes_bf16(opaque(q[k >> 1][2 * (k & 1)]), opaque(q[k >> 1][2 * (k & 1) + 1]));
  }
  G4_DEV float scale(int, int, int) const { return h2f(d); }
  G4_DEV float offset(int, int) const { return 0.f; }
};

template <>
struct MmFmt<T_Q4_0> {
  static constexpr int SPB = 1;
  static constexpr bool MIN = false;
  u32x4 q;
  uint32_t d;
  G4_DEV static const uint8_t *at(const uint8_t *W, int64_t e) { return W + (e >> 5) * 18; }
  G4_DEV void load(const uint8_t *p, int, int left, int i) {
    p += 18 * min(i, left - 1);
    d = *(const uint16_t *)p;
    q = *(const u32x4a2 *)(p + 2);
  }
  G4_DEV static int at(int k, int i) { return 4 * i + k; }
  // pieces 0 and 1 are the low nibbles of bytes 0..7 and 8..15, pieces 2 and 3 the high ones
  G4_DEV bf16x8 piece(int k, int, int) const {
    const int s = k < 2 ? 4 : 0, w = 2 * (k & 1);
    return sbytes_bf16(opaque(((q[w] << s) & 0xF0F0F0F0u) ^ 0x80808080u),
                       opaque(((q[w + 1] << s) & 0xF0F0F0F0u) ^ 0x80808080u));
  }
  G4_DEV float scale(int, int, int) const { return h2f(d) * 0.0625f; }
  G4_DEV float offset(int, int) const { return 0.f; }
};

// lane i: bytes 16 (i % 2) .. + 15 of the slice's group i / 2 (64 weights: the low
// nibbles are its first block, the high ones its second)
template <>
struct MmFmt<T_Q5_K> {
  static constexpr int SPB = 1;
  static constexpr bool MIN = true;
  u32x4 q, b, H;
  G4_DEV static const uint8_t *at(const uint8_t *W, int64_t e) { return W + (e >> 8) * 176; }
  G4_DEV void load(const uint8_t *p, int h, int, int i) {
    H = *(const u32x4 *)p;
    b = *(const u32x4 *)(p + 16 + 16 * (i & 1));
    q = *(const u32x4 *)(p + 48 + 64 * h + 16 * i);
  }
  G4_DEV static int at(int k, int i) { return 4 * (2 * (i >> 1) + (k >> 1)) + 2 * (i & 1) + (k & 1); }
  // byte 8 q: the nibble on bits 3..6, the fifth bit (bit s of its byte) on top
  G4_DEV static uint32_t u8(uint32_t nib, uint32_t hb, int s) {
    return (nib & 0x78787878u) | ((hb << (7 - s)) & 0x80808080u);
  }
  G4_DEV bf16x8 piece(int k, int h, int i) const {
    const int w = 2 * (k & 1), s = 4 * h + 2 * (i >> 1) + (k >> 1);
    return k < 2 ? ubytes_bf16(opaque(u8(q[w] << 3, b[w], s)), opaque(u8(q[w + 1] << 3, b[w + 1], s)))
                 : ubytes_bf16(opaque(u8(q[w] >> 1, b[w], s)), opaque(u8(q[w + 1] >> 1, b[w + 1], s)));
  }
  G4_DEV float scale(int, int h, int i) const {
    float sc, m;
    k_scale_min(H, 4 * h + i, sc, m);
    return h2f(H.x & 0xFFFFu) * 0.125f * sc;
  }
  G4_DEV float offset(int h, int i) const {
    float sc, m;
    k_scale_min(H, 4 * h + i, sc, m);
    return h2f(H.x >> 16) * m;
  }
};

// Half h of a super-block, block r = 0..3: its nibbles are the low (r < 2) or high
// ones of ql[64 h + 32 (r % 2) ..], its upper bits the pair r of qh[32 h ..].  Lane i:
// 16 bytes of ql, weights 16 (i % 2) .. + 15 of blocks i / 2 and i / 2 + 2.
template <>
struct MmFmt<T_Q6_K> {
  static constexpr int SPB = 2;
  static constexpr bool MIN = false;
  u32x4 q, b;
  uint32_t d, sc;
  G4_DEV static const uint8_t *at(const uint8_t *W, int64_t e) { return W + (e >> 8) * 210; }
  G4_DEV void load(const uint8_t *p, int h, int, int i) {
    q = *(const u32x4a2 *)(p + 64 * h + 16 * i);
    b = *(const u32x4a2 *)(p + 128 + 32 * h + 16 * (i & 1));
    sc = *(const uint16_t *)(p + 192 + 8 * h + 2 * i);
    d = *(const uint16_t *)(p + 208);
  }
  G4_DEV static int at(int k, int i) { return 4 * ((i >> 1) + 2 * (k >> 1)) + 2 * (i & 1) + (k & 1); }
  // byte 4 (q - 32): the nibble on bits 2..5, the bit pair r on top, the sign bit inverted
  G4_DEV static uint32_t s4(uint32_t nib, uint32_t qh, int r) {
    return ((nib & 0x3C3C3C3Cu) | ((qh << (6 - 2 * r)) & 0xC0C0C0C0u)) ^ 0x80808080u;
  }
  G4_DEV bf16x8 piece(int k, int, int i) const {
    const int w = 2 * (k & 1), r = (i >> 1) + 2 * (k >> 1);
    return k < 2 ? sbytes_bf16(opaque(s4(q[w] << 2, b[w], r)), opaque(s4(q[w + 1] << 2, b[w + 1], r)))
                 : sbytes_bf16(opaque(s4(q[w] >> 2, b[w], r)), opaque(s4(q[w + 1] >> 2, b[w + 1], r)));
  }
  G4_DEV float scale(int half, int, int) const { return h2f(d) * 0.25f * sbyte(sc, half); }
  G4_DEV float offset(int, int) const { return 0.f; }
};

// The two bf16 parts of eight F16 weights: the top 8 significant bits and the
// other 3 (the difference is exact).  Subnormals are 0, as in the vector path
// (h2f_vec).  Exponent 31, finite there, is infinite or NaN here and makes every
// sum it enters so: the caller forms such sums again.  (8192 x 2048, 19 and 64
// tokens: 24.2 and 38.5 us with h2f_vec's decode of each weight, 20.8 and 32.0 so,
// before the parts were made two blocks at a time.)
G4_DEV void f16_parts(const u32x4 &q, bf16x8 &hi, bf16x8 &lo) {
  u32x4 a, b;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float v[2], r[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      v[i] = h2f(i ? q[k] >> 16 : q[k]);
      v[i] = __builtin_fabsf(v[i]) < 0x1p-14f ? 0.f : v[i];
      r[i] = v[i] - __uint_as_float(__float_as_uint(v[i]) & 0xFFFF0000u);
    }
    a[k] = __builtin_amdgcn_perm(__float_as_uint(v[1]), __float_as_uint(v[0]), 0x07060302u);
    b[k] = __builtin_amdgcn_perm(__float_as_uint(r[1]), __float_as_uint(r[0]), 0x07060302u);
  }
  hi = __builtin_bit_cast(bf16x8, a);
  lo = __builtin_bit_cast(bf16x8, b);
}

// A matrix-core sum that is formed again in fp32 from the decoded weights:
//  - NaN or infinite: an infinite or NaN activation or weight (an infinity's residual
//    parts are NaN; F16 exponent 31 is finite), or a block sum that overflowed, the
//    integers being up to 128 times the weight's own scale;
//  - below 2^-60, not 0: activations so small that their residual parts are subnormal,
//    which the matrix cores do not take exactly.
G4_DEV bool redo(float s) {
  return !__builtin_isfinite(s) || (__builtin_fabsf(s) < 0x1p-60f && s != 0.f);
}

// Whether redo() holds for any of several sums, in four instructions each: the
// largest and the smallest magnitude but 0 as integers (twice the bits, less one: 0
// wraps to the largest).
struct RedoAny {
  uint32_t hi = 0u, lo = ~0u;
  G4_DEV void add(float s) {
    const uint32_t u = __float_as_uint(s) << 1;
    hi = max(hi, u);
    lo = min(lo, u - 1u);
  }
  G4_DEV bool any() const { return hi >= 0xFF000000u || lo < 0x42FFFFFFu; }
};

// The sums of one token (x, columns [c0, c1)) that the lanes of the set `lanes` hold
// in s, lane l's that of row l - l0 of the rows from element E on: formed again one
// after the other by the whole wave, adjacent lanes on adjacent columns.  (With each
// lane on its own, 8192 x 2048 Q5_K at 19 tokens took 2.3 ms for one NaN or infinite
// activation, where it takes 33 and 67 us; F16 at 512 tokens with one row of exponent
// 31 took 5.3 ms, now 0.5.)
template <int TYPE>
G4_DEV void form_again(const uint8_t *W, int64_t E, int64_t row_stride, int l0, uint64_t lanes, const float *x, int c0,
                       int c1, int dim1, float &s) {
  const int lane = threadIdx.x & 63;
  uint32_t infs = 0;  // bit k: column c0 + lane + 64 k (of at most 2048) is infinite
#pragma clang loop unroll(disable)
  for (int k = 0; c0 + 64 * k < c1; ++k) {
    const int c = c0 + lane + 64 * k;
    const float v = c < c1 ? x[c] : 0.f;
    if (__builtin_amdgcn_ballot_w64(v != v)) {  // with a NaN, every sum is NaN
      s = (lanes >> lane) & 1 ? __builtin_nanf("") : s;
      return;
    }
    infs |= (uint32_t)__builtin_isinf(v) << k;
  }
  // next to infinite activations the others do not count, where weights are finite
  // (F16 exponent 31 is)
  const bool inf_only = TYPE != T_BF16 && __builtin_amdgcn_ballot_w64(infs != 0) != 0;
  while (lanes) {
    const int l = __builtin_ctzll(lanes);
    lanes &= lanes - 1;
    const int64_t e = E + (int64_t)(l - l0) * row_stride;
    float t = 0.f;
    if (inf_only)
      for (uint32_t m = infs; m; m &= m - 1) {
        const int c = c0 + lane + 64 * __builtin_ctz(m);
        t = __builtin_fmaf(dot_elem<TYPE>(W, e + c, c, dim1), x[c], t);
      }
    else
#pragma clang loop unroll(disable)
      for (int cb = c0 + lane; cb < c1; cb += 512) {
        // eight columns' loads in flight; those past the end are the last one's, not added
        float w[8], v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int c = min(cb + 64 * k, c1 - 1);
          w[k] = dot_elem<TYPE>(W, e + c, c, dim1);
          v[k] = x[c];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) t = cb + 64 * k < c1 ? __builtin_fmaf(w[k], v[k], t) : t;
      }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) t += __shfl_xor(t, d, 64);
    s = lane == l ? t : s;
  }
}

}  // namespace g4
