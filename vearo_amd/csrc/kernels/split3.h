// split3.h -- f32 products on the bf16 matrix cores without losing f32 precision.
//
// An f32 value is the exact sum of three bf16 values, x = h + m + l: h is x
// rounded to bf16 (8 significant bits, round to nearest even), m the remainder
// x - h (exact in f32) rounded to bf16, l what is left (at most 8 bits, so exact
// again). bf16 has f32's exponent range and the matrix cores take and return
// subnormals, so (scaled, below) this holds from f32's smallest to ~5e33.
// A product then needs six of the nine part products,
//   x y = h h' + (h m' + m h') + (h l' + m m' + l h') + [m l' + l m' + l l'],
// the bracket being below 2^-24 |x y| (|m| <= 2^-8 |h|, |l| <= 2^-16 |h|, halved
// on average, signs random: ~2^-27 in the mean).
//
// What it buys: v_mfma_f32_32x32x16_bf16 does 16 times the products per cycle
// of v_mfma_f32_32x32x2_f32 (1024 against 64 multiply-adds a cycle and SIMD, so
// six of them are 2.7 times the f32 rate), and it sums eight products exactly
// before it rounds once into the f32 accumulator, where the f32 instruction
// rounds after every product. Six part products of 16 k are 12 roundings
// against 16, the five small ones at a step where little is lost. Measured on
// MI355X against 64-bit sums, 2-norm relative error of the f32 instruction ->
// this split, N(0, 1) operands: K = 64 1.45e-7 -> 1.09e-7, 768 4.98e-7 ->
// 4.22e-7, 3072 9.91e-7 -> 8.61e-7, 16384 2.29e-6 -> 2.08e-6; one-signed
// operands K = 16384 1.98e-6 -> 1.29e-6; a weight gradient's mixture of a few
// large and many tiny same-signed terms (dlogits^T x) K = 16384 6.3e-5 -> 5.1e-6.
//
// Scale. bf16 ends at 2^-133 where f32 ends at 2^-149, so the parts of values
// below ~2^-110 would lose bits: operands are multiplied by 2^16 before they are
// split (exact, subnormals included) and the sums by 2^-32 after.
//
// What it cannot do: an infinity or a NaN has no such parts (inf - inf), nor has
// a finite value that is infinite as bf16 once scaled (above 5.2e33); sums overflow
// from 7.9e28. All of these give an infinity or a NaN in every output they reach,
// so an accumulator that comes out finite is right, and a wave that finds one that
// is not recomputes its 32 x 32 tile on the f32 instruction, which has IEEE's answer,
// and takes from there the elements that were not finite, and only those: what one
// output is does not depend on the values of another's row or column.
#pragma once
#include "common.h"

typedef float vh_f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 vh_bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 vh_bf8 __attribute__((ext_vector_type(8)));
typedef float vh_f2 __attribute__((ext_vector_type(2)));
typedef uint32_t vh_u4 __attribute__((ext_vector_type(4)));
typedef float s3_f4u __attribute__((ext_vector_type(4), aligned(4)));  // at any float's address

// Two values -> their three parts, each pair packed in one register (x0 low):
// three v_cvt_pk_bf16_f32, four subtractions and four half extractions.
VH_DEV void s3_split2(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
  auto pk = [](float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((vh_f2{a, b}), vh_bf2));
  };
  auto lo = [](uint32_t p) { return __builtin_bit_cast(float, p << 16); };
  auto hi = [](uint32_t p) { return __builtin_bit_cast(float, p & 0xFFFF0000u); };
  h = pk(x0, x1);
  const float r0 = x0 - lo(h), r1 = x1 - hi(h);
  m = pk(r0, r1);
  l = pk(r0 - lo(m), r1 - hi(m));
}

// Eight consecutive k of one row -> the three parts as 16-byte fragments.
VH_DEV void s3_split8(const float (&x)[8], vh_u4 (&p)[3]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t h, m, l;
    s3_split2(x[2 * i], x[2 * i + 1], h, m, l);
    p[0][i] = h;
    p[1][i] = m;
    p[2][i] = l;
  }
}

// 4 x 4 transpose of t[0..3] across the wave's four 16-lane rows: lane 16 q + c ends
// with t[j] = what lane 16 j + c held in t[q]. Two register-pair swaps between
// wave halves, two between neighbouring rows (v_permlane32_swap, v_permlane16_swap).
VH_DEV void s3_transpose4(uint32_t (&t)[4]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const auto r = __builtin_amdgcn_permlane32_swap(t[j], t[j + 2], false, false);
    t[j] = r[0];
    t[j + 2] = r[1];
  }
#pragma unroll
  for (int j = 0; j < 4; j += 2) {
    const auto r = __builtin_amdgcn_permlane16_swap(t[j], t[j + 1], false, false);
    t[j] = r[0];
    t[j + 1] = r[1];
  }
}

// acc += a b over 16 k from the operands' part fragments (part 0 = h, 1 = m,
// 2 = l), part product T of six, the smallest first (measured: 4.22e-7 against
// 4.28e-7 the other way round at K = 768, 1.09e-7 against 1.35e-7 at K = 64).
VH_DEV vh_f32x16 s3_mfma(const vh_u4& a, const vh_u4& b, const vh_f32x16& acc) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(vh_bf8, a), __builtin_bit_cast(vh_bf8, b), acc,
                                                 0, 0, 0);
}
#define S3_SCALE 65536.0f                // on each operand (2^16)
#define S3_UNSCALE 2.3283064365386963e-10f  // on their products' sum (2^-32)
#define S3_PA(T) ((T) == 0 ? 2 : (T) == 1 ? 0 : (T) == 2 ? 1 : (T) == 3 ? 1 : 0)  // A's part in product T
#define S3_PB(T) ((T) == 0 ? 0 : (T) == 1 ? 2 : (T) == 2 ? 1 : (T) == 4 ? 1 : 0)  // B's part

// The registers of a 32 x 32 accumulator tile (bit r: register r) that hold an
// infinity or a NaN in a row below mlim and a column below nlim, both counted from the
// lane's first row and its column. One register after the other: sixteen lane masks at
// once would take the scalar registers that the callers' loops keep their state in.
VH_DEV uint32_t s3_nonfinite_regs(const vh_f32x16& acc, int64_t mlim, int64_t nlim) {
  const int ml = nlim <= 0 || mlim < 0 ? 0 : mlim < 32 ? (int)mlim : 32;
  uint32_t bad = 0;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const uint32_t below = (uint32_t)(8 * (r >> 2) + (r & 3) - ml) >> 31;
    bad |= __builtin_fabsf(acc[r]) < __builtin_inff() ? 0u : below << r;
    asm volatile("" : "+v"(bad));
  }
  return bad;
}

// Whether any of a wave's accumulators is an infinity or a NaN (x * 0 is then NaN).
template <int I, int J>
VH_DEV bool s3_nonfinite(const vh_f32x16 (&acc)[I][J]) {
  float z[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) z[r & 3] = __builtin_fmaf(acc[i][j][r], 0.0f, z[r & 3]);
  const float s = (z[0] + z[1]) + (z[2] + z[3]);
  return __builtin_amdgcn_ballot_w64(!(s == 0.0f)) != 0;
}
