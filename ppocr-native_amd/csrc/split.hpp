// f32 products on the bf16 matrix cores, at f32's precision.
//
// gfx950 multiplies bf16 sixteen times as fast as f32 (dense 2.5 PFLOP/s
// against 157 TFLOP/s). A finite float is exactly the sum of three bf16
// values at scales 1, 2^-8 and 2^-16,
//   a = a1 + 2^-8 a2 + 2^-16 a3:
// the nearest bf16 (8 significant bits), the nearest bf16 of 2^8 times what is
// left (at most 16 bits), and 2^8 times the rest (at most 8 bits). The scales
// keep the parts of small values above bf16's smallest step: a1 goes down to
// 2^-133, so 2^-16 a3 to f32's own 2^-149. (The method, without the scales:
// Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence
// Datatype For Higher-Precision Computations", 2019.)
//
// Of the nine products of two such triples, the six largest,
//   a1 b1 + 2^-8 (a1 b2 + a2 b1) + 2^-16 (a1 b3 + a2 b2 + a3 b1),
// leave out at most (2^-23 + 2^-32) |a b|, where an f32 multiply-add's product
// is exact: of one product alone up to two f32 roundings (2^-24 each) are
// lost, in a sum less than its own roundings. Each bf16 product is exact in
// f32. Each scale has an accumulator of its own; the products at 2^-8 and
// 2^-16 are at most 2^-7 of the whole, so the count of full-size roundings
// stays at one per product, as in f32. (Below 2^-126, f32's smallest normal
// value, what is left out is a subnormal factor's own step, 2^-149, times the
// other factor at most.)
//
// Infinities, NaN, values that round past bf16's largest, and sums within
// 2^-7 of f32's largest come out of this as an infinity or NaN: such an output
// is recomputed by f32 multiply-adds (conv_f32; the CTC head's rows, whose sum
// of exponentials it leaves NaN, by ctc_merge).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ppocr {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float split_f2 __attribute__((ext_vector_type(2)));
typedef float split_f4 __attribute__((ext_vector_type(4)));
typedef uint32_t split_u4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t split_pack(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(split_f2{a, b}, bf16x2));
}

// The three parts of two floats (a in the low halves).
__device__ __forceinline__ void split_pair(float a, float b, uint32_t &p1, uint32_t &p2, uint32_t &p3) {
  p1 = split_pack(a, b);
  const float ra = (a - __uint_as_float(p1 << 16)) * 256.0f, rb = (b - __uint_as_float(p1 & 0xffff0000u)) * 256.0f;
  p2 = split_pack(ra, rb);
  p3 = split_pack((ra - __uint_as_float(p2 << 16)) * 256.0f, (rb - __uint_as_float(p2 & 0xffff0000u)) * 256.0f);
}

// Eight consecutive reduction values as MFMA operands: element 2h in the low
// half of dword h.
__device__ __forceinline__ void split8(split_f4 lo, split_f4 hi, split_u4 &p1, split_u4 &p2, split_u4 &p3) {
  const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  uint32_t a[4], b[4], c[4];
#pragma unroll
  for (int h = 0; h < 4; h++) split_pair(x[2 * h], x[2 * h + 1], a[h], b[h], c[h]);
  p1 = split_u4{a[0], a[1], a[2], a[3]};
  p2 = split_u4{b[0], b[1], b[2], b[3]};
  p3 = split_u4{c[0], c[1], c[2], c[3]};
}
__device__ __forceinline__ void split8(split_f4 lo, split_f4 hi, bf16x8 (&p)[3]) {
  split_u4 a, b, c;
  split8(lo, hi, a, b, c);
  p[0] = __builtin_bit_cast(bf16x8, a), p[1] = __builtin_bit_cast(bf16x8, b), p[2] = __builtin_bit_cast(bf16x8, c);
}

// The six products in the order they are issued (smallest first) and each
// one's scale, 2^(-8 * scale): parts a[kSplitA[s]] and b[kSplitB[s]].
constexpr int kSplitA[6] = {2, 0, 1, 1, 0, 0}, kSplitB[6] = {0, 2, 1, 0, 1, 0}, kSplitScale[6] = {2, 2, 2, 1, 1, 0};

// A block's accumulators, one a scale, and their sum.
struct SplitAcc {
  split_f4 s[3];
};
__device__ __forceinline__ split_f4 split_sum(const SplitAcc &a) {
  constexpr float k = 1.0f / 256.0f;
  split_f4 v;
#pragma unroll
  for (int r = 0; r < 4; r++) v[r] = fmaf(fmaf(a.s[2][r], k, a.s[1][r]), k, a.s[0][r]);
  return v;
}

// The six products of one 16 x 16 x 32 step over MT x NT blocks, product by
// product, so that a block's dependent steps lie MT * NT apart.
template <int MT, int NT>
__device__ __forceinline__ void split_mma(const bf16x8 (&a)[MT][3], const bf16x8 (&b)[NT][3], SplitAcc (&acc)[MT][NT]) {
#pragma unroll
  for (int s = 0; s < 6; s++)
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++) {
        split_f4 &c = acc[i][j].s[kSplitScale[s]];
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][kSplitA[s]], b[j][kSplitB[s]], c, 0, 0, 0);
      }
}

}  // namespace ppocr
