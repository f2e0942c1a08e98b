// f32 products on the bf16 matrix cores without loss of precision.
//
// gfx950 multiplies bf16 sixteen times as fast as f32 (dense 2.5 PFLOP/s
// against 157 TFLOP/s). A float is the sum of three bf16 values, exactly:
// the nearest bf16 (8 significant bits), the nearest bf16 of what is left
// (at most 16 bits), and the rest (at most 8 bits). Of the nine products of
// two such triples, the six largest,
//   a1 b1 + (a1 b2 + a2 b1) + (a1 b3 + a2 b2 + a3 b1),
// leave out |a2 b3| + |a3 b2| + |a3 b3| <= (2^-23 + 2^-32) |a b|: each bf16
// product is exact in f32, so the sum is as good as an f32 multiply-add's
// (rounded to 2^-24), at 6/16 of its matrix-core time. The products other than a1 b1
// are at most 2^-7 of the whole, so summing them in an accumulator of their
// own keeps the count of full-size roundings at one per product, as in f32.
//
// Infinities, NaN, values that round past bf16's largest, and sums within
// 2^-7 of f32's largest come out of this as an infinity or NaN: a kernel
// recomputes such an output by f32 multiply-adds.
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
  const float ra = a - __uint_as_float(p1 << 16), rb = b - __uint_as_float(p1 & 0xffff0000u);
  p2 = split_pack(ra, rb);
  p3 = split_pack(ra - __uint_as_float(p2 << 16), rb - __uint_as_float(p2 & 0xffff0000u));
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

// The six products of one 16 x 16 x 32 step over MT x NT blocks: the largest
// to `hi`, the rest, smallest first, to `lo`. Product by product, so that a
// block's dependent steps lie MT * NT apart.
template <int MT, int NT>
__device__ __forceinline__ void split_mma(const bf16x8 (&a)[MT][3], const bf16x8 (&b)[NT][3], split_f4 (&hi)[MT][NT],
                                          split_f4 (&lo)[MT][NT]) {
  constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
  for (int s = 0; s < 6; s++)
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++) {
        split_f4 &c = s == 5 ? hi[i][j] : lo[i][j];
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][pa[s]], b[j][pb[s]], c, 0, 0, 0);
      }
}

}  // namespace ppocr
