// float32 products on the bfloat16 matrix cores (gfx950).
//
// A float is the sum of three bfloat16 values, x = h + m + l (round to nearest at each step:
// 8 + 8 + 8 significant bits and two signs hold all 24), and a product of two such sums is
// kept to its six largest terms: hh, hm, mh, hl, lh, mm (the three-term bfloat16 split of Henry,
// Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", ARITH 2019). The dropped terms ml, lm, ll are below 2^-24 of
// the product; every bfloat16 product is exact in float32 and the sums are float32, in fewer
// rounding steps than the K = 4 float32 instruction makes.
// Six v_mfma_f32_32x32x16_bf16 take 192 cycles where the float32 products of the same block take
// 512 (v_mfma_f32_16x16x4_f32), and the split costs 5.5 vector instructions an element.
//
// Non-finite inputs, and finite ones above the largest bfloat16 (3.39e38), make a NaN of the
// split (inf - inf) where float32 gives infinity or a finite sum. The executor's products (executor.hip:
// merge, GEMM, W_O) test their sums and form those that are not finite again in float32, unless a NaN
// of their row made them. The bias producers do not: their input rows are clamped (split8_clamped), so
// finite edges up to the largest float give what float32 gives, but a weight or a hidden value that is
// not finite, or above the largest bfloat16, gives NaN where float32 may give an infinity.
// A value under about 1e-33 has a part below the smallest normal float, which the products drop: their
// relative error is 2.4e-7 down to 1e-32 (256 terms), 3.6e-7 at 1e-34, 2.7e-5 at 1e-36, where float32
// stays at 2.0e-7.
#pragma once

#include "mhsea_device.h"

namespace hz {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// v_mfma_f32_32x32x16_bf16, lane l = 32 hh + c: A[row c][k 8 hh + j], B[k 8 hh + j][col c],
// j = 0..7; C/D element i = 0..15 at [row 8 (i / 4) + 4 hh + i % 4][col c].
__device__ __forceinline__ v16f mfma32_bf16(bf16x8 a, bf16x8 b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// v_mfma_f32_32x32x2_f32, lane l = 32 hh + c: A[row c][k hh], B[k hh][col c]; C/D as above.
__device__ __forceinline__ v16f mfma32_f32(float a, float b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// v_mfma_f32_16x16x32_bf16, lane l = 16 g + c: A[row c][k 8 g + j], B[k 8 g + j][col c], j = 0..7;
// C/D as v_mfma_f32_16x16x4_f32.
__device__ __forceinline__ v4f mfma16_bf16(bf16x8 a, bf16x8 b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Eight floats as three operands of eight bfloat16 each.
struct Split8 {
  v4u h, m, l;
};

__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pack2_bf16(a, b);
  a -= __uint_as_float(h << 16);
  b -= __uint_as_float(h & 0xffff0000u);
  m = pack2_bf16(a, b);
  a -= __uint_as_float(m << 16);
  b -= __uint_as_float(m & 0xffff0000u);
  l = pack2_bf16(a, b);
}

__device__ __forceinline__ Split8 split8(const float (&x)[8]) {
  Split8 s;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t h, m, l;
    split2(x[2 * j], x[2 * j + 1], h, m, l);
    s.h[j] = h;
    s.m[j] = m;
    s.l[j] = l;
  }
  return s;
}

// The same for inputs that may lie above the largest bfloat16: finite values keep finite parts.
__device__ __forceinline__ Split8 split8_clamped(const float (&x)[8]) {
  constexpr float kMaxBf16 = 3.38953139e38f;
  Split8 s;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a = x[2 * j], b = x[2 * j + 1];
    const uint32_t h = pack2_bf16(__builtin_amdgcn_fmed3f(a, -kMaxBf16, kMaxBf16),
                                  __builtin_amdgcn_fmed3f(b, -kMaxBf16, kMaxBf16));
    a -= __uint_as_float(h << 16);
    b -= __uint_as_float(h & 0xffff0000u);
    const uint32_t m = pack2_bf16(a, b);
    a -= __uint_as_float(m << 16);
    b -= __uint_as_float(m & 0xffff0000u);
    s.h[j] = h;
    s.m[j] = m;
    s.l[j] = pack2_bf16(a, b);
  }
  return s;
}

__device__ __forceinline__ bf16x8 as_bf16x8(v4u u) { return __builtin_bit_cast(bf16x8, u); }

// The six terms, smallest first: parts of a and of b (0 = h, 1 = m, 2 = l) of term t.
constexpr int kSplitTerms = 6;
constexpr int kSplitA[kSplitTerms] = {2, 0, 1, 1, 0, 0};
constexpr int kSplitB[kSplitTerms] = {0, 2, 1, 0, 1, 0};

// acc[m][cb] += A_m B_cb for MB row blocks and two column blocks, one K step of 32. W: this step's
// A operands in LDS, [m][part][64 lanes], this lane's already added. Two row blocks at a time, so
// four sums take turns on the matrix cores.
template <int MB>
__device__ __forceinline__ void mm_step(const v4u* W, const Split8& b0, const Split8& b1, v4f (&acc)[MB][2]) {
  const bf16x8 b[2][3] = {{as_bf16x8(b0.h), as_bf16x8(b0.m), as_bf16x8(b0.l)},
                          {as_bf16x8(b1.h), as_bf16x8(b1.m), as_bf16x8(b1.l)}};
  constexpr int G = MB >= 2 ? 2 : 1;
#pragma unroll
  for (int m0 = 0; m0 < MB; m0 += G) {
    bf16x8 a[G][3];
#pragma unroll
    for (int i = 0; i < G && m0 + i < MB; ++i)
#pragma unroll
      for (int part = 0; part < 3; ++part) a[i][part] = as_bf16x8(W[((m0 + i) * 3 + part) * 64]);
#pragma unroll
    for (int t = 0; t < kSplitTerms; ++t)
#pragma unroll
      for (int i = 0; i < G && m0 + i < MB; ++i)
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
          acc[m0 + i][cb] = mfma16_bf16(a[i][kSplitA[t]], b[cb][kSplitB[t]], acc[m0 + i][cb]);
  }
}

__device__ __forceinline__ bool finite_f32(float x) {
  return (__float_as_uint(x) & 0x7f800000u) != 0x7f800000u;
}

}  // namespace hz
