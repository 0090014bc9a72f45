// fp32 values as sums of three bf16 values, and their products on the bf16 matrix cores.
//
// 24 bits of significand are three times 8 (the splitting and its products: G. Henry, P. T. P. Tang, A. Heinecke, "Leveraging the
// bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", ARITH 2019).  The parts of x keep the exponent range of
// fp32 (a scale would have to be found first if they were fp16), and x0 y0 + (x0 y1 + x1 y0) + (x0 y2 + x1 y1 + x2 y0) misses x y by
// x1 y2 + x2 y1 + x2 y2: as |x1| <= 2^-8 |x| and |x2| <= 2^-17 |x|, at most about 2^-24 of it, one unit roundoff of fp32 (x = y just above one);
// 2^-27.5 in the root mean square of random values.
//
// The last bit of a bf16 denormal is 2^-133, so the third part of an x below 2^-110 would lose bits.  Operands are split times SPLIT_UP, which
// puts the last bit of any fp32 value there, denormals included (the matrix cores take bf16 denormals as they are), and what comes out is
// SPLIT_DOWN times their product.  Infinities, NaN, operands from 2^111.99 on and results from 2^96 on become infinities or NaN on the way and
// need a path of their own, see the users.
#pragma once
#include "ody_common.h"

constexpr float SPLIT_UP = 0x1p16f, SPLIT_DOWN = 0x1p-32f;

template <int N> struct FloatVec { typedef __attribute__((ext_vector_type(N))) float type; };
template <int N> struct Bf16Vec { typedef __attribute__((ext_vector_type(N))) __bf16 type; };

// x = p[0] + p[1] + p[2]: each part is what the parts before it left, rounded to 8 bits; the rests are exact in fp32, the last
// part as well.
template <int N>
struct Split3 {
  typedef typename FloatVec<N>::type vec;
  typedef typename Bf16Vec<N>::type part;
  part p[3];
  static __device__ __forceinline__ unsigned round2(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
  }
  // what round2 left of a (low half of w) and of b (high half)
  static __device__ __forceinline__ float rest_low(float a, unsigned w) { return a - __builtin_bit_cast(float, w << 16); }
  static __device__ __forceinline__ float rest_high(float b, unsigned w) { return b - __builtin_bit_cast(float, w & 0xffff0000u); }
  __device__ __forceinline__ explicit Split3(vec x) {
    typedef __attribute__((ext_vector_type(N / 2))) unsigned words;
    words w[3];
#pragma unroll
    for (int e = 0; e < N; e += 2) {
      float a = x[e], b = x[e + 1];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const unsigned t = round2(a, b);
        w[k][e / 2] = t;
        if (k < 2) a = rest_low(a, t), b = rest_high(b, t);
      }
    }
#pragma unroll
    for (int k = 0; k < 3; k++) p[k] = __builtin_bit_cast(part, w[k]);
  }
};

// hi += the largest product, lo += the five others
__device__ __forceinline__ void mfma_split3(const bf16x8 (&a)[3], const bf16x8 (&b)[3], f32x16& hi, f32x16& lo) {
  lo = mfma32(a[2], b[0], lo);
  hi = mfma32(a[0], b[0], hi);
  lo = mfma32(a[0], b[2], lo);
  lo = mfma32(a[1], b[1], lo);
  lo = mfma32(a[1], b[0], lo);
  lo = mfma32(a[0], b[1], lo);
}
