// m2dcommon.h -- device helpers shared by the kernels of a residual block (m2dblock.hip, m2dtrain.hip): bf16 <-> fp32,
// 16-byte chunks of a row, weights of either type, the bf16 matrix product, GELU.
#ifndef M2D_COMMON_H
#define M2D_COMMON_H
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace {

struct bf16_t { uint16_t v; };

__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {   // one v_cvt_pk_bf16_f32 (round to nearest even)
  const f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// A chunk is 16 bytes of a row: kV elements.
template <typename T> struct Chunk;
template <> struct Chunk<float> {
  static constexpr int kV = 4;
  static __device__ __forceinline__ void load(const float* p, float (&v)[4]) {
    const float4 q = *reinterpret_cast<const float4*>(p);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
  }
  static __device__ __forceinline__ void store(float* p, const float (&v)[4]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  }
  static __device__ __forceinline__ void store_rounded(float* p, float (&v)[4]) { store(p, v); }
  static __device__ __forceinline__ void unpack(const uint4& q, float (&v)[4]) {
    v[0] = __uint_as_float(q.x); v[1] = __uint_as_float(q.y); v[2] = __uint_as_float(q.z); v[3] = __uint_as_float(q.w);
  }
};
template <> struct Chunk<bf16_t> {
  static constexpr int kV = 8;
  static __device__ __forceinline__ void load(const bf16_t* p, float (&v)[8]) {
    const uint4 q = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[2 * j] = bf_lo(w[j]); v[2 * j + 1] = bf_hi(w[j]); }
  }
  static __device__ __forceinline__ void store(bf16_t* p, const float (&v)[8]) {
    *reinterpret_cast<uint4*>(p) = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
  }
  static __device__ __forceinline__ void unpack(const uint4& q, float (&v)[8]) {
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[2 * j] = bf_lo(w[j]); v[2 * j + 1] = bf_hi(w[j]); }
  }
  // stores v and leaves in v what a reader of p will find
  static __device__ __forceinline__ void store_rounded(bf16_t* p, float (&v)[8]) {
    const uint32_t w[4] = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
    *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[2 * j] = bf_lo(w[j]); v[2 * j + 1] = bf_hi(w[j]); }
  }
};

__device__ __forceinline__ float ldw(const void* w, int wbf16, int i) {
  return wbf16 ? __uint_as_float((uint32_t)static_cast<const uint16_t*>(w)[i] << 16) : static_cast<const float*>(w)[i];
}
// V weights from index i0 on (a multiple of V, the array 16-byte aligned), in the fewest loads
template <int V>
__device__ __forceinline__ void ldwv(const void* w, int wbf16, int i0, float (&o)[V]) {
  if (wbf16) {
    if constexpr (V == 8) {
      Chunk<bf16_t>::load(static_cast<const bf16_t*>(w) + i0, o);
    } else {
      const uint2 q = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(w) + i0);
      o[0] = bf_lo(q.x); o[1] = bf_hi(q.x); o[2] = bf_lo(q.y); o[3] = bf_hi(q.y);
    }
  } else {
#pragma unroll
    for (int h = 0; h < V / 4; ++h) {
      const float4 q = *reinterpret_cast<const float4*>(static_cast<const float*>(w) + i0 + 4 * h);
      o[4 * h] = q.x; o[4 * h + 1] = q.y; o[4 * h + 2] = q.z; o[4 * h + 3] = q.w;
    }
  }
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4_t mfma_bf16(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ uint4 ld16(const void* p) { return *reinterpret_cast<const uint4*>(p); }

// max(v, 0) that hands a NaN on, as the stock operator does (fmaxf returns the other operand): one v_maximum3_f32
__device__ __forceinline__ float relu(float v) { return __builtin_elementwise_maximum(v, 0.f); }
// StarReLU, s relu(v)^2 + b
__device__ __forceinline__ float star_relu(float v, float s, float b) {
  const float t = relu(v);
  return __builtin_fmaf(s * t, t, b);
}
// d times the slope of StarReLU at t = relu(v): nothing where the activation is flat, whatever d is (0 x infinity would
// be a NaN there; the stock operator selects)
__device__ __forceinline__ float star_relu_back(float d, float t, float s) { return t <= 0.f ? 0.f : d * (2.f * s * t); }

// Phi(-|v|), the smaller part of the normal distribution, as exp2 of a polynomial in |v|: log2 Phi(-a) is smooth (close to
// a parabola), so the least-maximum fit of degree 10 over a <= 6, weighted to an even error of Phi, is off by 6e-9 there,
// and 5e-6 of Phi's own value up to a = 5; its leading coefficient is negative, so beyond it only falls (below 1e-9, and
// to 0 at infinity).  10 multiply-adds and one v_exp_f32 (half rate), 12 issue slots, and no
// subtraction of nearly equal values.  Over |v| <= 12 GELU is off by at most 3.8e-7 (rms 4.4e-8) and its slope by 1.2e-7 (2.3e-8);
// the stock kernels, through erf, by 4.5e-7 (5.0e-8) and 1.4e-7 (2.5e-8).
__device__ __forceinline__ float normal_tail(float v) {
  const float a = fabsf(v);
  float p = __builtin_fmaf(a, -2.4380350183150767e-08f, 7.511680450988933e-07f);
  p = __builtin_fmaf(a, p, -9.884181963570882e-06f);
  p = __builtin_fmaf(a, p, 7.055919559206814e-05f);
  p = __builtin_fmaf(a, p, -2.607103087939322e-04f);
  p = __builtin_fmaf(a, p, -3.67715438187588e-05f);
  p = __builtin_fmaf(a, p, 6.989158224314451e-03f);
  p = __builtin_fmaf(a, p, -5.246833711862564e-02f);
  p = __builtin_fmaf(a, p, -4.592123329639435e-01f);
  p = __builtin_fmaf(a, p, -1.1511051654815674f);
  p = __builtin_fmaf(a, p, -1.f);
  return __builtin_amdgcn_exp2f(p);
}
// GELU in its exact form, v Phi(v)
__device__ __forceinline__ float gelu_exact(float v) {
  const float q = normal_tail(v);
  return v * (v < 0.f ? q : 1.f - q);
}
// its slope, Phi(v) + v phi(v): 1 or 0, plus v phi(v) -+ Phi(-|v|), so that one rounding is near 1
__device__ __forceinline__ float gelu_slope(float v) {
  const float ex = __builtin_amdgcn_exp2f(v * v * -0.72134752044448170f);      // exp(-v^2 / 2)
  const float q = normal_tail(v);
  const float t = __builtin_fmaf(v * 0.39894228040143268f, ex, v < 0.f ? q : -q);
  return t + (v < 0.f ? 0.f : 1.f);
}

// both, each as above
__device__ __forceinline__ void gelu_and_slope(float v, float& value, float& slope) {
  const float ex = __builtin_amdgcn_exp2f(v * v * -0.72134752044448170f);
  const float q = normal_tail(v);
  const bool neg = v < 0.f;
  value = v * (neg ? q : 1.f - q);
  slope = __builtin_fmaf(v * 0.39894228040143268f, ex, neg ? q : -q) + (neg ? 0.f : 1.f);
}

inline bool misaligned(const void* p, size_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) != 0; }

}  // namespace
#endif
