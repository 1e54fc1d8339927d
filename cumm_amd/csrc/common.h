// Shared device/host helpers for the gfx950 kernels of libcummhip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace cummhip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;

// element tags ---------------------------------------------------------------
struct F16 {};
struct BF16 {};
struct S8 {};

template <class T> struct Elem;
template <> struct Elem<F16> {
  using Acc = float;
  using AccV = v4f;
  static constexpr int kBytes = 2;
  static constexpr int kPerVec = 8;   // elements in one 16-byte fragment
  static constexpr int kMfmaK = 32;   // contraction length of one 16x16 MFMA
  static __device__ __forceinline__ v4f mfma(v4i a, v4i b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a),
                                                  __builtin_bit_cast(v8h, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ float to_float(uint16_t bits) {
    return (float)__builtin_bit_cast(_Float16, bits);
  }
  static __device__ __forceinline__ uint16_t from_float(float x) {
    return __builtin_bit_cast(uint16_t, (_Float16)x);  // v_cvt_f16_f32: round to nearest even
  }
  // two of them, the first in the low half (v_cvt_pk_f16_f32: the same bits)
  static __device__ __forceinline__ uint32_t from_floats(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{a, b}, v2h));
  }
};
template <> struct Elem<BF16> {
  using Acc = float;
  using AccV = v4f;
  static constexpr int kBytes = 2;
  static constexpr int kPerVec = 8;
  static constexpr int kMfmaK = 32;
  static __device__ __forceinline__ v4f mfma(v4i a, v4i b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a),
                                                   __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ float to_float(uint16_t bits) {
    return __builtin_bit_cast(float, (uint32_t)bits << 16);
  }
  // round to nearest even on bit 16, NaN -> 0x7FFF
  // (bfloat16_t(float), include/tensorview/gemm/dtypes/bfloat16.h:86-111 of the reference): the hardware's
  // conversion, which gives these bits for everything but NaN, denormals among it (all 2^32 compared)
  static __device__ __forceinline__ uint16_t from_float(float x) {
    const uint16_t h = (uint16_t)from_floats(x, x);
    return x != x ? (uint16_t)0x7FFF : h;
  }
  // two of them, the first in the low half; NaN becomes some NaN
  static __device__ __forceinline__ uint32_t from_floats(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{a, b}, v2bf));
  }
};
template <> struct Elem<S8> {
  using Acc = int;
  using AccV = v4i;
  static constexpr int kBytes = 1;
  static constexpr int kPerVec = 16;
  static constexpr int kMfmaK = 64;
  static __device__ __forceinline__ v4i mfma(v4i a, v4i b, v4i c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
  }
};

// Eight results rounded and packed, as from_float rounds each: half an instruction per element, and for bf16
// another half that looks for NaN.  NUMBERS: there is none among them.  ONE_BY_ONE: f16 sums straight from
// an fma, whose conversion the compiler can take into the fma; as pairs a few elements round the other way (3e-6 of
// the result; 200 k rows, 64 -> 128 channels with a source take 23.6 us either way).
template <class T, bool NUMBERS, bool ONE_BY_ONE = false>
__device__ __forceinline__ v4i round8(const float (&t)[8]) {
  v4i v;
  if constexpr (ONE_BY_ONE) {
    uint16_t *h = reinterpret_cast<uint16_t *>(&v);
#pragma unroll
    for (int x = 0; x < 8; ++x) h[x] = Elem<T>::from_float(t[x]);
    return v;
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) v[x] = (int)Elem<T>::from_floats(t[2 * x], t[2 * x + 1]);
  if constexpr (std::is_same_v<T, BF16> && !NUMBERS) {
    bool nan = false;
#pragma unroll
    for (int x = 0; x < 4; ++x) nan |= __builtin_isunordered(t[2 * x], t[2 * x + 1]);
    if (__builtin_expect(nan, 0)) {
#pragma unroll
      for (int x = 0; x < 4; ++x) v[x] = (int)((uint32_t)Elem<T>::from_float(t[2 * x]) | (uint32_t)Elem<T>::from_float(t[2 * x + 1]) << 16);
    }
  }
  return v;
}

// One bit per result of a ReLU, +0 or positive: which of eight packed two-byte results are not zero.  (The minimum
// is an asm statement because the compiler, which knows where the halves come from, makes a test for classes of
// floating-point numbers out of it: 300 instructions for 9.)
__device__ __forceinline__ uint32_t positive8(const v4i &v) {
  uint32_t bits = 0;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int two = v[x];
    uint32_t one;
    asm("v_pk_min_u16 %0, %1, %2" : "=v"(one) : "v"(two), "s"(0x00010001u));
    bits |= one << (2 * x);
  }
  return (bits | bits >> 15) & 0xFFu;      // (low halves in bits 0, 2, 4, 6, high ones in 16, 18, ...)
}

// activations: UnaryActivation, cumm/gemm/gemmmath/__init__.py:181-214 of the reference
__device__ __forceinline__ float apply_act(float x, int act, float act_alpha) {
  switch (act) {
  case 1: return x > 0.0f ? x : 0.0f;
  case 2: return 1.0f / (1.0f + expf(-x));
  case 3: return x >= 0.0f ? x : x * act_alpha;
  default: return x;
  }
}

// float -> s8: clamp to [-128,127] then round half to even; NaN -> 0
// (Int8Inference clamp + cvt.rni.sat.s8.f32, cumm/gemm/output_op/linear.py:327-351,
//  include/tensorview/gemm/math/numeric_convert.h:171-192 of the reference)
// Three instructions: round half to even, convert (the hardware conversion saturates and turns
// NaN into 0; written as asm because the C cast is undefined out of range), clamp the integer.
// Clamping after the rounding equals clamping before it: the bounds are integers.
__device__ __forceinline__ int f32_to_s8(float t) {
  const float q = __builtin_rintf(t);
  int i;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(q));
  i = i > 127 ? 127 : i;
  return i < -128 ? -128 : i;
}

// low bytes of four integers as one dword (three v_perm_b32)
__device__ __forceinline__ int pack4_bytes(int b0, int b1, int b2, int b3) {
  const uint32_t lo = __builtin_amdgcn_perm((uint32_t)b1, (uint32_t)b0, 0x0c0c0400u);
  const uint32_t hi = __builtin_amdgcn_perm((uint32_t)b3, (uint32_t)b2, 0x0c0c0400u);
  return (int)__builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v |= (uint32_t)__shfl_xor((int)v, off, 64);
  return v;
}

}  // namespace cummhip
