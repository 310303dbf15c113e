// fl_common.h — element access and host helpers shared by the gfx950 kernel sources.
#ifndef FL_COMMON_H_
#define FL_COMMON_H_

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "fields_amd.h"

namespace fl {

constexpr float kLog2e = 1.4426950408889634f;

typedef unsigned short bf16_bits;
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

typedef __amdgpu_buffer_rsrc_t rsrc_t;
// raw buffer over `bytes` from base: loads past it give 0, stores past it are dropped
__device__ __forceinline__ rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// round to nearest even
__device__ __forceinline__ uint32_t bf16_bits_of(float x) {
  return (uint32_t)__builtin_bit_cast(unsigned short, (__bf16)x);
}
// two values rounded to nearest even and packed, lo in bits 15..0 (one v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
  const f32x2 f = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}
__device__ __forceinline__ float bf16_round(float x) { return __uint_as_float(bf16_bits_of(x) << 16); }

template <typename T>
__device__ __forceinline__ float round_as(float v);
template <>
__device__ __forceinline__ float round_as<float>(float v) { return v; }
template <>
__device__ __forceinline__ float round_as<bf16_bits>(float v) { return bf16_round(v); }

template <typename T>
__device__ __forceinline__ float load_as(const T* p);
template <>
__device__ __forceinline__ float load_as<float>(const float* p) { return *p; }
template <>
__device__ __forceinline__ float load_as<bf16_bits>(const bf16_bits* p) {
  return __uint_as_float((uint32_t)*p << 16);
}

__device__ __forceinline__ void store_as(float* p, float v) { *p = v; }
__device__ __forceinline__ void store_as(bf16_bits* p, float v) { *p = (bf16_bits)bf16_bits_of(v); }

// N consecutive elements as fp32 (N = 1 or 8), the vector form in 16-byte accesses
template <typename T, int N>
struct Vec;
template <typename T>
struct Vec<T, 1> {
  __device__ __forceinline__ static void load(const T* p, float* o) { o[0] = load_as<T>(p); }
  __device__ __forceinline__ static void store(T* p, const float* v) { store_as(p, v[0]); }
};
template <>
struct Vec<float, 8> {
  __device__ __forceinline__ static void load(const float* p, float* o) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) { o[i] = a[i]; o[4 + i] = b[i]; }
  }
  __device__ __forceinline__ static void store(float* p, const float* v) {
    f32x4 a, b;
#pragma unroll
    for (int i = 0; i < 4; ++i) { a[i] = v[i]; b[i] = v[4 + i]; }
    *reinterpret_cast<f32x4*>(p) = a;
    *reinterpret_cast<f32x4*>(p + 4) = b;
  }
};
template <>
struct Vec<bf16_bits, 8> {
  __device__ __forceinline__ static void load(const bf16_bits* p, float* o) {
    const u32x4 w = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) { o[2 * i] = bf16_lo(w[i]); o[2 * i + 1] = bf16_hi(w[i]); }
  }
  __device__ __forceinline__ static void store(bf16_bits* p, const float* v) {
    u32x4 w;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = bf16_pair(v[2 * i], v[2 * i + 1]);
    *reinterpret_cast<u32x4*>(p) = w;
  }
};

// Sum over the wave's 64 lanes, the same bits in every lane, as the butterfly of lane distances 1, 2,
// 4, 8, 16, 32 gives them (mirrors stand for distances 4 and 8: by then their lanes hold equal
// sums). All in vector registers: six LDS round trips of a shuffle butterfly are a serial chain.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float wave_sum(float v) {
  v = dpp_add<0xb1>(v);   // quad_perm [1, 0, 3, 2]
  v = dpp_add<0x4e>(v);   // quad_perm [2, 3, 0, 1]
  v = dpp_add<0x141>(v);  // row_half_mirror
  v = dpp_add<0x140>(v);  // row_mirror
  const u32x2 a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a.x) + __uint_as_float(a.y);
  const u32x2 b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b.x) + __uint_as_float(b.y);
}

// 1 / (1 + e), subnormal results included: v_rcp_f32 gives 0 for those, so it takes a quarter of the
// divisor, and the scale back is exact up to the subnormal's own rounding.
__device__ __forceinline__ float rcp_one_plus(float e) {
  return __builtin_amdgcn_rcpf(fmaf(e, 0.25f, 0.25f)) * 0.25f;
}

// 1 / (1 + e^-x) of a bf16 x: one v_exp_f32 and one v_rcp_f32, whose bf16 rounding is the library form's for
// all 65,536 inputs.
__device__ __forceinline__ float sigmoid_bf16(float x) {
  return rcp_one_plus(__builtin_amdgcn_exp2f(x * -kLog2e));
}

// x / (1 + e^-x) to about an ulp: v_exp_f32 of the rounded product x log2(e) with the product's
// rounding error put back (first order), and one residual step on the reciprocal's quotient. The
// exponent is held within the first float whose rounded product reaches 128 (its error is positive, so that
// the corrected power is inf, not NaN): below, the quotient is -0, and NaN for -inf. Where the residual
// is 0 or NaN the plain quotient stands. For every bf16 x the result rounds to the stock op's bf16 value;
// without SUBNORMAL (two operations less) it is -0 from -87.3 down, where the stock value is under 1.1e-36.
template <bool SUBNORMAL = true>
__device__ __forceinline__ float silu_precise(float x) {
  constexpr float kL = -kLog2e, kLlo = -1.9259629911266175e-8f;  // -log2(e) = kL + kLlo
  constexpr float kLimit = 88.72283935546875f;
  const float xc = __builtin_amdgcn_fmed3f(x, -kLimit, kLimit);
  const float hi = xc * kL;
  const float lo = fmaf(xc, kLlo, fmaf(xc, kL, -hi));
  const float e0 = __builtin_amdgcn_exp2f(hi);
  const float corr = fmaf(e0, lo * 0.6931471805599453f, e0);
  const float d = 1.0f + corr, r = SUBNORMAL ? rcp_one_plus(corr) : __builtin_amdgcn_rcpf(d), q = x * r;
  const float res = fmaf(-q, d, x);
  return __builtin_fabsf(res) > 0.0f ? fmaf(res, r, q) : q;
}

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
inline int hip_status(hipError_t e) { return e == hipSuccess ? FL_OK : FL_ERR_HIP_BASE + (int)e; }
inline bool dtype_ok(int d) { return d == FL_DTYPE_F32 || d == FL_DTYPE_BF16; }
inline size_t esize(int d) { return d == FL_DTYPE_BF16 ? 2 : 4; }

}  // namespace fl

#endif  // FL_COMMON_H_
