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
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

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

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) v += __shfl_xor(v, m);
  return v;
}

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
inline int hip_status(hipError_t e) { return e == hipSuccess ? FL_OK : FL_ERR_HIP_BASE + (int)e; }
inline bool dtype_ok(int d) { return d == FL_DTYPE_F32 || d == FL_DTYPE_BF16; }
inline size_t esize(int d) { return d == FL_DTYPE_BF16 ? 2 : 4; }

}  // namespace fl

#endif  // FL_COMMON_H_
