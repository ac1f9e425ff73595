// Element access shared by the mixer kernels: activations and caches are bf16 (serving) or fp32, arithmetic is fp32.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lanes.h"

namespace elem {

typedef unsigned short bf16raw;

__device__ inline float bf2f(bf16raw v) { return __uint_as_float((unsigned int)v << 16); }
__device__ inline bf16raw f2bf(float f) { return __builtin_bit_cast(bf16raw, (__bf16)f); }  // round to nearest even (hardware conversion)

template <typename T> __device__ inline float ld(const T* p);
template <> __device__ inline float ld<float>(const float* p) { return *p; }
template <> __device__ inline float ld<bf16raw>(const bf16raw* p) { return bf2f(*p); }
template <typename T> __device__ inline void st(T* p, float v);
template <> __device__ inline void st<float>(float* p, float v) { *p = v; }
template <> __device__ inline void st<bf16raw>(bf16raw* p, float v) { *p = f2bf(v); }

// an element's bits as they are loaded, and its value: what is loaded long before it is used is not waited for by its conversion
__device__ inline unsigned int raw(const float* p) { return __float_as_uint(*p); }
__device__ inline unsigned int raw(const bf16raw* p) { return *p; }
template <typename T> __device__ inline float number(unsigned int v) { return __uint_as_float(sizeof(T) == 2 ? v << 16 : v); }

// four consecutive elements (aligned to four)
__device__ inline float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ inline float4 ld4(const bf16raw* p) {
  const ushort4 v = *reinterpret_cast<const ushort4*>(p);
  return make_float4(bf2f(v.x), bf2f(v.y), bf2f(v.z), bf2f(v.w));
}
__device__ inline void st4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
__device__ inline void st4(bf16raw* p, float4 v) {
  ushort4 o;
  o.x = f2bf(v.x); o.y = f2bf(v.y); o.z = f2bf(v.z); o.w = f2bf(v.w);
  *reinterpret_cast<ushort4*>(p) = o;
}

__device__ inline float wave_sum(float v) { return lanes::sum(v); }
__device__ inline float wave_max(float v) { return lanes::max(v); }

// On the hardware's exponential, logarithm and reciprocal (about one unit in the last place each).
__device__ inline float fast_exp(float x) { return __builtin_amdgcn_exp2f(1.4426950408889634f * x); }
__device__ inline float sigmoid(float x) { return __builtin_amdgcn_rcpf(1.f + fast_exp(-x)); }
__device__ inline float silu(float x) { return x * sigmoid(x); }
// max(x, 0) + log(1 + e^-|x|); where e is small the logarithm is its series (1 + e would lose it)
__device__ inline float softplus(float x) {
  const float e = fast_exp(-fabsf(x));
  const float series = e * (1.f - e * (0.5f - e * (0.33333333f - e * 0.25f)));
  return fmaxf(x, 0.f) + (e < 0.02f ? series : 0.69314718f * __builtin_amdgcn_logf(1.f + e));
}

}  // namespace elem
