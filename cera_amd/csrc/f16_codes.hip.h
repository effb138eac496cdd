// Block codes as f16, two at a time: a byte put into the mantissa of 1024 is the whole number 1024 + byte.
#pragma once
#include "common.hip.h"

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ h2v as_h2(uint32_t v) { return __builtin_bit_cast(h2v, v); }
__device__ __forceinline__ h2v fma2(h2v a, h2v b, h2v c) { return __builtin_elementwise_fma(a, b, c); }
__device__ __forceinline__ h2v both(float v) { return h2v{static_cast<_Float16>(v), static_cast<_Float16>(v)}; }
// bytes 0 and 2, or 1 and 3, of v as 1024 + byte
__device__ __forceinline__ h2v bytes02(uint32_t v) { return as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04020400u)); }
__device__ __forceinline__ h2v bytes13(uint32_t v) { return as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04030401u)); }
// byte j of v, twice, as 1024 + byte
template <int J> __device__ __forceinline__ h2v byte_twice(uint32_t v) { return as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04000400u | J | J << 16)); }
