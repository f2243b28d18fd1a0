// What the sources of libhstu_block.so share: bf16 conversions, wave sums, the error text.

#ifndef HSTU_BLOCK_COMMON_H_
#define HSTU_BLOCK_COMMON_H_

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include "hstu_block.h"

// Stores the message that hstu_block_last_error() returns on this thread; returns `code`.
__attribute__((visibility("hidden"))) int block_fail(int code, const char* fmt, ...);
__attribute__((visibility("hidden"))) void block_clear_error();
// Raises the dynamic-LDS limit of a kernel, once per device (`granted`: 64 entries of the caller).
__attribute__((visibility("hidden"))) int block_allow_lds(const void* fn, int bytes, int* granted);

namespace {

// The arguments as this version has them: a struct of versions 3 or 4 (of the given sizes: prefixes of today's) with zeros in
// what it does not have, any other as it is.
template <typename A>
const A* block_today(const A* a, A& own, size_t v3, size_t v4) {
  if (!a || !((a->version == 3 && a->struct_size == v3) || (a->version == 4 && a->struct_size == v4))) return a;
  memset(&own, 0, sizeof(own));
  memcpy(&own, a, a->struct_size);
  own.struct_size = sizeof(own);
  own.version = HSTU_BLOCK_ABI_VERSION;
  return &own;
}

typedef __bf16 bf16_t;
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

inline bool block_aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

__device__ __forceinline__ void unpack8(const uint4& v, float (&f)[8]) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __builtin_bit_cast(float, w[i] << 16);
    f[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xffff0000u);
  }
}

__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  floatx2 f = {lo, hi};
  bf16x2 r = __builtin_convertvector(f, bf16x2);
  return __builtin_bit_cast(uint32_t, r);
}

__device__ __forceinline__ uint4 pack8(const float (&y)[8]) {
  return uint4{pack2(y[0], y[1]), pack2(y[2], y[3]), pack2(y[4], y[5]), pack2(y[6], y[7])};
}

__device__ __forceinline__ float round_bf16(float x) { return (float)(bf16_t)x; }

// x sigmoid(x) by the hardware's exp2 and reciprocal (1 ulp each)
__device__ __forceinline__ float silu(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x));
}

// d silu / dx
__device__ __forceinline__ float silu_grad(float x) {
  const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x));
  return sg * __builtin_fmaf(x, 1.0f - sg, 1.0f);
}

// the sum over aligned groups of N lanes
template <int N>
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
  for (int d = N / 2; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

}  // namespace

#endif  // HSTU_BLOCK_COMMON_H_
