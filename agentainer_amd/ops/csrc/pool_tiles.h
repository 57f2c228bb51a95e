// What the paged attention kernels that multiply on MFMA share: vector types
// of operands and transposing LDS reads, and pool elements on the way to them.
#pragma once

#include "common.h"

namespace {

typedef __bf16 bf16v8 __attribute__((ext_vector_type(8)));
typedef float f32v8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// 8 pool elements as they are loaded (short: bf16 pools, unsigned char: e4m3)
template <typename CT>
struct Raw;
template <>
struct Raw<short> {
  typedef bf16x8 type;
};
template <>
struct Raw<unsigned char> {
  typedef u8x8 type;
};

// the same as bf16; every e4m3 value is a bf16 value
__device__ __forceinline__ bf16x8 to_bf16(const bf16x8 v) { return v; }
__device__ __forceinline__ bf16x8 to_bf16(const u8x8 v) {
  f32v8 f;
  float t[8];
  fp8x8_to_f32(v, t);
#pragma unroll
  for (int j = 0; j < 8; ++j) f[j] = t[j];
  union {
    bf16v8 b;
    bf16x8 s;
  } cv;
  cv.b = __builtin_convertvector(f, bf16v8);
  return cv.s;
}

}  // namespace
