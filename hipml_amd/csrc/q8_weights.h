// Q8_0 weight matrices: what the projection kernels (proj.hip, gemm.hip) share.
#pragma once

#include "common.h"

namespace hipml {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint2a4 __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t uint3a4 __attribute__((ext_vector_type(3), aligned(4)));

constexpr int kQ8Block = 34;

// 8 int8 (two dwords) -> 8 f16 holding the same integers, exactly.
__device__ __forceinline__ half8 int8x8_to_f16(uint32_t w0, uint32_t w1)
{
    const uint32_t x0 = w0 ^ 0x80808080u, x1 = w1 ^ 0x80808080u;
    const uint32_t hi = 0x64646464u;
    uint4v r;
    r[0] = __builtin_amdgcn_perm(hi, x0, 0x04010400u);
    r[1] = __builtin_amdgcn_perm(hi, x0, 0x04030402u);
    r[2] = __builtin_amdgcn_perm(hi, x1, 0x04010400u);
    r[3] = __builtin_amdgcn_perm(hi, x1, 0x04030402u);
    half8 h = __builtin_bit_cast(half8, r);
    const half8 off = {1152, 1152, 1152, 1152, 1152, 1152, 1152, 1152};
    return h - off;
}

} // namespace hipml
