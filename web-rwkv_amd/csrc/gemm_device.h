// Device-side helpers shared by the matrix-core kernels (gemm.hip, gemm_short.hip).
#pragma once

#include "wrq_device.h"

namespace wrq {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));

union HalfPack {
    uint32_t u[4];
    half8 h;
};

__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
    return (uint32_t)f2h(a) | ((uint32_t)f2h(b) << 16);
}

__device__ __forceinline__ half2v as_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ uint32_t as_u32(half2v v) { return __builtin_bit_cast(uint32_t, v); }

__device__ __forceinline__ float dot2_ones(uint32_t v, float acc) {
    // acc + lo(v) + hi(v) with f32 accumulation: v_dot2_f32_f16 against (1.0, 1.0)
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, v), half2v{(_Float16)1.0f, (_Float16)1.0f}, acc, false);
}

__device__ __forceinline__ float row16_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xf, 0xf, true));
    return v;
}

} // namespace wrq
