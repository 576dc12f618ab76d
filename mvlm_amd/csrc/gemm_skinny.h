// What the two kernels of the skinny GEMM share (gemm_skinny.hip has the
// arithmetic's account and the choice between them).
#pragma once

#include "common.h"
#include "device_math.h"

namespace mvlm {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8v;

// top 16 bits of two floats -> one packed bf16 pair (truncation)
__device__ __forceinline__ uint32_t pack_hi16(float lo_elem, float hi_elem) {
    return __builtin_amdgcn_perm(__float_as_uint(hi_elem), __float_as_uint(lo_elem), 0x07060302u);
}

// x[0..7] -> three bf16x8 parts with x = p1 + p2 + p3 (+ |residual| < 2^-24 |x|)
__device__ __forceinline__ void split3(const float (&x)[8], u32x4& p1, u32x4& p2, u32x4& p3) {
    float r1[8], r2[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float a = __uint_as_float(__float_as_uint(x[j]) & 0xFFFF0000u);
        r1[j] = x[j] - a;                                   // exact
        const float b = __uint_as_float(__float_as_uint(r1[j]) & 0xFFFF0000u);
        r2[j] = r1[j] - b;                                  // exact
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        p1[j] = pack_hi16(x[2 * j], x[2 * j + 1]);
        p2[j] = pack_hi16(r1[2 * j], r1[2 * j + 1]);
        p3[j] = pack_hi16(r2[2 * j], r2[2 * j + 1]);
    }
}

__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v, a), __builtin_bit_cast(bf16x8v, b), c,
                                                   0, 0, 0);
}

constexpr int SKINNY_MAX_GROUP = 8;

// The kernel that walks K (gemm_skinny_kwalk.hip): whether its LDS, which stages
// the block scales of whole rows, holds these weights', its time, and its launch.
bool skinny_kwalk_fits(int count, const mvlm_weight* const* ws, int num_cus);
double skinny_kwalk_us(int M, int count, const mvlm_weight* const* ws, int num_cus);
hipError_t launch_skinny_kwalk(hipStream_t s, int M, int count, const float* const* Xs, const mvlm_weight* const* ws,
                               float* const* Ys, int num_cus, const Epilogue* eps);

}  // namespace mvlm
