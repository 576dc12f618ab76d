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

// A lane's 8 codes of a block as bf16 (small integers, exact).  Q4_0: raw is
// one dword, the result the raw nibbles c (0..15), low nibbles first; the -8
// of (c - 8) comes in through the block sums of x.  A nibble in a byte is the
// fp8 (E4M3) number c * 2^-9, denormal or not, so one scaled conversion makes
// two of them.
template <bool Q4>
__device__ __forceinline__ u32x4 codes_to_bf16(u32x2 raw) {
    u32x4 out;
    if constexpr (Q4) {
        const uint32_t lo = raw[0] & 0x0F0F0F0Fu, hi = (raw[0] >> 4) & 0x0F0F0F0Fu;
        out[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, false));
        out[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, true));
        out[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, false));
        out[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, true));
    } else {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (float)(int8_t)(raw[j >> 2] >> (8 * (j & 3)));
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = pack_hi16(v[2 * j], v[2 * j + 1]);
    }
    return out;
}

constexpr int SKINNY_MAX_GROUP = 8;

// The kernel that walks K (gemm_skinny_kwalk.hip): whether its LDS, which stages
// the block scales of whole rows, holds these weights', its time, and its launch.
bool skinny_kwalk_fits(int count, const mvlm_weight* const* ws, int num_cus);
double skinny_kwalk_us(int M, int count, const mvlm_weight* const* ws, int num_cus);
hipError_t launch_skinny_kwalk(hipStream_t s, int M, int count, const float* const* Xs, const mvlm_weight* const* ws,
                               float* const* Ys, int num_cus, const Epilogue* eps);

}  // namespace mvlm
