// Activations and operand conversions shared by the projection kernels
// (sf_gemm.hip, sf_frag.hip).
#pragma once

#include <math.h>

#include "sf_device.h"

namespace sfk {

__device__ __forceinline__ float gelu_tanh(float x) {
    // GeluOp, src/backend/cuda/ops/elementwise.cuh:35-54: 0.5 x (1 + tanh u),
    // u = sqrt(2 / pi) (x + 0.044715 x^3), evaluated as x / (1 + e^(-2u))
    // (0.5 (1 + tanh u) = 1 / (1 + e^(-2u))): one hardware exp2 and one
    // reciprocal, ~1 ulp each; x -> -inf gives -0, x -> +inf gives x.
    const float kAlpha = 0.7978845608028654f;
    const float kBeta = 0.044715f;
    const float kM2Log2e = -2.f * 1.4426950408889634f;
    const float u = kAlpha * (x + kBeta * x * x * x);
    return x * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(kM2Log2e * u));
}

__device__ __forceinline__ float silu(float x) { return x / (1.f + expf(-x)); }

__device__ __forceinline__ float apply_act(int act, float v) {
    return act == 1 ? gelu_tanh(v) : (act == 2 ? silu(v) : v);
}

// Eight bf16 weights -> fp16x8 (round to nearest; exact in fp16's normal range).
__device__ __forceinline__ f16x8 bf16x8_to_f16x8(u32x4 w) {
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = pack_f16x2_rn(__uint_as_float(w[e] << 16), __uint_as_float(w[e] & 0xffff0000u));
    return u32x4_as_f16x8(o);
}

// Eight int8 codes -> fp16x8 (exact).  (Building 1024 + (code + 128) as an
// fp16 bit pattern with one byte permute per two codes and subtracting 1152
// in packed fp16 is exact too, but made the int8 batch-1 loop slower:
// 11.83 vs 11.75 ms.)
__device__ __forceinline__ f16x8 i8x8_to_f16x8(uint2 raw) {
    u32x4 o;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const uint32_t src = p < 2 ? raw.x : raw.y;
        const int sh = (p & 1) * 16;
        o[p] = pack_f16x2_rn((float)(int)(int8_t)(src >> sh), (float)(int)(int8_t)(src >> (sh + 8)));
    }
    return u32x4_as_f16x8(o);
}

// Eight int8 codes -> bf16x8 (exact: |code| <= 128 needs 8 significant bits).
__device__ __forceinline__ bf16x8 i8x8_to_bf16x8(uint2 raw) {
    uint32_t w[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const uint32_t src = p < 2 ? raw.x : raw.y;
        const int sh = (p & 1) * 16;
        const float lo = (float)(int)(int8_t)(src >> sh);
        const float hi = (float)(int)(int8_t)(src >> (sh + 8));
        w[p] = __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
    }
    return u32x4_as_bf16x8(u32x4{w[0], w[1], w[2], w[3]});
}

}  // namespace sfk
