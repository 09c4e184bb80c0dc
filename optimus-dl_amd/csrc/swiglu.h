// SwiGLU and its gradients on packed pairs of bf16: the arithmetic of odl_fp8_swiglu_* to the last bit, for the kernels that
// write its result as bf16 (fused.hip) and for those that quantise it on the spot (quant.hip, mx.hip).
#pragma once

#include "common.h"

#pragma clang fp contract(off)

namespace odl {

// 1 / d for 1 <= d < 2^120: integer first guess, three Newton steps in fused multiply-adds.
__device__ __forceinline__ float recip_newton(float d) {
    float y = bits_to_float(0x7EF311C7u - float_to_bits(d));
    y = __fmaf_rn(y, __fmaf_rn(-d, y, 1.0f), y);
    y = __fmaf_rn(y, __fmaf_rn(-d, y, 1.0f), y);
    y = __fmaf_rn(y, __fmaf_rn(-d, y, 1.0f), y);
    return y;
}

// logistic function 1 / (1 + exp(-g)): range reduction by ln 2 in two pieces, degree-5 polynomial
// for (exp(r) - 1 - r) / r^2, exact scaling by 2^k, reciprocal as above.  A NaN argument is
// evaluated as 0 here (every use below multiplies by the argument again, which restores the NaN).
// The polynomial and the two pieces of ln 2 are those of the single-precision exp of the Cephes Mathematical Library
// (S. L. Moshier, expf.c); the reciprocal's first guess is the exponent negated in the integer domain.
__device__ __forceinline__ float sigmoid_det(float g) {
    float t = (g != g) ? 0.0f : -g;
    const bool zero = t > 80.0f;                 // exp(-g) beyond 2^115: the quotient is taken as 0
    t = __builtin_amdgcn_fmed3f(t, -80.0f, 80.0f);
    const float kf = __builtin_rintf(__fmul_rn(t, 1.44269504f));
    float r = __fmaf_rn(kf, -0.693359375f, t);
    r = __fmaf_rn(kf, 2.12194440e-4f, r);
    float p = 1.9875691500e-4f;
    p = __fmaf_rn(p, r, 1.3981999507e-3f);
    p = __fmaf_rn(p, r, 8.3334519073e-3f);
    p = __fmaf_rn(p, r, 4.1665795894e-2f);
    p = __fmaf_rn(p, r, 1.6666665459e-1f);
    p = __fmaf_rn(p, r, 5.0000001201e-1f);
    const float z = __fmul_rn(r, r);
    const float y = __fadd_rn(__fmaf_rn(p, z, r), 1.0f);
    const float e = __fmul_rn(y, bits_to_float((uint32_t)((int)kf + 127) << 23));
    const float s = recip_newton(__fadd_rn(1.0f, e));
    return zero ? 0.0f : s;
}

// Roundings to bf16 use the hardware's round-to-nearest-even conversion of a pair (subnormal
// results are kept: the kernels run with fp32 denormals enabled).

// h = bf16( bf16(g * sigmoid(g)) * u ), the two roundings of silu(gate) * up evaluated in bf16, for
// the two elements of a packed pair
__device__ __forceinline__ uint32_t swiglu_fwd_pair(uint32_t gw, uint32_t uw) {
    const float g0 = bf16_lo(gw), g1 = bf16_hi(gw);
    const uint32_t s = pack_bf16x2(__fmul_rn(g0, sigmoid_det(g0)), __fmul_rn(g1, sigmoid_det(g1)));
    return pack_bf16x2(__fmul_rn(bf16_lo(s), bf16_lo(uw)), __fmul_rn(bf16_hi(s), bf16_hi(uw)));
}

// d_up = bf16(dh * s), d_gate = bf16( bf16(dh * u) * (sig * (1 + g * (1 - sig))) ), s = bf16(g * sig)
__device__ __forceinline__ void swiglu_bwd_pair(uint32_t dw, uint32_t gw, uint32_t uw, uint32_t &dg, uint32_t &du) {
    const float g0 = bf16_lo(gw), g1 = bf16_hi(gw), d0 = bf16_lo(dw), d1 = bf16_hi(dw);
    const float sig0 = sigmoid_det(g0), sig1 = sigmoid_det(g1);
    const uint32_t s = pack_bf16x2(__fmul_rn(g0, sig0), __fmul_rn(g1, sig1));
    du = pack_bf16x2(__fmul_rn(d0, bf16_lo(s)), __fmul_rn(d1, bf16_hi(s)));
    const uint32_t ds = pack_bf16x2(__fmul_rn(d0, bf16_lo(uw)), __fmul_rn(d1, bf16_hi(uw)));
    const float ds0 = __fmul_rn(sig0, __fmaf_rn(g0, __fsub_rn(1.0f, sig0), 1.0f));
    const float ds1 = __fmul_rn(sig1, __fmaf_rn(g1, __fsub_rn(1.0f, sig1), 1.0f));
    dg = pack_bf16x2(__fmul_rn(bf16_lo(ds), ds0), __fmul_rn(bf16_hi(ds), ds1));
}

// Four pairs of h, or of d_gate and d_up, from 16 bytes of each operand.
__device__ __forceinline__ u32x4 swiglu_fwd8(const u32x4 g, const u32x4 u) {
    return u32x4{swiglu_fwd_pair(g.x, u.x), swiglu_fwd_pair(g.y, u.y), swiglu_fwd_pair(g.z, u.z), swiglu_fwd_pair(g.w, u.w)};
}

__device__ __forceinline__ void swiglu_bwd8(const u32x4 d, const u32x4 g, const u32x4 u, u32x4 &dg, u32x4 &du) {
    uint32_t a[4], b[4];
    swiglu_bwd_pair(d.x, g.x, u.x, a[0], b[0]);
    swiglu_bwd_pair(d.y, g.y, u.y, a[1], b[1]);
    swiglu_bwd_pair(d.z, g.z, u.z, a[2], b[2]);
    swiglu_bwd_pair(d.w, g.w, u.w, a[3], b[3]);
    dg = u32x4{a[0], a[1], a[2], a[3]};
    du = u32x4{b[0], b[1], b[2], b[3]};
}

}  // namespace odl
