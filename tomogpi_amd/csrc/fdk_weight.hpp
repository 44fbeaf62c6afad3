// The FDK distance weight num / sqrt(q), bit for bit the quotient of the two
// correctly rounded FP32 operations, without their general sequences (scaling,
// special values), which are most of a voxel update's instructions.
#pragma once

#include <hip/hip_runtime.h>

namespace tomo {

// num and q within these bounds: no step below under- or overflows.
constexpr float kFdkLeast = 0x1p-40f, kFdkMost = 0x1p60f;

// y: 1 / sqrt(q) from the hardware, to an ulp.  s: a Newton step and the
// residual step s + (q - s^2) / 2s, by fma.  r: two Newton steps on 1 / s, from
// a start an ulp high (from below, the step for the largest mantissa ends on a
// tie).  Then one residual step on num r (Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990).  Checked over all
// values: s and r are the correctly rounded root and reciprocal for each of the
// 8.4e8 q in the bounds, and the quotient for each of the 2^46 pairs of
// mantissas.  About 11 cycles per wave and CU, the general forms about 26.
__device__ __forceinline__ float fdk_weight(float num, float q) {
    const float y = __builtin_amdgcn_rsqf(q), h = 0.5f * y;
    float s = q * y;
    s = fmaf(s, fmaf(-s, h, 0.5f), s);
    s = fmaf(fmaf(-s, s, q), h, s);
    float r = y * 0x1.000002p+0f;
    r = fmaf(fmaf(-s, r, 1.0f), r, r);
    r = fmaf(fmaf(-s, r, 1.0f), r, r);
    const float t = num * r;
    return fmaf(fmaf(-s, t, num), r, t);
}

}  // namespace tomo
