// fp32 hyperbolic tangent for kernels whose inner loop is bound by it.
#pragma once

#include <cmath>

#ifdef __HIPCC__
#define SANA_SOFT __host__ __device__ inline
#else
#define SANA_SOFT inline
#endif

namespace sana {

// tanh for |x| < 1 (NaN for NaN, +0 for -0): x + x^3 P(x^2), P the polynomial of degree 6 of
// least maximal relative error there (4.7e-9, by Remez exchange).
SANA_SOFT float soft_tanh_below_1(float x) {
    const float t = x * x;
    float p = -0.000358452002f;
    p = std::fma(p, t, 0.00230136467f);
    p = std::fma(p, t, -0.00794610661f);
    p = std::fma(p, t, 0.0214866567f);
    p = std::fma(p, t, -0.0538798012f);
    p = std::fma(p, t, 0.133323446f);
    p = std::fma(p, t, -0.333332956f);
    return std::fma(x * t, p, x);
}

// tanh without branches: from |x| = 1 on 1 - 2 / (c + 1) with c = e^2|x| as 2^h (1 + l ln 2),
// h = 2|x| log2(e) rounded and l what the rounding left (log2(e) in two floats), r
// what c + 1 lost, and one Newton step on the reciprocal.
// Largest error on MI355X over all x, in ulp: 1.04 (tanhf 1.41).
SANA_SOFT float soft_tanh(float x) {
    const float a = std::fabs(x), b = a < 16.0f ? 2.0f * a : 32.0f;  // (1 when rounded, from 9.02 on)
    const float h = b * 1.44269502f, l = std::fma(b, 1.92596303e-8f, std::fma(b, 1.44269502f, -h));
#ifdef __HIP_DEVICE_COMPILE__
    const float e = __builtin_amdgcn_exp2f(h);
#else
    const float e = std::exp2(h);
#endif
    const float c = std::fma(e, l * 0.693147182f, e), d = c + 1.0f, r = 1.0f - (d - c);
#ifdef __HIP_DEVICE_COMPILE__
    float q = __builtin_amdgcn_rcpf(d);
#else
    float q = 1.0f / d;
#endif
    q = std::fma(std::fma(-r, q, std::fma(-d, q, 1.0f)), q, q);
    const float big = std::fma(-2.0f, q, 1.0f);
    return a < 1.0f ? soft_tanh_below_1(x) : std::copysign(x == x ? big : x, x);
}

}  // namespace sana
