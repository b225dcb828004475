// sx_special_device.h -- FP64 functions shared by the multipole sums.
#pragma once

#include "sx_internal.h"

namespace sx {

// Taylor coefficients of sin (x^17 .. x^3) and cos (x^16 .. x^4), read by scalar
// loads: as literals they would be kept in vector registers, which the sums need.
static __constant__ const double kTaylor[15] = {
    1.0 / 355687428096000.0, -1.0 / 1307674368000.0, 1.0 / 6227020800.0, -1.0 / 39916800.0, 1.0 / 362880.0,
    -1.0 / 5040.0,           1.0 / 120.0,            -1.0 / 6.0,         //
    1.0 / 20922789888000.0,  -1.0 / 87178291200.0,   1.0 / 479001600.0,  -1.0 / 3628800.0,   1.0 / 40320.0,
    -1.0 / 720.0,            1.0 / 24.0};

// Wave-uniform, read-only tables, read by scalar loads.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T *uniform(const T *p) {
    return (const __attribute__((address_space(4))) T *)p;
}

// sin and cos of 0 <= x <= kMultipoleMaxArg: two-term reduction by pi/2 with
// fused products (the second constant takes pi/2 to 2^-106), then the Taylor
// series on [-pi/4, pi/4], truncated below 1e-17.
__device__ __forceinline__ void sincos_reduced(double x, double &s, double &c) {
    int zo = 0;
    asm volatile("" : "+s"(zo));
    const auto C = uniform(kTaylor) + zo;
    const double k = rint(x * 0.63661977236758134308);
    double r = fma(-k, 1.57079632679489661923, x);
    r = fma(-k, 6.12323399573676603587e-17, r);
    const double z = r * r;
    double ps = C[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) ps = fma(ps, z, C[i]);
    const double sr = fma(ps * z, r, r);
    double pc = C[8];
#pragma unroll
    for (int i = 9; i < 15; ++i) pc = fma(pc, z, C[i]);
    const double cr = fma(pc * z, z, fma(-0.5, z, 1.0));
    const int q = (int)k;
    const bool swap = q & 1;
    s = swap ? cr : sr;
    c = swap ? sr : cr;
    if (q & 2) s = -s;
    if ((q + 1) & 2) c = -c;
}

// 1 / x from the hardware reciprocal by two Newton steps, x normal.
__device__ __forceinline__ double reciprocal(double x) {
    double i = __builtin_amdgcn_rcp(x);
    i = fma(fma(-x, i, 1.0), i, i);
    return fma(fma(-x, i, 1.0), i, i);
}

}  // namespace sx
