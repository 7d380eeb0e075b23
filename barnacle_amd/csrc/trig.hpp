// trig.hpp -- sine and cosine of a float as the float rounding of the
// double-precision result (MathF.Sin / MathF.Cos on the CPU renderer's side),
// for host and device.
#pragma once
#include <math.h>

#ifndef __host__
#define __host__
#define __device__
#endif

namespace bnd {

// Both at once for |x| < 2^20: x less its nearest multiple of pi/2 as a double
// and the rest of it (Cody and Waite's reduction with a 106-bit pi/2), and the
// Taylor series of both functions on [-pi/4, pi/4], whose remainders lie below
// 2^-61.  Every float in [-2 pi, 2 pi] gives the floats that a correctly
// rounded double result would.  The library's double-precision functions take
// any argument, one function at a time: four of them made up half of the
// instructions that shading a glossy vertex executes.
__host__ __device__ inline void sincos_f(float xf, float& s, float& c) {
    const double x = (double)xf;
    const double k = rint(x * 0x1.45f306dc9c883p-1);                 // 2 / pi
    const double h = fma(-k, 0x1.921fb54442d18p+0, x);
    const double l = k * 0x1.1a62633145c07p-54;
    const double r = h - l;
    const double e = (h - r) - l;
    const double z = r * r;
    double p = 0x1.952c77030ad4ap-49;                                // 1 / 17!
    p = fma(p, z, -0x1.ae7f3e733b81fp-41);
    p = fma(p, z, 0x1.6124613a86d09p-33);
    p = fma(p, z, -0x1.ae64567f544e4p-26);
    p = fma(p, z, 0x1.71de3a556c734p-19);
    p = fma(p, z, -0x1.a01a01a01a01ap-13);
    p = fma(p, z, 0x1.1111111111111p-7);
    p = fma(p, z, -0x1.5555555555555p-3);
    const double sn = r + fma(r * z, p, e * fma(-0.5, z, 1.0));
    double q = 0x1.ae7f3e733b81fp-45;                                // 1 / 16!
    q = fma(q, z, -0x1.93974a8c07c9dp-37);
    q = fma(q, z, 0x1.1eed8eff8d898p-29);
    q = fma(q, z, -0x1.27e4fb7789f5cp-22);
    q = fma(q, z, 0x1.a01a01a01a01ap-16);
    q = fma(q, z, -0x1.6c16c16c16c17p-10);
    q = fma(q, z, 0x1.5555555555555p-5);
    const double w = fma(-0.5, z, 1.0);
    const double cs = w + (fma(-0.5, z, 1.0 - w) + fma(z * z, q, -r * e));
    const int n = (int)k;
    const float fs = (float)sn, fc = (float)cs;
    s = n & 1 ? fc : fs;
    c = n & 1 ? fs : fc;
    s = n & 2 ? -s : s;
    s = xf == 0.0f ? xf : s;                                         // -0 is its own sine
    c = (n + 1) & 2 ? -c : c;
}

}  // namespace bnd
