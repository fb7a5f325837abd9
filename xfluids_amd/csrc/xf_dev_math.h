// Device-side FP64 exp / log with a fixed IEEE-754 operation sequence.
//
// The plain-FP64 form must reproduce the CPU restatement of XFluids bit for
// bit, including the chemistry step-size decisions that amplify one-ulp
// differences.  Vendor math libraries differ between host and device, so both
// sides use the same published methods:
//   exp: Cody & Waite reduction x = k ln2 + r with fused multiply-adds (ln2
//        split into the nearest double and a tail), Taylor series of exp(r) to
//        degree 13 by fused Horner steps, scaling by 2^k through the exponent
//        field in two factors.
//   log: x = m 2^e, m in [sqrt(1/2), sqrt(2)), f = m - 1 (exact),
//        s = f/(2+f), log(1+f) = f - s (f - R), R = sum_{k=1..11} 2 s^{2k}/(2k+1).
// Accuracy: within 2 ulp of a correctly rounded result over the ranges used.
// All files including this header are compiled with -ffp-contract=off; the
// fused multiply-adds of exp are explicit fma calls on both sides.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace xf {

// a double constant materialised in a scalar register pair where it is used
__device__ __forceinline__ double sconst(double c)
{
    asm volatile("" : "+s"(c));
    return c;
}

// a / b rounded as IEEE division for operands whose exponents stay clear of
// the ends of the range: the hardware's own sequence (reciprocal estimate, two
// Newton steps, quotient, one remainder correction) without the operand
// scaling and the special-case fix-up around it, which do nothing there.  Eight
// instructions instead of eleven, and no dependence through the carry register.
// a = +0 gives +0; callers keep |b| and |a| within [2^-500, 2^500] otherwise.
__device__ __forceinline__ double ddiv_core(double a, double b)
{
    double y = __builtin_amdgcn_rcp(b);
    y = fma(y, fma(-b, y, 1.0), y);
    y = fma(y, fma(-b, y, 1.0), y);
    const double q = a * y;
    return fma(fma(-b, q, a), y, q);
}

// RN(a / b) from y = RN(1 / b): Markstein's corrected quotient, with the same
// bounds on the operands as ddiv_core
__device__ __forceinline__ double dquot(double a, double b, double y)
{
    const double q = a * y;
    return fma(fma(-b, q, a), y, q);
}

// sqrt(x), correctly rounded, for x in [2^-700, 2^700]: the hardware estimate
// and the refinement the compiler emits, without its scaling of small x and the
// selects for 0 and infinity (10 instructions instead of 18)
__device__ __forceinline__ double dsqrt_core(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = y * 0.5;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    g = fma(fma(-g, g, x), h, g);
    return fma(fma(-g, g, x), h, g);
}

// exp of NX arguments at once.  The chains are independent, so their fused
// steps fill each other's latency, and each coefficient is put into scalar
// registers once for all of them.  Straight-line: rounding to an integer and
// scaling by 2^k are one instruction each (v_rndne, v_ldexp, which rounds a
// subnormal result once, as the two exact factors of the CPU restatement do),
// and the results outside the finite range come out by themselves: below, x is
// taken at -746, where p 2^-1076 rounds to 0; above, k stays at 1024 while r >= 0
// grows, so p 2^1024 is +inf; a NaN goes through r.
template <int NX> __device__ __forceinline__ void dexp_n(const double *x, double *out)
{
    double r[NX], p[NX];
    int k[NX];
#pragma unroll
    for (int i = 0; i < NX; i++) {
        const double xc = x[i] < -746.0 ? -746.0 : x[i];
        const double kf = __builtin_rint(fmin(xc, 710.0) * 0x1.71547652b82fep+0);
        k[i] = (int)kf;
        // ln2 = LN2_HI + LN2_LO with LN2_HI the double nearest ln2: the first fma
        // is exact (|result| < 1/2 and a multiple of 2^-54)
        r[i] = fma(-kf, 0x1.62e42fefa39efp-1, xc);
        r[i] = fma(-kf, 0x1.abc9e3b39803fp-56, r[i]);
        p[i] = 0x1.6124613a86d09p-33;
    }
    // the coefficients are forced into scalar registers right at their use:
    // the fma then reads them from there, where a literal in a vector
    // register per coefficient (hoisted out of loops) would cost two moves
    // and two vector registers each
    auto step = [&](double c) {
#pragma unroll
        for (int i = 0; i < NX; i++) p[i] = fma(p[i], r[i], c);
    };
    step(sconst(0x1.1eed8eff8d898p-29));
    step(sconst(0x1.ae64567f544e4p-26));
    step(sconst(0x1.27e4fb7789f5cp-22));
    step(sconst(0x1.71de3a556c734p-19));
    step(sconst(0x1.a01a01a01a01ap-16));
    step(sconst(0x1.a01a01a01a01ap-13));
    step(sconst(0x1.6c16c16c16c17p-10));
    step(sconst(0x1.1111111111111p-7));
    step(sconst(0x1.5555555555555p-5));
    step(sconst(0x1.5555555555555p-3));
    step(0x1.0p-1);
    step(1.0);
    step(1.0);
#pragma unroll
    for (int i = 0; i < NX; i++) out[i] = __builtin_amdgcn_ldexp(p[i], k[i]);
}

__device__ __forceinline__ double dexp(double x)
{
    double e;
    dexp_n<1>(&x, &e);
    return e;
}

// log of a positive finite x: the hardware's exponent and mantissa split
// (exact for subnormal x too) in place of the bit operations
__device__ __forceinline__ double dlog_pos(double x)
{
    double m = __builtin_amdgcn_frexp_mant(x); // [1/2, 1)
    int e = __builtin_amdgcn_frexp_exp(x);
    // m in (sqrt(1/2), sqrt(2)]: doubled, exactly, when m <= sqrt(2) / 2
    const int lo = m > 0x1.6a09e667f3bcdp-1 ? 0 : 1;
    m = __builtin_amdgcn_ldexp(m, lo);
    e -= lo;
    const double f = m - 1.0;
    const double s = ddiv_core(f, 2.0 + f); // 2 + f in [1.7, 2.5), f = 0 or |f| >= 2^-53
    const double z = s * s;
    double R = 0x1.642c8590b2164p-4;
    R = 0x1.8618618618618p-4 + z * R;
    R = 0x1.af286bca1af28p-4 + z * R;
    R = 0x1.e1e1e1e1e1e1ep-4 + z * R;
    R = 0x1.1111111111111p-3 + z * R;
    R = 0x1.3b13b13b13b14p-3 + z * R;
    R = 0x1.745d1745d1746p-3 + z * R;
    R = 0x1.c71c71c71c71cp-3 + z * R;
    R = 0x1.2492492492492p-2 + z * R;
    R = 0x1.999999999999ap-2 + z * R;
    R = 0x1.5555555555555p-1 + z * R;
    R = z * R;
    const double t = f - s * (f - R);
    const double ed = (double)e;
    return ed * 0x1.62e42fee00000p-1 + (t + ed * 0x1.a39ef35793c76p-33);
}

__device__ __forceinline__ double dlog(double x)
{
    double v = dlog_pos(x);
    if (__builtin_expect(!(x > 0.0 && x < __longlong_as_double(0x7ff0000000000000LL)), 0)) {
        // NaN -> itself, negative -> NaN, zero -> -inf, +inf -> itself
        v = x;
        if (x < 0.0) v = __longlong_as_double(0x7ff8000000000000LL);
        if (x == 0.0) v = -__longlong_as_double(0x7ff0000000000000LL);
    }
    return v;
}

// max/min with the reference's operand semantics on finite data
__device__ __forceinline__ double dmax(double a, double b) { return a > b ? a : b; }
__device__ __forceinline__ double dmin(double a, double b) { return a < b ? a : b; }

} // namespace xf
