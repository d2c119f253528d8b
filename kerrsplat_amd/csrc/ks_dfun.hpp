// Elementary functions of the transfer's coefficient fits in its scalars (double, f32, duals), in the forms the fits
// need: several powers of one base from one logarithm, exponentials and bounded sines without the library's
// large-argument and special-value code at every call.
//
// The library's FP64 pow is 224 vector instructions (154 of them FP64), log 98, exp 42, log1p 113, sin or cos 151, and a
// pair of a splat and a sample takes up to 22 powers. Here a base costs about 60 (its logarithm to 2^-64 relative),
// each power of it 20, exp 22, log1p 66, a bounded sine 30. Measured against 64-bit-mantissa values the FP64 functions are
// within 1.0 to 1.5 ulp, 0.29 to 0.37 ulp in the root mean square (a correctly rounded one 0.29).
#pragma once
#include "ks_ddual.hpp"

namespace ksd {

// ---- FP64 ---------------------------------------------------------------------------------------------------------
KS_DEV double rcp_start(double d) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcp(d);
#else
    return (double)(1.0f / (float)d);
#endif
}
KS_DEV double frexp_split(double x, int& e) {
#if defined(__HIP_DEVICE_COMPILE__)
    e = __builtin_amdgcn_frexp_exp(x);
    return __builtin_amdgcn_frexp_mant(x);
#else
    return ::frexp(x, &e);
#endif
}
// 2^(t + tl), |tl| far below one: k = rint(t), then 2^r on |r| <= 1/2 as 1 + r (ln 2 + r g(r)), g the polynomial through
// (2^r - 1 - r ln 2) / r^2 at the ten Chebyshev nodes of the interval (6e-17 off). pm1 is 2^r - 1, k the exponent.
KS_DEV void exp2_parts(double t, double tl, double& pm1, double& k) {
    k = ::rint(t);
    const double r = (t - k) + tl;
    double g = 4.4541034105870405e-10;
    g = ::fma(g, r, 7.070977866508138e-09);
    g = ::fma(g, r, 1.0178067267449427e-07);
    g = ::fma(g, r, 1.3215451633221434e-06);
    g = ::fma(g, r, 1.5252733820795803e-05);
    g = ::fma(g, r, 0.00015403530424776529);
    g = ::fma(g, r, 0.0013333558146423213);
    g = ::fma(g, r, 0.009618129107618665);
    g = ::fma(g, r, 0.05550410866482158);
    g = ::fma(g, r, 0.24022650695910075);
    pm1 = r * ::fma(g, r, 0.6931471805599453);
}
KS_DEV double exp2_ext(double t, double tl) {
    double p, k;
    exp2_parts(t, tl, p, k);
    return ::ldexp(1.0 + p, (int)::fmax(::fmin(k, 4000.0), -4000.0));
}
// e^x: x log2 e to twice the precision, then exp2_ext; 0 and infinity beyond |x| = 1e5, NaN for NaN
KS_DEV double fexp(double x) {
    const double t = x * 1.4426950408889634;
    const double e = exp2_ext(t, ::fma(x, 2.0355273740931033e-17, ::fma(x, 1.4426950408889634, -t)));
    return ::fabs(x) < 1e5 ? e : (x > 0.0 ? INFINITY : (x < 0.0 ? 0.0 : x));
}

// log2 x = hi + lo to 2^-64 relative: x = 2^e m with m in [sqrt(1/2), sqrt(2)), s = (m - 1) / (m + 1) as a sum of two,
// log2 m = (2 / ln 2) atanh s, whose series past s^3 / 3 is a polynomial in s^2 (eight Chebyshev nodes, 1.3e-17 off).
// Zero and infinity give -+2^60 (whose powers are 0 and infinity for any exponent above 1e-15), other bases NaN.
template <class T> struct PowBase;
template <> struct PowBase<double> { double hi, lo; };
KS_DEV PowBase<double> pow_base(double x) {
    int e;
    double m = frexp_split(x, e);
    const int up = m < 0.7071067811865476 ? 1 : 0;
    m = ::ldexp(m, up);
    const double f = m - 1.0, d = m + 1.0, dl = m - (d - 1.0), de = (double)(e - up);
    double r = rcp_start(d);
    r = ::fma(::fma(-d, r, 1.0), r, r);
    r = ::fma(::fma(-d, r, 1.0), r, r);
    const double s = f * r;
    double sl = ::fma(-s, dl, ::fma(-s, d, f)) * r;
    const double z = s * s, zl = ::fma(s, s, -z) + 2.0 * (s * sl);
    double q = 0.058615893119382576;
    q = ::fma(q, z, 0.05853118169745603);
    q = ::fma(q, z, 0.06667402346923655);
    q = ::fma(q, z, 0.07692297481259215);
    q = ::fma(q, z, 0.09090909167696401);
    q = ::fma(q, z, 0.11111111110827943);
    q = ::fma(q, z, 0.14285714285714682);
    q = ::fma(q, z, 0.2);
    // atanh s = s + s (z / 3 + z^2 q)
    const double ph = z * (1.0 / 3.0);
    const double pl = ::fma(z * z, q, ::fma(z, 1.0 / 3.0, -ph) + ::fma(z, 1.850371707708594e-17, zl * (1.0 / 3.0)));
    const double u = s * ph, A = s + u;
    const double Al = ((s - A) + u) + (::fma(s, ph, -u) + ::fma(s, pl, ::fma(sl, ph, sl)));
    const double H = A * 2.8853900817779268;
    const double Hl = ::fma(A, 2.8853900817779268, -H) + ::fma(A, 4.0710547481862066e-17, Al * 2.8853900817779268);
    PowBase<double> b;
    b.hi = de + H;
    b.lo = ((de - b.hi) + H) + Hl;
    if (!(x > 0.0 && x < INFINITY)) {
        b.hi = x == 0.0 ? -1152921504606846976.0 : (x > 0.0 ? 1152921504606846976.0 : NAN);
        b.lo = 0.0;
    }
    return b;
}
KS_DEV double pow_of(const PowBase<double>& b, double y) {
    const double t = y * b.hi;
    return exp2_ext(t, ::fma(y, b.lo, ::fma(y, b.hi, -t)));
}
KS_DEV double ln_of(const PowBase<double>& b) {
    return ::fma(b.hi, 0.6931471805599453, ::fma(b.hi, 2.3190468138462996e-17, b.lo * 0.6931471805599453));
}
// log(1 + y), y >= 0: the logarithm of the rounded sum and the part that rounding left out
KS_DEV double log1p_pos(double y) {
    const double u = 1.0 + y, t = u - 1.0;
    const double c = (1.0 - (u - t)) + (y - t);
    const PowBase<double> b = pow_base(u);
    return ::fma(b.hi, 0.6931471805599453, ::fma(b.hi, 2.3190468138462996e-17, ::fma(b.lo, 0.6931471805599453, c * rcp_start(u))));
}
// sine and cosine: the angle less its nearest multiple of pi / 2 (two fused steps, exact to 1e-16 up to 1e5 rad), then the
// Taylor series of both on |r| <= pi / 4, whose first dropped terms are below 1e-19. About 35 instructions against the
// library's 150, whose large-argument reduction is inlined at every call. sincos_small: |x| < 1e5 only.
KS_DEV void sincos_small(double x, double* s, double* c) {
    const double n = ::rint(x * 0.6366197723675814);
    const double w = ::fma(-n, 1.5707963267948966, x), r = ::fma(-n, 6.123233995736766e-17, w);
    const double rl = ::fma(-n, 6.123233995736766e-17, w - r), q = r * r;
    double ps = -1.0 / 6.0 + q * (1.0 / 120.0 + q * (-1.0 / 5040.0 + q * (1.0 / 362880.0 + q * (-1.0 / 39916800.0 +
                q * (1.0 / 6227020800.0 + q * (-1.0 / 1307674368000.0 + q * (1.0 / 355687428096000.0)))))));
    double pc = -0.5 + q * (1.0 / 24.0 + q * (-1.0 / 720.0 + q * (1.0 / 40320.0 + q * (-1.0 / 3628800.0 + q * (1.0 / 479001600.0 +
                q * (-1.0 / 87178291200.0 + q * (1.0 / 20922789888000.0 + q * (-1.0 / 6402373705728000.0))))))));
    const double sr = r + ::fma(r * q, ps, rl), cr = 1.0 + ::fma(q, pc, -(r * rl));
    const int m = (int)n;
    const double sv = (m & 1) ? cr : sr, cv = (m & 1) ? sr : cr;
    *s = (m & 2) ? -sv : sv;
    *c = ((m + 1) & 2) ? -cv : cv;
}
KS_COLD void sincos_large(double x, double* s, double* c) { ::sincos(x, s, c); }
KS_DEV void phase_sincos(double x, double* s, double* c) {
    if (!(::fabs(x) < 1e5)) { sincos_large(x, s, c); return; }
    sincos_small(x, s, c);
}

// ---- FP32: the powers on the hardware's base-2 functions (hw_pow), exp the library's ---------------------------------
template <> struct PowBase<f32> { float x, l; };
KS_DEV PowBase<f32> pow_base(f32 x) { PowBase<f32> b; b.x = x.v; b.l = hw_log2(x.v); return b; }
KS_DEV f32 pow_of(const PowBase<f32>& b, f32 y) { const float p = hw_exp2(y.v * b.l); return f32(y.v == 0.0f ? 1.0f : p); }
KS_DEV f32 pow_of(const PowBase<f32>& b, double y) { return pow_of(b, f32(y)); }
KS_DEV f32 ln_of(const PowBase<f32>& b) { return log(f32(b.x)); }
KS_DEV f32 fexp(f32 x) { return exp(x); }
// log(1 + y), y >= 0: 30 instructions against the library's 117
KS_DEV f32 log1p_pos(f32 y) {
    const float u = 1.0f + y.v, t = u - 1.0f, c = (1.0f - (u - t)) + (y.v - t);
    return f32(fmaf(c, 1.0f / u, logf(u)));
}
// three fused steps of the reduction, Taylor series to r^9 and r^10 (3e-9 off); the library's takes 127 instructions
KS_DEV void sincos_small(f32 x, f32* s, f32* c) {
    const float n = rintf(x.v * 0.636619772f);
    float w = fmaf(-n, 1.57079637f, x.v);
    w = fmaf(-n, -4.37113883e-08f, w);
    const float r = fmaf(-n, -1.71512488e-15f, w), rl = fmaf(-n, -1.71512488e-15f, w - r), q = r * r;
    const float ps = -1.0f / 6.0f + q * (1.0f / 120.0f + q * (-1.0f / 5040.0f + q * (1.0f / 362880.0f)));
    const float pc = -0.5f + q * (1.0f / 24.0f + q * (-1.0f / 720.0f + q * (1.0f / 40320.0f + q * (-1.0f / 3628800.0f))));
    const float sr = r + fmaf(r * q, ps, rl), cr = 1.0f + fmaf(q, pc, -(r * rl));
    const int m = (int)n;
    const float sv = (m & 1) ? cr : sr, cv = (m & 1) ? sr : cr;
    *s = f32((m & 2) ? -sv : sv);
    *c = f32(((m + 1) & 2) ? -cv : cv);
}
// (a splat's phase keeps the library's: its rounding moves rho_V, see is_fp32)
KS_DEV void phase_sincos(f32 x, f32* s, f32* c) { sincos(x, s, c); }

// ---- duals: the value's function and its chain rule -------------------------------------------------------------------
template <int N, class S> struct PowBase<DN<N, S>> { DN<N, S> x; PowBase<S> b; S ix; };
template <int N, class S> KS_DEV PowBase<DN<N, S>> pow_base(const DN<N, S>& x) {
    PowBase<DN<N, S>> o;
    o.x = x; o.b = pow_base(x.v); o.ix = x.v != 0.0 ? S(1.0 / x.v) : S(0.0);
    return o;
}
template <int N, class S> KS_DEV DN<N, S> pow_of(const PowBase<DN<N, S>>& b, double y) {
    const S p = pow_of(b.b, y);
    return chain(p, S(y * p * b.ix), b.x);
}
template <int N, class S> KS_DEV DN<N, S> pow_of(const PowBase<DN<N, S>>& b, const DN<N, S>& y) {
    const S p = pow_of(b.b, y.v), dx = y.v * p * b.ix, dy = b.x.v > 0.0 ? S(p * ln_of(b.b)) : S(0.0);
    DN<N, S> r;
    r.v = p;
    for (int i = 0; i < N; ++i) r.d[i] = dx * b.x.d[i] + dy * y.d[i];
    return r;
}
template <int N, class S> KS_DEV DN<N, S> ln_of(const PowBase<DN<N, S>>& b) { return chain(ln_of(b.b), b.ix, b.x); }
template <int N, class S> KS_DEV DN<N, S> fexp(const DN<N, S>& x) { const S e = fexp(x.v); return chain(e, e, x); }
template <int N, class S> KS_DEV DN<N, S> log1p_pos(const DN<N, S>& y) { return chain(log1p_pos(y.v), S(1.0 / (1.0 + y.v)), y); }
template <int N, class S> KS_DEV void sincos_small(const DN<N, S>& x, DN<N, S>* s, DN<N, S>* c) {
    S sv, cv;
    sincos_small(x.v, &sv, &cv);
    *s = chain(sv, cv, x); *c = chain(cv, S(-sv), x);
}
template <int N, class S> KS_DEV void phase_sincos(const DN<N, S>& x, DN<N, S>* s, DN<N, S>* c) {
    S sv, cv;
    phase_sincos(x.v, &sv, &cv);
    *s = chain(sv, cv, x); *c = chain(cv, S(-sv), x);
}
// x^e (0 < e < 1) of x >= 0, zero with zero partials at x = 0, where the derivative is unbounded (the reference's
// safe_sqrt makes the same choice for the square root, frames.jl:83-97)
template <class T> KS_DEV T pow_nonneg(T x, double e) { return x > 0.0 ? pow_of(pow_base(x), e) : T(0.0); }

}  // namespace ksd
