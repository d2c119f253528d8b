// One sample's splat sum and step in the transfer's scalar (double or f32): the context of an item, the
// knot-interpolated Gaussian exponent, the per-sample coefficient sum over a candidate list, the step applied to a
// segment map, and the path weight. Shared by the transfer kernels and the host-side work model.
// Reference: transport.jl:254-290, polarized.jl:110-150, populations.jl:13-104, trajectories.jl:93-128.
#pragma once
#include <cstddef>
#include "ks_kernels.hpp"

namespace ksd {

// ---- splat sums ----------------------------------------------------------------------------------------------
// What a sample's splat sum needs besides the sample itself, in the transfer's scalar S (double or
// f32); the geometry of a sample (metric, tetrad, photon momentum) is always built in FP64.
template <class S>
struct TransCtxT {
    const SplatCT<S>* __restrict__ sp; const S* __restrict__ knots; const S* __restrict__ ktimes;
    int ns, nknots;
    double a, rp, rm, eta, lam, t_obs;          // FP64: geometry and emission times
    S aS, alpha, beta, thetao_sin, nu, L;
};
using TransCtx = TransCtxT<double>;
template <class S>
KS_DEV TransCtxT<S> make_ctx(double a, double rp, double rm, double thetao_sin, double alpha, double beta, double eta, double lam,
                             const SplatCT<S>* sp, int ns, const S* knots, const S* ktimes, int nknots, double t_obs, double nu, double L) {
    TransCtxT<S> c;
    c.sp = sp; c.knots = knots; c.ktimes = ktimes; c.ns = ns; c.nknots = nknots;
    c.a = a; c.rp = rp; c.rm = rm; c.eta = eta; c.lam = lam; c.t_obs = t_obs;
    c.aS = S(a); c.alpha = S(alpha); c.beta = S(beta); c.thetao_sin = S(thetao_sin); c.nu = S(nu); c.L = S(L);
    return c;
}

// The Gaussian exponent at (t, x, y, z) of a splat whose centre follows knots (trajectories.jl:93-128): the offset
// from the knot-interpolated centre (knot_centre), no pattern rotation.
template <class S>
KS_DEV S knot_gexp(const SplatCT<S>& sc, S cx, S cy, S cz, S t, S x, S y, S z) {
    S d0 = x - cx, d1 = y - cy, d2 = z - cz;
    S u0 = sc.R[0] * d0 + sc.R[3] * d1 + sc.R[6] * d2;
    S u1 = sc.R[1] * d0 + sc.R[4] * d1 + sc.R[7] * d2;
    S u2 = sc.R[2] * d0 + sc.R[5] * d1 + sc.R[8] * d2;
    S q0 = u0 * sc.is[0], q1 = u1 * sc.is[1], q2 = u2 * sc.is[2];
    S tt = (t - sc.t0) * sc.iw;
    return q0 * q0 + q1 * q1 + q2 * q2 + tt * tt;
}

// A splat's Gaussian weight at (t, x, y, z), zero where the transport does not count it (outside its support sphere,
// or below the weight cutoff);
// at: t among the splat's knot times, where the caller has it.
template <int KIND, class S>
KS_DEV S splat_weight(const SplatCT<S>& sc, const S* __restrict__ knots, const S* __restrict__ ktimes, S t, S x, S y, S z, const KnotAt<S>* at = nullptr) {
    S gexp;
    if (KIND == MODEL_KNOT || sc.nk > 0) {
        const KnotAt<S> k = at ? *at : knot_at(ktimes + sc.kt0, sc.nk, t);
        S cx, cy, cz;
        knot_centre(knots + 3 * ((int64_t)sc.knot0 + k.kk), sc.nk < 2, k.w, cx, cy, cz);
        gexp = knot_gexp(sc, cx, cy, cz, t, x, y, z);
    } else {
        S sph, cph;
        if (outside_support(sc, t, x, y, z, sph, cph)) return S(0.0);
        gexp = gauss_exponent(sc, t, x, y, z, sph, cph);
    }
    if (gexp > GEXP_SKIP) return S(0.0);
    const S G_ = fexp(-0.5 * gexp);
    return G_ > WEIGHT_CUTOFF ? G_ : S(0.0);
}

// One splat's share of a sample of geometry G, given its weight G_ > 0: the invariant j (c[0..3]), alpha (c[4..7]) and
// rho (c[8..10]) in screen axes; false when it has none (element and screen_coefficients, transport.jl:223-276).
template <int KIND, class S>
KS_DEV bool splat_contribution(const SplatCT<S>& sc, const GeoT<S>& G, S aS, S alpha, S beta, S thetao_sin, S nu, S G_, S c[11]) {
    const FrameT<S> fr = local_frame(G, aS, alpha, beta, thetao_sin, nu, sc.u, sc.gam, sc.q, sc.bh);
    const S nh = fr.nh, inh = fr.inh;
    const S cb = dmin(dmax(fr.cosB, -1.0), 1.0);
    S sth, cth;
    // FP64 takes cos = cb and the product form of the sine; the FP32 path keeps acos and sincos: with the
    // product form, or with the sine taken in FP64 from cb, its images moved further from the FP64 images
    // (9.0e-7 against 6.2e-7 of peak I, 16 x 16 pixels, N = 256, 4 thermal splats), which the sine's
    // accuracy alone does not explain
    if constexpr (std::is_same<S, double>::value) pitch_sincos(cb, sth, cth);
    else sincos(acos(cb), &sth, &cth);
    const S ne = splat_density(sc) * G_;
    const S nuf = fr.nu, inu = inh * (1.0 / NU0);
    CoefT<S> cf;
    if constexpr (KIND == MODEL_THERMAL || KIND == MODEL_KNOT) cf = thermal(ne, sc.p1, sc.g[0], sc.p2, sc.p3, sc.Bmag, fr.nu, nh, inh, sth, cth);
    else if constexpr (KIND == MODEL_POWERLAW) cf = power_coefs(FactorGet<S>{sc.kk}, ne, nuf, inu, sth, cth);
    else if constexpr (KIND == MODEL_KAPPA) cf = kappa_coefs(FactorGet<S>{sc.kk}, ne, nuf, inu, sth, cth);
    else if (sc.kind == MODEL_THERMAL || sc.kind == MODEL_KNOT) cf = thermal(ne, sc.p1, sc.g[0], sc.p2, sc.p3, sc.Bmag, fr.nu, nh, inh, sth, cth);
    else if (sc.kind == MODEL_POWERLAW) cf = power_coefs(FactorGet<S>{sc.kk}, ne, nuf, inu, sth, cth);
    else cf = kappa_coefs(FactorGet<S>{sc.kk}, ne, nuf, inu, sth, cth);
    if (!(cf.jI > 0.0 || cf.aI > 0.0 || cf.rQ != 0.0 || cf.rV != 0.0)) return false;
    const S fe = cap_factor(cf.jI, cf.jQ, cf.jV), fa = cap_factor(cf.aI, cf.aQ, cf.aV);
    const S i2 = inh * inh, s2c = fr.s2, c2c = fr.c2;
    const S jQ = fe * cf.jQ * i2, aQ = fa * cf.aQ * nh, rQ = cf.rQ * nh;
    c[0] = cf.jI * i2; c[1] = jQ * c2c; c[2] = jQ * s2c; c[3] = fe * cf.jV * i2;
    c[4] = cf.aI * nh; c[5] = aQ * c2c; c[6] = aQ * s2c; c[7] = fa * cf.aV * nh;
    c[8] = rQ * c2c; c[9] = rQ * s2c; c[10] = cf.rV * nh;
    return true;
}

// The splat sum of one sample (accumulate_elements, transport.jl:254-276): invariant j, alpha, rho in
// screen axes; false when no splat contributes. One sample at a time, for the work model; the transfer packs the pairs of
// a wavefront's samples instead (transfer_task). With a candidate list only those splats are visited.
template <int KIND, class S>
KS_DEV bool sample_coefficients(const TransCtxT<S>& c, double st, double r, double th, bool nur, bool nuth, S x, S y, S z,
                                S j4[4], S a4[4], S r3[3], const uint16_t* cand = nullptr, int ncand = 0) {
    const S t = S(c.t_obs - st);
    for (int i = 0; i < 4; ++i) { j4[i] = S(0.0); a4[i] = S(0.0); }
    r3[0] = r3[1] = r3[2] = S(0.0);
    bool active = false, geo_ready = false;
    GeoT<S> G;
    const int nloop = cand ? ncand : c.ns;
    for (int ci = 0; ci < nloop; ++ci) {
        const SplatCT<S>& sc = c.sp[cand ? (int)cand[ci] : ci];
        const S G_ = splat_weight<KIND>(sc, c.knots, c.ktimes, t, x, y, z);
        if (!(G_ > 0.0)) continue;
        if (!geo_ready) {
            Geo Gd;
            make_geo(c.a, r, th, c.eta, c.lam, nur, nuth, Gd);
            G = geo_as<S>(Gd);
            geo_ready = true;
        }
        S v[11];
        if (!splat_contribution<KIND>(sc, G, c.aS, c.alpha, c.beta, c.thetao_sin, c.nu, G_, v)) continue;
        for (int q = 0; q < 4; ++q) { j4[q] += v[q]; a4[q] += v[4 + q]; }
        for (int q = 0; q < 3; ++q) r3[q] += v[8 + q];
        active = true;
    }
    return active;
}

// Whether a splat may pass the weight cutoff at a sample, in FP32 on the hardware's sine and cosine, for both
// precisions: false only when splat_weight is zero. The Gaussian exponent is taken to within 2 d (5.3 + d) of its value
// near the cutoff (27.63 = 5.26^2), where d = pm0 + pm1 |t| bounds the error of the splat's scaled coordinates; a bound
// that is not finite lets every sample through. About 45 instructions against 150 to 400 for the weight and 400 to 3000
// for the contribution, which then run on the passing pairs alone, 64 at a time.
// The sample's offset from the splat's centre in the splat's frame (pattern_offset, knot_offset) is apart from the test of
// the offset, so that a caller can place the sample among the knot times once for all splats that share them.
struct SplatTest { float x, y, z, R[9], is[3], t0, iw, omega, pm0, pm1; int knot0, nk, kt0, kind; };     // a SplatCf's first fields
static_assert(sizeof(SplatTest) == 96 && offsetof(SplatCf, kind) + 4 == sizeof(SplatTest), "the prefilter's fields lead SplatCf");
KS_DEV SplatTest splat_test(const SplatCf& c) { SplatTest t; __builtin_memcpy(&t, &c, sizeof t); return t; }
KS_DEV void pattern_offset(const SplatTest& c, float t, float x, float y, float z, float e[3]) {
    float sp, cp;
    hw_sincos(c.omega * (t - c.t0), sp, cp);
    // Rz(-ph) (X - Rz(ph) c) = Rz(-ph) X - c
    e[0] = x * cp + y * sp - c.x; e[1] = y * cp - x * sp - c.y; e[2] = z - c.z;
}
KS_DEV void knot_offset(const f32* __restrict__ K, bool one, float w, float x, float y, float z, float e[3]) {
    f32 cx, cy, cz;
    knot_centre(K, one, f32(w), cx, cy, cz);
    e[0] = x - cx.v; e[1] = y - cy.v; e[2] = z - cz.v;
}
KS_DEV bool offset_may_weigh(const SplatTest& c, float t, const float e[3]) {
    float g = (t - c.t0) * c.iw;
    g = g * g;
    for (int b = 0; b < 3; ++b) {
        const float q = (c.R[b] * e[0] + c.R[3 + b] * e[1] + c.R[6 + b] * e[2]) * c.is[b];
        g += q * q;
    }
    const float d = c.pm1 * fabsf(t) + c.pm0;
    return !(g > 27.641f + 2.0f * d * (5.3f + d));
}
template <int KIND>
KS_DEV bool may_weigh(const SplatTest& c, const f32* __restrict__ knots, const f32* __restrict__ ktimes, float t, float x, float y, float z) {
    float e[3];
    if (KIND == MODEL_KNOT || c.nk > 0) {
        const KnotAt<f32> a = knot_at(ktimes + c.kt0, c.nk, f32(t));
        knot_offset(knots + 3 * ((int64_t)c.knot0 + a.kk), c.nk < 2, a.w.v, x, y, z, e);
    } else {
        pattern_offset(c, t, x, y, z, e);
    }
    return offset_may_weigh(c, t, e);
}
template <int KIND>
KS_DEV bool may_weigh(const SplatCf& c, const f32* __restrict__ knots, const f32* __restrict__ ktimes, float t, float x, float y, float z) {
    return may_weigh<KIND>(splat_test(c), knots, ktimes, t, x, y, z);
}

// g^2 Sigma dtau of a thin sample, g the ZAMO redshift (Splats.jl:113-128)
KS_DEV double thin_weight(double a, double lam, double r, double th, double dtau) {
    double s_, c_; sincos(th, &s_, &c_);
    double S_ = r * r + a * a * c_ * c_, Dl = r * r - 2.0 * r + a * a;
    double Xi = (r * r + a * a) * (r * r + a * a) - a * a * Dl * s_ * s_;
    double g = sqrt(Dl * S_ / Xi) / (1.0 - 2.0 * a * r / Xi * lam);
    return g * g * S_ * dtau;
}

// The FP64 step of an FP32 sample, out of line (the rare samples with a Faraday depth |rho| Delta above
// FARADAY_FP64, where the step's polynomial in K' cancels strongly): O and E in FP64, rounded to FP32. The
// per-sample sums are passed by address here: the transfer measured 13% slower with them passed by value (Step32).
KS_COLD void step_f64_for_f32(const f32 j4[4], const f32 a4[4], const f32 r3[3], f32 D, f32 O[16], f32 E[4]) {
    double jd[4], ad[4], rd[3], Od[16], Ed[4];
    for (int i = 0; i < 4; ++i) { jd[i] = val(j4[i]); ad[i] = val(a4[i]); }
    for (int i = 0; i < 3; ++i) rd[i] = val(r3[i]);
    transfer_step(jd, ad, rd, val(D), Od, Ed);
    for (int i = 0; i < 16; ++i) O[i] = f32(Od[i]);
    for (int i = 0; i < 4; ++i) E[i] = f32(Ed[i]);
}
// One sample's step applied to a segment map, in the transfer's scalar.
template <class S>
KS_DEV void map_step(SegMapT<S>& sm, const S j4[4], const S a4[4], const S r3[3], S D) {
    if constexpr (!std::is_same<S, double>::value) {
        const S fd = sqrt(r3[0] * r3[0] + r3[1] * r3[1] + r3[2] * r3[2]) * D;
        if (fd > FARADAY_FP64) {
            S O[16], E[4];
            step_f64_for_f32(j4, a4, r3, D, O, E);
            sm.advance(O, E);
            return;
        }
    }
    sm.step(j4, a4, r3, D);
}

// Delta = (L / nu-hat) Sigma dtau (transport.jl:282-284)
KS_DEV double path_weight(double L, double nu, double a, double r, double th, double dtau) {
    double ct = cos(th);
    return L / (nu * (1.0 / NU0)) * (r * r + a * a * ct * ct) * dtau;
}

}  // namespace ksd
