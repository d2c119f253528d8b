// Host check of the power-law fits in FP32 over field strengths of 1e-24 to 1e21 G and pitch angles down to 1e-9: every
// coefficient whose FP64 value FP32 can hold is finite (where nu / nu_c passes FP32's range the emission is zero, not
// infinity times zero), and agrees with FP64 to 1e-3 where FP32's intermediate powers are in range (nu / nu_c within
// 1e-6 .. 1e6 and values above 1e-25). The powers are good to |y log2 x| 2^-23, 4e-6 there, and 1 - (nu_min / nu)^(p/2 - 1)
// loses what it cancels, at the least 1 / 30 of one. Exit status 0 when all do.
#include <cmath>
#include <cstdio>
#include <random>
#include "../../kerrsplat_amd/csrc/ks_dsample.hpp"
#include "../../kerrsplat_amd/csrc/ks_hostsplat.hpp"
using namespace ksd;
template <class S> void coefs(const SplatC& c, double ne, double nu, double sth, double cth, double v[8]) {
    SplatCT<S> sc;
    splat_as(c, sc);
    const S nuf = S(nu), inu = S(1.0 / nu);
    const CoefT<S> f = power_coefs(FactorGet<S>{sc.kk}, S(ne), nuf, inu, S(sth), S(cth));
    const S q[8] = {f.jI, f.jQ, f.jV, f.aI, f.aQ, f.aV, f.rQ, f.rV};
    for (int i = 0; i < 8; ++i) v[i] = val(q[i]);
}
int main() {
    std::mt19937_64 rng(3);
    std::uniform_real_distribution<double> U(0, 1);
    long n = 0, infinite = 0, off = 0, compared = 0;
    for (int trial = 0; trial < 200000; ++trial) {
        double p[22] = {5, 0, 0, 0, 0, 0, 1, 0, 0, 0, 0, 20, 0};
        p[13] = 2.2 + 5 * U(rng);
        p[14] = log(1.0) + U(rng) * log(300.0);
        p[15] = U(rng) < 0.3 ? log(10.0) + 2 * (2 * U(rng) - 1) : -55.0 + 103.0 * U(rng);
        for (int q = 16; q < 21; ++q) p[q] = 0.5;
        SplatC c; SplatAdj sa;
        host_splat_constants(MODEL_POWERLAW, 22, 0, p, 1e6, false, nullptr, nullptr, 0, c, sa);
        const double ne = pow(10.0, 8 * U(rng)), nu = 230e9 * pow(10.0, 2 * U(rng) - 1);
        const double th = U(rng) < 0.3 ? pow(10.0, -9 * U(rng)) : M_PI / 2 * U(rng), sth = sin(th), cth = cos(th);
        const double X = nu * c.kk.v[PL_INUC] / sth, numin = 1.0 / (X * c.kk.v[PL_RG]);
        double v32[8], v64[8];
        coefs<f32>(c, ne, nu, sth, cth, v32);
        coefs<double>(c, ne, nu, sth, cth, v64);
        for (int i = 0; i < 8; ++i) {
            if (!(fabs(v64[i]) < 1e30)) continue;
            ++n;
            if (!std::isfinite(v32[i]) && ++infinite < 6) printf("infinite: lnB %g sin %g p %g coefficient %d: %g, %g in FP64\n", p[15], sth, p[13], i, v32[i], v64[i]);
            if (!(X > 1e-6 && X < 1e6 && fabs(v64[i]) > 1e-25) || (i == 6 && fabs(1 - pow(numin, p[13] / 2 - 1)) < 1.0 / 30)) continue;
            ++compared;
            if (!(fabs(v32[i] - v64[i]) <= 1e-3 * fabs(v64[i])) && ++off < 6) printf("off: lnB %g sin %g p %g X %g coefficient %d: %g, %g in FP64\n", p[15], sth, p[13], X, i, v32[i], v64[i]);
        }
    }
    printf("values %ld, not finite %ld; compared %ld, off %ld\n", n, infinite, compared, off);
    return infinite != 0 || off != 0;
}
