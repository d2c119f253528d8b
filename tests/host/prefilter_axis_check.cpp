// Host check of the FP32 prefilter for pattern splats near the spin axis: centres 0 to 3 M off it, widths 0.02 to 3 M drawn
// per axis, times up to 1e4 M, samples crowded around the weight cutoff. The prefilter turns the sample by the pattern's
// phase, so an error of the phase moves the sample by its own distance from the axis, whatever the centre's. The device's
// phase error is modelled by turning the sample by 4e-6 (the hardware's sine and cosine) and 1.2e-7 of the phase (the
// roundings of x / 2 pi) either way. Exit status 0 when no sample at which splat_weight is positive was rejected.
#include <cstdio>
#include <random>
#include "../../kerrsplat_amd/csrc/ks_dsample.hpp"
#include "../../kerrsplat_amd/csrc/ks_hostsplat.hpp"
using namespace ksd;
int main() {
    std::mt19937_64 rng(23);
    std::uniform_real_distribution<double> U(0, 1);
    std::normal_distribution<double> G(0, 1);
    long bad = 0, in = 0, total = 0;
    for (int trial = 0; trial < 200000; ++trial) {
        double p[21];
        const double r = U(rng) < 0.1 ? 0.0 : 3.0 * pow(10.0, -3.0 * U(rng)), ph = 2 * M_PI * U(rng);
        p[0] = r * cos(ph); p[1] = r * sin(ph); p[2] = 4 * G(rng);
        for (int q = 0; q < 3; ++q) p[3 + q] = log(0.02) + U(rng) * log(150.0);
        for (int q = 0; q < 4; ++q) p[6 + q] = G(rng);
        p[10] = 20 * G(rng);
        p[11] = U(rng) < 0.3 ? log(3.0) : log(1e9);
        for (int q = 12; q < 20; ++q) p[q] = 0.5;
        p[20] = (U(rng) < 0.5 ? -1 : 1) * (0.01 + 0.3 * U(rng));
        SplatC c; SplatAdj sa;
        host_splat_constants(MODEL_THERMAL, 21, 0, p, 0.0, false, nullptr, nullptr, 0, c, sa);
        SplatCf cf;
        splat_as(c, cf);
        // a sample at Gaussian exponent g just inside the cutoff, in a random direction of the splat's axes
        const double t = p[10] + pow(10.0, 4 * U(rng)) * (2 * U(rng) - 1);
        const double tt = (t - c.t0) * c.iw, g = 27.631 * (1.0 - pow(10.0, -7 * U(rng))) - tt * tt;
        if (!(g > 0)) continue;
        double n[3], nn = 0, e[3] = {0, 0, 0};
        for (int q = 0; q < 3; ++q) { n[q] = G(rng); nn += n[q] * n[q]; }
        for (int q = 0; q < 3; ++q)
            for (int b = 0; b < 3; ++b) e[b] += c.R[3 * b + q] * n[q] / sqrt(nn) * sqrt(g) / c.is[q];
        const double a = c.omega * (t - c.t0);
        const double x = (c.x + e[0]) * cos(a) - (c.y + e[1]) * sin(a), y = (c.x + e[0]) * sin(a) + (c.y + e[1]) * cos(a), z = c.z + e[2];
        ++total;
        const bool w64 = splat_weight<MODEL_THERMAL>(c, (const double*)nullptr, (const double*)nullptr, t, x, y, z) > 0.0;
        const bool w32 = splat_weight<MODEL_THERMAL>(cf, (const f32*)nullptr, (const f32*)nullptr, f32(t), f32(x), f32(y), f32(z)) > 0.0;
        in += w64;
        for (int s = -1; s <= 1; ++s) {
            const double d = s * (4e-6 + 1.2e-7 * fabs(a));
            const bool may = may_weigh<MODEL_THERMAL>(cf, (const f32*)nullptr, (const f32*)nullptr, (float)t, (float)(x * cos(d) - y * sin(d)),
                                                      (float)(x * sin(d) + y * cos(d)), (float)z);
            if ((w64 || w32) && !may && ++bad < 6)
                printf("MISS trial %d t %g rho %g is %g %g %g\n", trial, t, hypot(c.x, c.y), c.is[0], c.is[1], c.is[2]);
        }
    }
    printf("samples %ld, inside the cutoff %ld, wrongly rejected %ld\n", total, in, bad);
    return bad != 0 || in < total / 2;
}
