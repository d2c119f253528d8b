// Host check of the transfer's FP32 prefilter (the device code is host-callable): may_weigh never rejects a sample at
// which splat_weight is positive, in FP64 or FP32, for pattern and knot splats of widths 0.02 to 3 M, samples crowded
// around the weight cutoff, times up to 1e4 M. The hardware's sine and cosine are taken 4e-6 off (the bound the
// prefilter assumes of them) by turning the sample's position about the axis. Exit status 0 when none was rejected.
#include <cstdio>
#include <random>
#include <vector>
#include "../../kerrsplat_amd/csrc/ks_dsample.hpp"
#include "../../kerrsplat_amd/csrc/ks_hostsplat.hpp"
using namespace ksd;
int main() {
    std::mt19937_64 rng(11);
    std::uniform_real_distribution<double> U(0, 1);
    std::normal_distribution<double> G(0, 1);
    long bad = 0, in = 0, kept = 0, total = 0;
    for (int trial = 0; trial < 200000; ++trial) {
        const bool knots = trial % 2;
        const int nk = knots ? 1 + (int)(6 * U(rng)) : 0;
        double p[21];
        const double r = 3 + 8 * U(rng), ph = 2 * M_PI * U(rng);
        p[0] = r * cos(ph); p[1] = r * sin(ph); p[2] = G(rng);
        for (int q = 0; q < 3; ++q) p[3 + q] = log(0.02) + U(rng) * log(150.0);
        for (int q = 0; q < 4; ++q) p[6 + q] = G(rng);
        p[10] = 20 * G(rng);
        p[11] = U(rng) < 0.3 ? log(3.0) : log(1e9);
        for (int q = 12; q < 20; ++q) p[q] = 0.5;
        p[20] = U(rng) < 0.1 ? 0.0 : (U(rng) < 0.5 ? -1 : 1) * (0.01 + 0.3 * U(rng));
        std::vector<double> K(3 * std::max(nk, 1)), kt(std::max(nk, 1));
        for (int k = 0; k < nk; ++k) {
            kt[k] = (k ? kt[k - 1] : -100.0) + 1 + 99 * U(rng);
            for (int q = 0; q < 3; ++q) K[3 * k + q] = p[q] + 6 * G(rng);
        }
        SplatC c; SplatAdj sa;
        host_splat_constants(MODEL_THERMAL, 21, 0, p, 0.0, knots, K.data(), kt.data(), nk, c, sa);
        SplatCf cf;
        splat_as(c, cf);
        std::vector<f32> Kf(K.begin(), K.end()), ktf(kt.begin(), kt.end());
        // a sample at Gaussian exponent g around the cutoff, in a random direction of the splat's axes
        const double span = U(rng) < 0.3 ? 3.0 : pow(10.0, 4 * U(rng));
        const double t = p[10] + span * (2 * U(rng) - 1);
        const double tt = (t - c.t0) * c.iw, g = 27.631 * (1.0 - pow(10.0, -7 * U(rng))) - tt * tt;
        if (!(g > 0)) continue;
        double n[3], nn = 0;
        for (int q = 0; q < 3; ++q) { n[q] = G(rng); nn += n[q] * n[q]; }
        double e[3] = {0, 0, 0};
        for (int q = 0; q < 3; ++q)
            for (int b = 0; b < 3; ++b) e[b] += c.R[3 * b + q] * n[q] / sqrt(nn) * sqrt(g) / c.is[q];
        double x, y, z;
        if (knots) {
            double cx, cy, cz;
            knot_centre(c, K.data(), kt.data(), t, cx, cy, cz);
            x = cx + e[0]; y = cy + e[1]; z = cz + e[2];
        } else {
            const double a = c.omega * (t - c.t0);
            x = (c.x + e[0]) * cos(a) - (c.y + e[1]) * sin(a); y = (c.x + e[0]) * sin(a) + (c.y + e[1]) * cos(a); z = c.z + e[2];
        }
        ++total;
        const bool w64 = splat_weight<MODEL_THERMAL>(c, K.data(), kt.data(), t, x, y, z) > 0.0;
        const bool w32 = splat_weight<MODEL_THERMAL>(cf, Kf.data(), ktf.data(), f32(t), f32(x), f32(y), f32(z)) > 0.0;
        in += w64;
        for (int s = -1; s <= 1; ++s) {
            const double d = knots ? 0.0 : 4e-6 * s;
            const bool may = may_weigh<MODEL_THERMAL>(cf, Kf.data(), ktf.data(), (float)t, (float)(x * cos(d) - y * sin(d)), (float)(x * sin(d) + y * cos(d)), (float)z);
            kept += may;
            if ((w64 || w32) && !may && ++bad < 6)
                printf("MISS trial %d knots %d t %g rho %g is %g %g %g\n", trial, nk, t, hypot(c.x, c.y), c.is[0], c.is[1], c.is[2]);
        }
    }
    // and far samples are rejected (the prefilter is of use): 6 support radii out
    long far = 0;
    for (int trial = 0; trial < 1000; ++trial) {
        double p[21] = {8, 0, 0, -0.5, -0.5, -0.5, 1, 0, 0, 0, 0, 20, 0, 1, 1, 1, 1, 0, 0, 0, 0.05};
        SplatC c; SplatAdj sa; SplatCf cf;
        host_splat_constants(MODEL_THERMAL, 21, 0, p, 0.0, false, nullptr, nullptr, 0, c, sa);
        splat_as(c, cf);
        const double d = 6 * sqrt(c.rsup2);
        far += may_weigh<MODEL_THERMAL>(cf, (const f32*)nullptr, (const f32*)nullptr, (float)(100 * G(rng)), (float)(d * (1 + U(rng))), (float)d, 0.0f);
    }
    printf("samples %ld, inside the cutoff %ld, kept %ld of %ld, far samples kept %ld, wrongly rejected %ld\n", total, in, kept, 3 * total, far, bad);
    return bad != 0 || far != 0 || in < total / 2;
}
