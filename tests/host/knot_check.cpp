// Host check of the knot interval (knot_at) at the times that a model keeps (knot_times_as): for knot times that FP32 may not
// tell apart, the kept ones increase and stay within FP32's rounding and a step a knot of them, and the interval gives the
// centre that holds the first knot up to its time, the last one from its time on, and interpolates in between, at times on
// the knots, beside them and far outside. Exit status 0 when every centre is finite and agrees to rounding.
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>
#include "../../kerrsplat_amd/csrc/ks_hostsplat.hpp"
using namespace ksd;
template <class S> double centre(const std::vector<double>& kt, const std::vector<double>& K, double t, bool held) {
    std::vector<S> ktS(kt.size()), KS(3 * K.size());
    knot_times_as(kt.data(), (int)kt.size(), ktS.data());
    for (size_t k = 0; k < kt.size(); ++k)
        if ((k && !(ktS[k] > ktS[k - 1])) || fabs(val(ktS[k]) - kt[k]) > 1.2e-7 * (k + 1) * fmax(fabs(kt[k]), 1.0)) return NAN;
    for (size_t k = 0; k < K.size(); ++k) KS[3 * k] = KS[3 * k + 1] = KS[3 * k + 2] = S(K[k]);
    const int nk = (int)kt.size();
    const S tS = S(t);
    if (!held) {
        const KnotAt<S> a = knot_at(ktS.data(), nk, tS);
        if (a.kk < 0 || a.kk > (nk > 1 ? nk - 2 : 0)) return NAN;
        S x, y, z;
        knot_centre(KS.data() + 3 * a.kk, nk < 2, a.w, x, y, z);
        return val(x);
    }
    // the sequential rule, in the same scalar
    if (tS <= ktS[0]) return val(KS[0]);
    if (tS >= ktS[nk - 1]) return val(KS[3 * (nk - 1)]);
    int k = 0;
    while (k < nk - 2 && ktS[k + 1] <= tS) ++k;
    const S w = (tS - ktS[k]) / (ktS[k + 1] - ktS[k]);
    return val((1.0 - w) * KS[3 * k] + w * KS[3 * k + 3]);
}
template <class S> long check(std::mt19937_64& rng, double eps, long& n) {
    std::uniform_real_distribution<double> U(0, 1);
    long bad = 0;
    for (int trial = 0; trial < 20000; ++trial) {
        const int nk = 1 + (int)(6 * U(rng));
        std::vector<double> kt(nk), K(nk);
        for (int k = 0; k < nk; ++k) {
            // steps of 1 to 100, or far below FP32's spacing at the time
            const double t0 = k ? kt[k - 1] : -150.0 + 300.0 * U(rng);
            kt[k] = k == 0 ? t0 : t0 + (U(rng) < 0.4 ? 1e-9 * (1 + U(rng)) : 1 + 99 * U(rng));
            K[k] = 20 * U(rng) - 10;
        }
        std::vector<double> ts = {kt[0] - 1e6, kt[nk - 1] + 1e6, kt[0] - 3.0, kt[nk - 1] + 3.0};
        for (int k = 0; k < nk; ++k) for (double d : {0.0, 1e-10, -1e-10, 1e-4, -1e-4, 0.7}) ts.push_back(kt[k] + d);
        for (double t : ts) {
            const double got = centre<S>(kt, K, t, false), ref = centre<S>(kt, K, t, true);
            ++n;
            // rounding of the weight: the time's and the step's, 1 at the least apart where the step is not lost
            if (!(fabs(got - ref) <= 40.0 * eps) && ++bad < 6) printf("nk %d t %.12g: %g instead of %g\n", nk, t, got, ref);
        }
    }
    return bad;
}
int main() {
    std::mt19937_64 rng(5);
    long n = 0;
    const long b32 = check<f32>(rng, 6e-8, n), b64 = check<double>(rng, 1.2e-16, n);
    printf("times %ld, wrong in FP32 %ld, in FP64 %ld\n", n, b32, b64);
    return b32 != 0 || b64 != 0;
}
