// Host check of the transfer's elementary functions (the device code is host-callable) against 64-bit-mantissa values: the
// largest error over two million arguments of the ranges that the fits use, in units of the last place, and the values at
// zero, infinity and NaN. Exit status 0 when every error is below 2 ulp: a function's last operation rounds half an ulp, the
// corrections it adds carry at most another half, and an ulp doubles from one end of a binade to the other.
#include <cmath>
#include <cstdio>
#include <random>
#include "../../kerrsplat_amd/csrc/ks_dfun.hpp"
using namespace ksd;
static int bad = 0;
struct Worst {
    const char* name; int bits; double mx = 0.0;
    void add(double got, long double ref) {
        const long double a = fabsl(ref);
        if (!(a > (bits == 53 ? 1e-300L : 1e-36L)) || !std::isfinite((double)ref)) return;
        const double e = (double)(fabsl((long double)got - ref) / ldexpl(1.0L, ilogbl(a) - bits + 1));
        if (!(e <= mx)) mx = e;
    }
    void end() { printf("%s %.3f\n", name, mx); if (!(mx < 2.0)) ++bad; }
};
static void same(const char* what, double got, double want) {
    if (!(got == want || (std::isnan(got) && std::isnan(want)))) { printf("%s: %g, not %g\n", what, got, want); ++bad; }
}
int main() {
    std::mt19937_64 rng(5);
    std::uniform_real_distribution<double> U(0, 1);
    Worst wp{"pow", 53}, we{"exp", 53}, wl{"ln", 53}, w1{"log1p", 53}, ws{"sin", 53}, wc{"cos", 53}, f1{"log1p, FP32", 24}, fs{"sin, FP32", 24}, fc{"cos, FP32", 24};
    for (long i = 0; i < 2000000; ++i) {
        const double x = i % 3 == 0 ? 0.5 + 1.5 * U(rng) : (i % 7 == 0 ? 1 + 1e-6 * (U(rng) - 0.5) : std::pow(10.0, -12 + 24 * U(rng)));
        const double y = (U(rng) - 0.5) * (i % 2 ? 20 : 4), z = -700 * U(rng) * (i % 2 ? 1 : 0.01) + (i % 5 == 0 ? 300 * U(rng) : 0);
        const double w = std::pow(10.0, -20 + 26 * U(rng)), an = (U(rng) - 0.5) * (i % 2 ? 20 : 1e4);
        wp.add(pow_of(pow_base(x), y), powl(x, y));
        we.add(fexp(z), expl(z));
        wl.add(ln_of(pow_base(x)), logl(x));
        w1.add(log1p_pos(w), log1pl(w));
        double s, c;
        sincos_small(an, &s, &c);
        ws.add(s, sinl(an)); wc.add(c, cosl(an));
        const float wf = (float)w, af = (float)(an * 0.1);
        f32 s_, c_;
        sincos_small(f32(af), &s_, &c_);
        f1.add(log1p_pos(f32(wf)).v, log1pl(wf)); fs.add(s_.v, sinl(af)); fc.add(c_.v, cosl(af));
    }
    for (Worst* w : {&wp, &we, &wl, &w1, &ws, &wc, &f1, &fs, &fc}) w->end();
    const double inf = INFINITY, tiny = 5e-324;
    same("0^0.3", pow_of(pow_base(0.0), 0.3), 0.0);
    same("0^-0.3", pow_of(pow_base(0.0), -0.3), inf);
    same("(-0)^0.3", pow_of(pow_base(-0.0), 0.3), 0.0);
    same("inf^0.3", pow_of(pow_base(inf), 0.3), inf);
    same("inf^-0.3", pow_of(pow_base(inf), -0.3), 0.0);
    same("3^0", pow_of(pow_base(3.0), 0.0), 1.0);
    same("(-1)^0.3", pow_of(pow_base(-1.0), 0.3), NAN);
    same("NaN^0.3", pow_of(pow_base(NAN), 0.3), NAN);
    same("smallest^0.5", pow_of(pow_base(tiny), 0.5), std::sqrt(tiny));
    same("largest^2", pow_of(pow_base(1e300), 2.0), inf);
    same("exp(-inf)", fexp(-inf), 0.0);
    same("exp(inf)", fexp(inf), inf);
    same("exp(NaN)", fexp(NAN), NAN);
    same("exp(0)", fexp(0.0), 1.0);
    same("exp(-1e4)", fexp(-1e4), 0.0);
    same("log1p(0)", log1p_pos(0.0), 0.0);
    return bad ? 1 : 0;
}
