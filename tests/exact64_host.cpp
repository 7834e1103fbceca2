// hlld64 / hllc64 of kr_exact64.h against the general hlld / hllc of
// kr_physics.h, compiled for the host: the GPU builtins they use are restated
// below (a refined reciprocal from a float's precision, as the kernels form
// it).  argv: samples, lowest exponent of the tiny values.  Prints
// "<in range> <different>" for each of the two.
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <type_traits>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)
static inline double host_rcp(double d) {
    if (d == 0 || !std::isfinite(d)) return 1 / d;
    int e;
    const double m = std::frexp(d, &e);
    return std::ldexp((double)(float)(1 / m), -e);
}
static inline double host_fixup(double q, double d, double n) {
    if (std::isnan(n) || std::isnan(d) || (n == 0 && d == 0) || (std::isinf(n) && std::isinf(d))) return NAN;
    const double s = std::signbit(n) != std::signbit(d) ? -1 : 1;
    if (d == 0 || std::isinf(n)) return s * INFINITY;
    if (n == 0 || std::isinf(d)) return s * 0.0;
    return s * std::fabs(q);
}
static inline double host_scale(double, double d, bool, bool *) { return d; }
static inline double host_fmas(double a, double b, double c, bool) { return std::fma(a, b, c); }
#define __builtin_amdgcn_rcp host_rcp
#define __builtin_amdgcn_div_fixup host_fixup
#define __builtin_amdgcn_div_scale host_scale
#define __builtin_amdgcn_div_fmas host_fmas
#define __builtin_amdgcn_rcpf(x) (1.f / (x))
#define __builtin_amdgcn_sqrtf __builtin_sqrtf
#define __builtin_amdgcn_rsqf(x) (1.f / __builtin_sqrtf(x))
static inline int __double2hiint(double x) {
    int64_t b;
    std::memcpy(&b, &x, 8);
    return (int)(b >> 32);
}
static inline long long __double_as_longlong(double x) {
    long long b;
    std::memcpy(&b, &x, 8);
    return b;
}
static inline bool __any(bool b) { return b; }
static inline bool __all(bool b) { return b; }

#include "kr_exact64.h"

int main(int, char **argv) {
    const long samples = std::atol(argv[1]);
    const double low = std::atof(argv[2]);
    std::mt19937_64 rng(7);
    auto unit = [&] { return std::uniform_real_distribution<double>(0, 1)(rng); };
    auto power = [&](double lo, double hi) {
        return std::ldexp(1 + unit(), (int)std::floor(lo + (hi - lo) * unit()));
    };
    // a value near x: equal, a few ulps off, or anything between
    auto near = [&](double x) {
        return unit() < 0.4 ? x : x * (1 + (unit() - 0.5) * std::ldexp(1, -(int)(52 * unit())));
    };
    const double gamma = 5. / 3., cv = 1 / (gamma - 1);
    const kr::Gam64 k{gamma, cv, 1 / cv + 1};
    for (int nv : {8, 5}) {
        long in = 0, bad = 0;
        for (long i = 0; i < samples; ++i) {
            // units up to 2^58 around 1, speeds about 1 / 8 to 4 of the sound's
            const double range = (int)(3 * unit()) * 29, b0 = range * (2 * unit() - 1), b1 = range * (2 * unit() - 1);
            double l[8] = {power(b0 - 1, b0 + 1), power(b1 - 1, b1 + 1)}, r[8] = {near(l[0]), near(l[1])};
            const double c = std::sqrt(l[1] / l[0]), b = std::sqrt(l[1]);
            double big = l[0] + l[1] + r[0] + r[1];
            for (int v = 2; v < nv; ++v) {
                const double s = v < 5 ? c : b, p = unit();
                const double x = p < 0.25   ? 0
                                 : p < 0.5  ? s * power(-3, 2)
                                 : p < 0.6  ? s * power(-60, -40)
                                 : p < 0.7  ? power(low, low + 20)
                                 : p < 0.85 ? power(low, low + 400)
                                            : power(-560, -400);
                l[v] = unit() < 0.5 ? -x : x;
                const double q = unit();
                r[v] = q < 0.8 ? near(l[v]) : (q < 0.9 ? 0 : power(low, low + 300));
                big += std::fabs(l[v]) + std::fabs(r[v]);
            }
            r[5] = l[5];                        // one normal field at the face
            double f[8] = {0}, g[8] = {0};
            if (nv == 8) {
                kr::hlld64(f, l, r, k);
                kr::hlld<double>(g, l, r, gamma);
            } else {
                kr::hllc64(f, l, r, k);
                kr::hllc<double>(g, l, r, gamma);
            }
            in += big < 0x1p60;
            for (int v = 0; v < nv; ++v)
                if (v != 5 && f[v] != g[v] && !(std::isnan(f[v]) && std::isnan(g[v]))) {
                    ++bad;
                    break;
                }
        }
        std::printf("%ld %ld\n", in, bad);
    }
    return 0;
}
