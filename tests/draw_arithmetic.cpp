// The draws' arithmetic (csrc/sn_device.h) on the host, against 64-bit mantissas.
// The hardware's reciprocal and reciprocal root are stood in for by ones that
// are off by up to 2^-24 relative, one way or the other: the iterations after
// them have to make up for it.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <random>
using std::min;

static uint64_t state = 88172645463325252ull;
static double off()   // 1 + e, |e| <= 2^-24
{
    state ^= state << 13; state ^= state >> 7; state ^= state << 17;
    return 1.0 + ldexp((double)(int64_t)state, -63 - 24);
}
static double sn_rcp(double x) { return 1.0 / x * off(); }
static double sn_rsq(double x) { return 1.0 / sqrt(x) * off(); }
static double sn_mant(double x) { int e; return frexp(x, &e); }
static int sn_exp(double x) { int e; (void)frexp(x, &e); return e; }
#define __builtin_amdgcn_rcp sn_rcp
#define __builtin_amdgcn_rsq sn_rsq
#define __builtin_amdgcn_frexp_mant sn_mant
#define __builtin_amdgcn_frexp_exp sn_exp
#include "sn_device.h"

static double ulp(double x) { return nextafter(fabs(x), INFINITY) - fabs(x); }

int main()
{
    std::mt19937_64 g(1);
    const uint64_t one = 1ull << 53, root = (uint64_t)(0.70710678118654752440 * (double)one);
    // ---- ln u: ends of the range, powers of two, about sqrt(1/2) and 1 ----
    double worst = 0.0;
    auto log_of = [&](uint64_t j) {
        if (j == 0 || j >= one) return;
        const double u = ldexp((double)j, -53);
        const long double want = logl((long double)u);
        worst = std::max(worst, (double)(fabsl((long double)sn::log_unit(u) - want) / ulp((double)want)));
    };
    for (uint64_t j = 1; j < 100000; j++) { log_of(j); log_of(one - j); log_of(root - 50000 + j); }
    for (int e = 0; e <= 53; e++)
        for (int64_t d = -500; d <= 500; d++) log_of((1ull << e) + d);
    for (int i = 0; i < 2000000; i++) { log_of(g() >> 11); log_of(g() >> (11 + g() % 53)); }
    // ---- sqrt of x = 1 - S, S = (a^2 + b^2) 2^-52 ----
    long roots = 0;
    auto root_of = [&](uint64_t j) {   // x = j 2^-52
        const double x = ldexp((double)j, -52);
        if (j > 0 && j <= 1ull << 52) roots += sn::sqrt_unit(x) != sqrt(x);
    };
    for (uint64_t j = 1; j < 300000; j++) { root_of(j); root_of((1ull << 52) - j); root_of((1ull << 52) + 1 - j); }
    for (int i = 0; i < 3000000; i++) root_of(g() >> (12 + (i & 1) * (g() % 52)));
    // ---- the threshold -ln u / beta: the rounded quotient on both sides of its guards ----
    long quotients = 0;
    const double betas[] = {1e-300, 0.9e-200, 1e-200, 1.1e-200, 1e-9, 0.3, 1.0, 300.0 / 299.0, 3.0, 12345.678, 0.99e200, 1e200, 1.01e200, 1e300};
    for (double beta : betas)
        for (int i = 0; i < 100000; i++) {
            const uint64_t j = i < 1000 ? (uint64_t)i + 1 : i < 2000 ? one - 1 - (i - 1000) : std::max<uint64_t>(g() >> 11, 1);
            const double u = ldexp((double)j, -53), l = -sn::log_unit(u);
            quotients += sn::metropolis_threshold(u, beta, 1.0 / beta) != l / beta;
        }
    const bool limits = sn::metropolis_threshold(0.0, 1.0, 1.0) == INFINITY &&
                        sn::metropolis_threshold(0.5, 0.0, INFINITY) == INFINITY &&
                        sn::metropolis_threshold(0.5, INFINITY, 0.0) == 0.0;
    printf("%.4f %ld %ld %d\n", worst, roots, quotients, (int)limits);
}
