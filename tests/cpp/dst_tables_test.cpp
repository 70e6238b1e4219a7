// The tables of every transform plan (dst_tables.h) against extended precision:
// each value within half a unit in the last place.  Host code only.
#include <cstdio>
#include <vector>

#include "dst_tables.h"

using namespace ibpmg;
typedef long double LD;

// The reference's own angle, up to 2 pi, is off by three roundings of 2^-62, which the
// doubled sines double: 2e-18 of slack on half a unit.
static double worst = 0;
static void check(const char* what, int n, int k, double got, LD want) {
    const double off = (double)std::fabs((LD)got - want);
    const double half = want == 0 ? 0 : std::ldexp(0.5, std::ilogb((double)want) - 52);
    if (off > half + 2e-18) std::printf("n = %d: %s[%d] off by %.1e, half a unit is %.1e\n", n, what, k, off, half);
    worst = std::max(worst, off - half);
}

int main() {
    const LD pi = 4 * std::atan(1.0L);
    int plans = 0;
    for (int n = 2; n <= 1024; ++n) {
        int m = n;
        for (int p : {2, 3, 5})
            while (m % p == 0) m /= p;
        if (m != 1) continue;
        ++plans;
        const int M = 2 * n, N = n - 1, e = nx_ext(n);
        std::vector<double> tw(2 * M), t16(512), re(plan_reals(N));
        plan_tables(M, tw.data(), t16.data(), re.data());
        const double *cosn = re.data(), *sin1 = cosn + t1_ld(N), *ring = sin1 + t1_ld(N);
        auto ang = [&](long k) { return 2 * pi * (LD)(k % M) / M; };
        for (int k = 0; k < M; ++k) {
            check("re w", n, k, tw[2 * k], std::cos(ang(k)));
            check("im w", n, k, tw[2 * k + 1], -std::sin(ang(k)));
        }
        if (plan_has_tw16(M))
            for (int r = 0; r < 16; ++r)
                for (int j = 0; j < 16; ++j) check("t16", n, 16 * r + j, t16[2 * (16 * r + j)], std::cos(ang((long)M / 256 * j * r)));
        for (int i = 1; i < n; ++i) {
            check("cosn", n, i, cosn[i - 1], std::cos(ang(i)));
            check("sin1", n, i, sin1[i - 1], 2 * std::sin(ang(i)));
            check("ring", n, i, ring[i - 1], 2 * std::sin(ang((long)i * e)));
            check("ring", n, i, ring[N + i - 1], 2 * std::sin(ang((long)i * (e + n / 2))));
        }
        for (int i = N; i < t1_ld(N); ++i) check("pad", n, i, cosn[i] + sin1[i], 0);
    }
    std::printf("%d plans, at most %.1e past half a unit\n", plans, worst);
    return !(worst <= 2e-18 && plans == 86);
}
