// dst_tables.h -- host values of a transform plan's tables (FftPlan).
#pragma once
#include <cmath>
#include <cstddef>

#include "common.h"

namespace ibpmg {

// Doubles of the real tables cosn, sin1 (t1_ld(N) each) and ring (2 N).
inline size_t plan_reals(int N) { return 2 * (size_t)t1_ld(N) + 2 * (size_t)N; }

// Whether a plan of FFT length M has the second-stage table tw16.
inline bool plan_has_tw16(int M) { return M == 1024 || M == 2048; }

// exp(-2 pi i k / M), k < M (M even), as pairs into tw, each part rounded from extended
// precision.  (cos and sin of an angle rounded to double are off by up to its
// error, 1e-15 near 2 pi, which was most of a transform's error.)  An eighth of
// them (a quarter where 4 does not divide M) are evaluated, the others mirrored.
inline void twiddle_table(int M, double* tw) {
    const long double twopi = 8.0L * std::atan(1.0L);
    auto put = [&](int k, double c, double s) {   // cos and sin of 2 pi k / M, mirrored into every quadrant
        const int h = M / 2;
        auto set = [&](int q, double x, double y) { tw[2 * (q % M)] = x; tw[2 * (q % M) + 1] = y; };
        set(k, c, 0.0 - s);   // (no negative zeros)
        set(h - k, 0.0 - c, 0.0 - s);
        set(h + k, 0.0 - c, s);
        set(M - k, c, s);
    };
    const int last = M % 4 == 0 ? M / 8 : M / 4;
    for (int k = last; k >= 1; --k) {
        const long double a = twopi * k / M;
        const double c = (double)std::cos(a), s = (double)std::sin(a);
        put(k, c, s);
        if (M % 4 == 0) put(M / 4 - k, s, c);
    }
    if (M % 4 == 0) put(M / 4, 0.0, 1.0);
    put(0, 1.0, 0.0);
}

// tw (M pairs), t16 (256 pairs, where plan_has_tw16) and the real tables one
// after another, whose angles pi l e / n are whole multiples of 2 pi / M and so
// taken from tw: the argument itself goes up to 800, where a sine of the rounded
// one is off by 1e-13.
inline void plan_tables(int M, double* tw, double* t16, double* reals) {
    twiddle_table(M, tw);
    if (plan_has_tw16(M)) {
        const int tstep = M / 256;
        for (int r = 0; r < 16; ++r)
            for (int jm = 0; jm < 16; ++jm)
                for (int h = 0; h < 2; ++h) t16[2 * (16 * r + jm) + h] = tw[2 * ((tstep * jm * r) % M) + h];
    }
    const int n = M / 2, N = n - 1, e = nx_ext(n);
    double *cosn = reals, *sin1 = cosn + t1_ld(N), *ring = sin1 + t1_ld(N);
    for (int i = N; i < t1_ld(N); ++i) cosn[i] = sin1[i] = 0.0;
    for (int i = 1; i < n; ++i) {
        cosn[i - 1] = tw[2 * i];   // EllipticSolver2d.cc:47-48
        sin1[i - 1] = -2. * tw[2 * i + 1];
        ring[i - 1] = -2. * tw[2 * (int)((long)i * e % M) + 1];
        ring[N + i - 1] = -2. * tw[2 * (int)((long)i * (e + n / 2) % M) + 1];
    }
}

}  // namespace ibpmg
