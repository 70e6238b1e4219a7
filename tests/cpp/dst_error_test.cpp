// Error of one transform per compiled length, with the radices, small DFTs,
// twiddle powers and tables of the FP64 passes, against extended precision: no
// larger than that of radices 8, 4, 2, 5, 3 with twiddles from angles rounded to
// double and every power from w^1 (the transform before the passes were compiled
// per length).  Host code only, compiled to fuse multiply-adds as the device does.
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "dst_passes.h"
#include "dst_tables.h"

using namespace ibpmg;
typedef long double LD;
typedef std::vector<double2> Row;

template <int R, int N>
static void butterfly_of(const double2* loaded, bool twiddled, double2* v) {
    if (twiddled) {
        double2 w[R];
        twiddle_powers<R, N>(loaded, w);
        for (int r = 1; r < R; ++r) v[r] = cmul(v[r], w[r]);
    }
    dft_any<R>(v);
}
template <int R>
static void butterfly(const double2* loaded, int n, bool twiddled, double2* v) {
    if (!twiddled || n == 1) butterfly_of<R, 1>(loaded, twiddled, v);
    else if (R == 2) butterfly_of<R, 1>(loaded, twiddled, v);
    else if (R <= 4) butterfly_of<R, (R <= 4 ? 2 : 3)>(loaded, twiddled, v);
    else if (R <= 8) butterfly_of<R, 3>(loaded, twiddled, v);
    else butterfly_of<R, 4>(loaded, twiddled, v);
}

static bool stage(int R, const double2* loaded, int n, bool twiddled, double2* v) {
    switch (R) {
    case 2: butterfly<2>(loaded, n, twiddled, v); return true;
    case 3: butterfly<3>(loaded, n, twiddled, v); return true;
    case 4: butterfly<4>(loaded, n, twiddled, v); return true;
    case 5: butterfly<5>(loaded, n, twiddled, v); return true;
    case 6: butterfly<6>(loaded, n, twiddled, v); return true;
    case 8: butterfly<8>(loaded, n, twiddled, v); return true;
    case 9: butterfly<9>(loaded, n, twiddled, v); return true;
    case 10: butterfly<10>(loaded, n, twiddled, v); return true;
    default: return false;
    }
}

static bool fft(Row& z, const double2* tw, const Radices& q, bool from_first) {
    const int M = (int)z.size();
    Row o(M);
    for (int s = 0, Ns = 1; s < q.n; Ns *= q.r[s++]) {
        const int R = q.r[s], MR = M / R, step = M / (Ns * R), n = from_first ? 1 : twiddle_loads(q, s);
        for (int j = 0; j < MR; ++j) {
            double2 v[16], loaded[4];
            for (int r = 0; r < R; ++r) v[r] = z[j + r * MR];
            for (int p = 0; p < n && (1 << p) < R; ++p) loaded[p] = tw[j % Ns * step << p];
            if (!stage(R, loaded, n, s > 0, v)) return false;
            for (int r = 0; r < R; ++r) o[j / Ns * Ns * R + j % Ns + r * Ns] = v[r];
        }
        z.swap(o);
    }
    return true;
}

// z's transform (odd, purely) in extended precision: -2 i times the sine sums
static void exact(const Row& z, std::vector<LD>& x, std::vector<LD>& y) {
    const int M = (int)z.size(), n = M / 2;
    std::vector<LD> sn(M);
    const LD pi = 4 * std::atan(1.0L);
    for (int k = 0; k < M; ++k) sn[k] = std::sin(2 * pi * k / M);
    x.assign(n, 0);
    y.assign(n, 0);
    for (int k = 1; k < n; ++k)
        for (int e = 1; e < n; ++e) {   // sum z exp(-i t) = -2 i sum z sin t
            const LD t = 2 * sn[(long)k * e % M];
            x[k] += z[e].y * t;
            y[k] -= z[e].x * t;
        }
}

int main() {
    int bad = 0;
    for (int n = 2; n <= 1024; ++n) {
        int m = n;
        for (int p : {2, 3, 5})
            while (m % p == 0) m /= p;
        if (m != 1) continue;
        const int M = 2 * n, rows = std::max(8, 30000 / n);   // (60000 values: 1% of sampling)
        const Radices q = radices(M);
        Radices plain{0, {1, 1, 1, 1, 1, 1, 1, 1}};
        m = M;
        for (int r : {8, 4, 2, 5, 3})
            for (; m % r == 0; m /= r) plain.r[plain.n++] = r;
        std::vector<double> tw(2 * M);
        twiddle_table(M, tw.data());
        Row angles(M);
        for (int k = 0; k < M; ++k) {
            const double a = -8.0 * std::atan(1.0) * (double)k / (double)M;
            angles[k] = make_double2(std::cos(a), std::sin(a));
        }
        double here = 0, before = 0;
        std::mt19937_64 g(M);
        std::normal_distribution<double> nd;
        for (int row = 0; row < rows; ++row) {
            Row z(M, make_double2(0, 0));
            for (int k = 1; k < n; ++k) {
                z[k] = make_double2(nd(g), nd(g));
                z[M - k] = make_double2(-z[k].x, -z[k].y);
            }
            std::vector<LD> x, y;
            exact(z, x, y);
            Row a = z, b = z;
            if (!fft(a, (const double2*)tw.data(), q, false) || !fft(b, angles.data(), plain, true)) {
                std::printf("n = %d: a radix without a butterfly\n", n);
                return 1;
            }
            for (int k = 1; k < n; ++k) {
                here += (double)((a[k].x - x[k]) * (a[k].x - x[k]) + (a[k].y - y[k]) * (a[k].y - y[k]));
                before += (double)((b[k].x - x[k]) * (b[k].x - x[k]) + (b[k].y - y[k]) * (b[k].y - y[k]));
            }
        }
        const bool worse = here > before;
        bad += worse;
        if (worse) std::printf("n = %d: error %.3f times that before\n", n, std::sqrt(here / before));
    }
    std::printf("%d lengths with a larger error\n", bad);
    return bad != 0;
}
