// dst_dev.h -- device pieces shared by the DST passes: complex arithmetic and the
// small DFTs (for the host too, where their error is measured), getBC / getRHS at
// a point, and the workgroup order.
#pragma once
#include "ops.h"

namespace ibpmg {

__host__ __device__ inline double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__host__ __device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__host__ __device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
// -i * a
__host__ __device__ inline double2 cmi(double2 a) { return make_double2(a.y, -a.x); }
// The same for the FP32 transforms (float2).
__host__ __device__ inline float2 cmul(float2 a, float2 b) {
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__host__ __device__ inline float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__host__ __device__ inline float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__host__ __device__ inline float2 cmi(float2 a) { return make_float2(a.y, -a.x); }

// Real type of a complex type, and a complex value from two reals.
template <class C> struct RealOf;
template <> struct RealOf<double2> { typedef double T; };
template <> struct RealOf<float2> { typedef float T; };
template <class C>
__host__ __device__ inline C cpx(typename RealOf<C>::T x, typename RealOf<C>::T y) {
    C r;
    r.x = x;
    r.y = y;
    return r;
}

typedef double DoublePair __attribute__((ext_vector_type(2), aligned(8)));

// Radix-R DFT in place (R = 2, 3, 4, 5, 8), FP64 (double2) or FP32 (float2):
// the same operations in the same order for both, constants rounded to the
// type.
template <int R, class C>
__host__ __device__ inline void dft(C* v) {
    typedef typename RealOf<C>::T T;
    if constexpr (R == 2) {
        C a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else if constexpr (R == 3) {
        const T h = T(0.86602540378443864676);   // sin(2 pi / 3)
        C t1 = cadd(v[1], v[2]);
        C t2 = csub(v[1], v[2]);
        C m = cpx<C>(v[0].x - T(0.5) * t1.x, v[0].y - T(0.5) * t1.y);
        C r = cmi(t2);
        v[0] = cadd(v[0], t1);
        v[1] = cpx<C>(m.x + h * r.x, m.y + h * r.y);
        v[2] = cpx<C>(m.x - h * r.x, m.y - h * r.y);
    } else if constexpr (R == 4) {
        C s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
        C s13 = cadd(v[1], v[3]), d13 = cmi(csub(v[1], v[3]));
        v[0] = cadd(s02, s13);
        v[1] = cadd(d02, d13);
        v[2] = csub(s02, s13);
        v[3] = csub(d02, d13);
    } else if constexpr (R == 5) {
        const T c1 = T(0.30901699437494742410);    // cos(2 pi / 5)
        const T c2 = T(-0.80901699437494742410);   // cos(4 pi / 5)
        const T s1 = T(0.95105651629515357212);    // sin(2 pi / 5)
        const T s2 = T(0.58778525229247312917);    // sin(4 pi / 5)
        C t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
        C t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
        C a1 = cpx<C>(v[0].x + c1 * t1.x + c2 * t2.x, v[0].y + c1 * t1.y + c2 * t2.y);
        C a2 = cpx<C>(v[0].x + c2 * t1.x + c1 * t2.x, v[0].y + c2 * t1.y + c1 * t2.y);
        C b1 = cpx<C>(s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y);
        C b2 = cpx<C>(s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y);
        b1 = cmi(b1);   // -i b1
        b2 = cmi(b2);
        v[0] = cadd(v[0], cadd(t1, t2));
        v[1] = cadd(a1, b1);
        v[4] = csub(a1, b1);
        v[2] = cadd(a2, b2);
        v[3] = csub(a2, b2);
    } else {
        static_assert(R == 8, "radix 2, 3, 4, 5 or 8");
        // radix 8 = two radix-4 DFTs of the even and odd samples + radix-2 merge
        const T c = T(0.70710678118654752440);
        C a[4] = {v[0], v[2], v[4], v[6]};
        C b[4] = {v[1], v[3], v[5], v[7]};
        dft<4>(a);
        dft<4>(b);
        const C t0 = b[0];
        const C t1 = cpx<C>(c * (b[1].x + b[1].y), c * (b[1].y - b[1].x));    // W8^1 b1
        const C t2 = cpx<C>(b[2].y, -b[2].x);                                // W8^2 b2 = -i b2
        const C t3 = cpx<C>(c * (b[3].y - b[3].x), -c * (b[3].x + b[3].y));   // W8^3 b3
        v[0] = cadd(a[0], t0); v[4] = csub(a[0], t0);
        v[1] = cadd(a[1], t1); v[5] = csub(a[1], t1);
        v[2] = cadd(a[2], t2); v[6] = csub(a[2], t2);
        v[3] = cadd(a[3], t3); v[7] = csub(a[3], t3);
    }
}

// 16-point DFT as 4 x 4: X[k1 + 4 k2] = sum_n2 W16^(n2 k1) W4^(n2 k2)
// sum_n1 x[4 n1 + n2] W4^(n1 k1).
__host__ __device__ inline double2 mul_w16(double2 a, int k) {   // a * exp(-2 pi i k / 16), k in {1,2,3,6,9}
    const double c1 = 0.92387953251128675613;   // cos(pi / 8)
    const double s1 = 0.38268343236508977173;   // sin(pi / 8)
    const double h = 0.70710678118654752440;    // cos(pi / 4)
    switch (k) {
    case 1: return make_double2(c1 * a.x + s1 * a.y, c1 * a.y - s1 * a.x);
    case 2: return make_double2(h * (a.x + a.y), h * (a.y - a.x));
    case 3: return make_double2(s1 * a.x + c1 * a.y, s1 * a.y - c1 * a.x);
    case 6: return make_double2(h * (a.y - a.x), -h * (a.x + a.y));
    default: return make_double2(-c1 * a.x - s1 * a.y, s1 * a.x - c1 * a.y);   // 9
    }
}

__host__ __device__ inline void dft16(double2* v) {
    double2 a[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
        double2 c[4] = {v[n2], v[n2 + 4], v[n2 + 8], v[n2 + 12]};
        dft<4>(c);
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) a[n2][k1] = c[k1];
    }
    a[1][1] = mul_w16(a[1][1], 1); a[1][2] = mul_w16(a[1][2], 2); a[1][3] = mul_w16(a[1][3], 3);
    a[2][1] = mul_w16(a[2][1], 2); a[2][2] = cmi(a[2][2]);        a[2][3] = mul_w16(a[2][3], 6);
    a[3][1] = mul_w16(a[3][1], 3); a[3][2] = mul_w16(a[3][2], 6); a[3][3] = mul_w16(a[3][3], 9);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        double2 c[4] = {a[0][k1], a[1][k1], a[2][k1], a[3][k1]};
        dft<4>(c);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = c[k2];
    }
}

// R1 R2-point DFT, R1 and R2 coprime, as an R1 x R2 one without twiddles (the
// Good-Thomas index maps): X[k] = Y[k mod R1][k mod R2], Y the 2-D DFT of
// x[(R2 n1 + R1 n2) mod R].
template <int R1, int R2>
__host__ __device__ inline void dft_pfa(double2* v) {
    constexpr int R = R1 * R2;
    double2 a[R1][R2];
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) {
#pragma unroll
        for (int n2 = 0; n2 < R2; ++n2) a[n1][n2] = v[(R2 * n1 + R1 * n2) % R];
        dft<R2>(a[n1]);
    }
#pragma unroll
    for (int k2 = 0; k2 < R2; ++k2) {
        double2 c[R1];
#pragma unroll
        for (int n1 = 0; n1 < R1; ++n1) c[n1] = a[n1][k2];
        dft<R1>(c);
#pragma unroll
        for (int n1 = 0; n1 < R1; ++n1) a[n1][k2] = c[n1];
    }
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = a[k % R1][k % R2];
}

// 9-point DFT as 3 x 3, twiddles exp(-2 pi i {1, 2, 4} / 9).
__host__ __device__ inline void dft9(double2* v) {
    const double c1 = 0.76604444311897803520, s1 = 0.64278760968653932632;   // 2 pi / 9
    const double c2 = 0.17364817766693034885, s2 = 0.98480775301220805937;   // 4 pi / 9
    const double c4 = -0.93969262078590838405, s4 = 0.34202014332566873304;  // 8 pi / 9
    double2 a[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < 3; ++n1) a[n2][n1] = v[3 * n1 + n2];
        dft<3>(a[n2]);
    }
    a[1][1] = cmul(a[1][1], make_double2(c1, -s1));
    a[1][2] = cmul(a[1][2], make_double2(c2, -s2));
    a[2][1] = cmul(a[2][1], make_double2(c2, -s2));
    a[2][2] = cmul(a[2][2], make_double2(c4, -s4));
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
        double2 c[3] = {a[0][k1], a[1][k1], a[2][k1]};
        dft<3>(c);
#pragma unroll
        for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = c[k2];
    }
}

// DFT of any radix of the compiled FP64 passes.
template <int R>
__host__ __device__ inline void dft_any(double2* v) {
    if constexpr (R == 6) dft_pfa<2, 3>(v);
    else if constexpr (R == 9) dft9(v);
    else if constexpr (R == 10) dft_pfa<2, 5>(v);
    else dft<R>(v);
}

// The scratch rows T as the transform's real type: FP64, or
// FP32 in the FP32 passes (the same buffers, half of each used).
template <class T>
__device__ inline const IBPM_GLOBAL T* tin(const double* p) { return (const IBPM_GLOBAL T*)p; }
template <class T>
__device__ inline IBPM_GLOBAL T* tout(double* p) { return (IBPM_GLOBAL T*)p; }


// Logical (row block, job) of this workgroup.  Workgroups are handed to the
// 8 XCDs round-robin in launch order, so logical neighbours are mapped to the
// same XCD: consecutive workgroups of pass 2 read and write neighbouring pieces
// of the same cache lines, and those pieces then meet in one XCD's L2 instead
// of being fetched by, and written back partially from, several.
__device__ inline int2 xcd_block() {
    constexpr int X = 8;
    const int gx = gridDim.x, total = gx * gridDim.y;
    const int flat = blockIdx.x + blockIdx.y * gx;
    const int xcd = flat % X, idx = flat / X, q = total / X, r = total % X;
    const int lf = (xcd < r) ? xcd * (q + 1) + idx : r * (q + 1) + (xcd - r) * q + idx;
    return make_int2(lf % gx, lf / gx);
}

// getBC (reference Scalar.cc:91-127) evaluated at one boundary index.
// (Global-address-space reads: a flat load would also count against the LDS
// counter, and the barrier after the right-hand side would wait for it.)
__device__ inline double bc_bottom(const EllJob& J, int i) {
    if (J.bcring) return i == 0 ? gin(J.bcring)[0] : gin(J.bcring)[2 * (J.nx + J.ny) - i];
    const int ii = i / 2 + nx_ext(J.nx), jj = nx_ext(J.ny);
    const double a = gin(J.uc)[sidx(J.nx, J.ny, ii, jj)];
    return (i & 1) ? 0.5 * (a + gin(J.uc)[sidx(J.nx, J.ny, ii + 1, jj)]) : a;
}
__device__ inline double bc_top(const EllJob& J, int i) {
    if (J.bcring) return gin(J.bcring)[J.ny + i];
    const int ii = i / 2 + nx_ext(J.nx), jj = J.ny / 2 + nx_ext(J.ny);
    const double a = gin(J.uc)[sidx(J.nx, J.ny, ii, jj)];
    return (i & 1) ? 0.5 * (a + gin(J.uc)[sidx(J.nx, J.ny, ii + 1, jj)]) : a;
}
__device__ inline double bc_left(const EllJob& J, int j) {
    if (J.bcring) return gin(J.bcring)[j];
    const int ii = nx_ext(J.nx), jj = j / 2 + nx_ext(J.ny);
    const double a = gin(J.uc)[sidx(J.nx, J.ny, ii, jj)];
    return (j & 1) ? 0.5 * (a + gin(J.uc)[sidx(J.nx, J.ny, ii, jj + 1)]) : a;
}
__device__ inline double bc_right(const EllJob& J, int j) {
    if (J.bcring) return gin(J.bcring)[2 * J.ny + J.nx - j];
    const int ii = J.nx / 2 + nx_ext(J.nx), jj = j / 2 + nx_ext(J.ny);
    const double a = gin(J.uc)[sidx(J.nx, J.ny, ii, jj)];
    return (j & 1) ? 0.5 * (a + gin(J.uc)[sidx(J.nx, J.ny, ii, jj + 1)]) : a;
}

// Right-hand side of one level at (i, j), 1-based: coarsified copy in the
// central region of levels >= 1 (EllipticSolver.cc:54-55), then getRHS
// (EllipticSolver2d.cc:125-144 / 166-185).
__device__ inline double rhs_value(const EllJob& J, int i, int j) {
    const int ex = nx_ext(J.nx), ey = nx_ext(J.ny);
    const bool central = J.lev >= 1 && i > ex && i < J.nx / 2 + ex && j > ey && j < J.ny / 2 + ey;
    const long k = sidx(J.nx, J.ny, i, j);
    double v = (central ? gin(J.R)[k] : gin(J.f)[k]) * J.in_scale;
    if (J.uc || J.bcring) {
        const double c = J.bc_coef;
        if (j == 1) v -= bc_bottom(J, i) * c;
        if (j == J.ny - 1) v -= bc_top(J, i) * c;
        if (i == 1) v -= bc_left(J, j) * c;
        if (i == J.nx - 1) v -= bc_right(J, j) * c;
    }
    return v;
}

// Points of a coarse level (lev >= 1) that getBC of the next finer level
// reads: the rectangle i = ex..ex+nx/2, j = ey..ey+ny/2 traced by the finer
// domain's boundary (Scalar.cc:91-127).
__device__ inline bool on_bc_ring(const EllJob& J, int i, int j) {
    const int ex = nx_ext(J.nx), ey = nx_ext(J.ny);
    const int i1 = ex + J.nx / 2, j1 = ey + J.ny / 2;
    return ((j == ey || j == j1) && i >= ex && i <= i1) || ((i == ex || i == i1) && j >= ey && j <= j1);
}

}  // namespace ibpmg
