// dst_passes.h -- the FP64 DST passes of one level, compiled per transform
// length M = 2 n (n cells, N = n - 1 unknowns): kernels over arrays of EllJob.
//
// A solve of all levels is
//   pass 1, every level: rows of the right-hand side -> DST along j -> T.  No
//           boundary values enter here, so levels do not wait for each other.
//   then, coarsest level first:
//     pass 2: column pairs of T, plus the boundary values' share (EllJob::bcv)
//             -> DST along i -> 1 / eigenvalue -> DST along i -> T in place
//     bc:     from T, the values the next finer level's getBC reads, as that
//             level's bcv
//   pass 3, every level: rows of T -> DST along j -> u
// so that only pass 2 and bc are serial in the level; passes 1 and 3 of a
// small batch, whose launches are a few microseconds of latency each, run as
// one launch over all levels.
//
// The boundary terms of getRHS (EllipticSolver2d.cc:125-144) in the space of
// pass 2, where a row i holds modes l of DST-I along j: the terms at j = 1 and
// j = ny - 1 of row i have the transform 2 sin(pi l / ny) (bottom_i +
// (-1)^(l+1) top_i), the terms at i = 1 and i = nx - 1 that of left and right.
//
// A transform is a Stockham FFT of the odd extension, two rows or columns as
// real and imaginary part: the first stage's inputs come straight from
// memory (pass 2 and bc: from LDS), stages exchange through LDS, the last hands
// its outputs on.
//
// What bounds them: on one flow of 200^2 to 512^2 a launch is its workgroups'
// latency (a dependent chain of descriptor, rows, transform, store; about half
// of it outside the transform), so lanes are spent on shortening it: M / 4
// threads, two per butterfly of a radix near 8, so that loads and outputs are
// spread wider.  Against M / 8: a 200^2 step 244 instead of 273 us, 400^2 x 4
// levels 1.11 instead of 1.17 ms; 16 flows of 400^2 x 4, where lanes count, 2%
// slower (4.3 ms).  Every length is compiled with its own radices: a plan read
// at run time spent most of a 128^2 level's 24 us on index division, against
// 13 us here.
//
// On a cylinder at 400^2 x 4 levels a solve takes, in us per launch, one pass 1
// and one pass 3 over all levels (8.9 and 6.9), four pass 2 (7.7) and three bc
// (6.2), 16 us less than twelve passes level by level (7.4, 7.8, 5.6).
#pragma once
#include "dst_dev.h"

namespace ibpmg {

struct Radices {
    int n;
    int r[8];
};

constexpr int dst_threads(int M) { return M / 4 <= 64 ? 64 : (M / 4 + 63) / 64 * 64; }

// Weight of one butterfly of radix R in the choice of a length's radices, in
// instructions with its twiddles.  The weights, and the 90 for a stage's exchange
// (two barriers and an LDS round trip), were counted, not fitted: what was measured
// is the outcome, times by workload and the error by length.  With radices 12, 15,
// 16 and 20 in the set no length takes one.
constexpr int radix_cost(int R) {
    return R == 2 ? 12 : R == 3 ? 28 : R == 4 ? 34 : R == 5 ? 58 : R == 6 ? 70 : R == 8 ? 92 : R == 9 ? 130 : 140;
}

struct RadixSearch {
    int best_cost;
    Radices best;
};
// Every factorisation of rem into descending radices; a stage costs its
// rounds of butterflies over the workgroup plus an exchange.
constexpr void search_radices(int M, int rem, int cap, Radices cur, int cost, RadixSearch& out) {
    if (rem == 1) {
        if (cur.n > 0 && (out.best_cost < 0 || cost < out.best_cost)) {
            out.best_cost = cost;
            out.best = cur;
        }
        return;
    }
    constexpr int set[] = {10, 9, 8, 6, 5, 4, 3, 2};
    if (cur.n == 8) return;
    for (int R : set) {
        if (R > cap || rem % R) continue;
        const int rounds = (M / R + dst_threads(M) - 1) / dst_threads(M);
        Radices next = cur;
        next.r[next.n++] = R;
        search_radices(M, rem / R, R, next, cost + rounds * radix_cost(R) + 90, out);
    }
}
// Descending, except that the last radix is the smallest even one: only half
// of the outputs of an even last stage are needed (k < M / 2).
constexpr Radices radices(int M) {
    RadixSearch s{-1, {0, {1, 1, 1, 1, 1, 1, 1, 1}}};
    search_radices(M, M, 10, Radices{0, {1, 1, 1, 1, 1, 1, 1, 1}}, 0, s);
    Radices q = s.best;
    int last = q.n - 1;
    while (last > 0 && q.r[last] % 2) --last;
    const int R = q.r[last];
    for (int k = last; k + 1 < q.n; ++k) q.r[k] = q.r[k + 1];
    q.r[q.n - 1] = R;
    return q;
}

// A butterfly's twiddles w^r, r < R, of stage s >= 1: products of w^1 alone, whose
// rounding then grows with r (w^7 carries seven times that of w^1), or of the
// loaded w^1, w^2, w^4, w^8.  Loading costs more than the products: everywhere, the
// flux at 1000 x 600 x 5 levels takes 212 instead of 188 us, ten steps at 400^2 x 4
// 10.7 instead of 10.0 ms.  So it is done only where the products leave a larger
// error than radices 8, 4, 2, 5, 3 from rounded angles had: in transforms of two
// stages, whose one twiddled stage is half of the work (6 to 36 cells), and at
// radices 9 and 10.  Error relative to those at 6, 8, 12, 15, 20, 25, 32, 36, 125,
// 225, 324, 405 cells: 1.16, 1.24, 1.06, 1.08, 1.09, 1.28, 1.08, 1.04, 1.04, 1.04,
// 1.05, 1.13 from w^1 alone; now 0.95, 0.91, 0.86, 0.73, 0.76, 0.68, 0.67, 0.73,
// 0.76, 0.74, 0.89, 0.68, and no length above 1.
constexpr int twiddle_loads(const Radices& q, int s) {
    if (q.n != 2 && q.r[s] <= 8) return 1;
    int n = 0;
    for (int p = 1; p < q.r[s]; p *= 2) ++n;
    return n;
}
// w[1..R-1] from the N loaded powers.
template <int R, int N>
__host__ __device__ __forceinline__ void twiddle_powers(const double2* loaded, double2* w) {
#pragma unroll
    for (int p = 0; p < N; ++p) w[1 << p] = loaded[p];
#pragma unroll
    for (int r = 2; r < R; ++r) {
        const int h = N == 1 ? r - r / 2 : r < 4 ? 2 : r < 8 ? 4 : 8;   // else the highest loaded power
        if (r != h) w[r] = cmul(w[r - h], w[h]);
    }
}

// FFT of length M in a workgroup of BT threads; element e of a stage is LDS slot
// e + e / R1 (a pad after every R1 elements where R1 is even, so that the first
// stage's writes, R1 apart, spread over the banks).
template <int M, int BT>
struct LdsFft {
    static constexpr Radices Q = radices(M);
    static constexpr int R1 = Q.r[0], PAD = (Q.n > 1 && R1 % 2 == 0) ? 1 : 0;
    static constexpr int kSlots = Q.n > 1 ? M + M / R1 * PAD : 1;
    static constexpr int ns(int s) {
        int p = 1;
        for (int k = 0; k < s; ++k) p *= Q.r[k];
        return p;
    }
    static constexpr int rounds(int s) { return (M / Q.r[s] + BT - 1) / BT; }
    static constexpr int loads(int s) { return twiddle_loads(Q, s); }
    static constexpr int first_tw(int s) {
        int p = 0;
        for (int k = 1; k < s; ++k) p += rounds(k) * loads(k);
        return p;
    }
    static constexpr int kTw = first_tw(Q.n);
    // the loaded powers of w^(jm M / (Ns R)) of every butterfly this thread takes in stages 1..
    double2 tw[kTw > 0 ? kTw : 1];

    template <int S = 1>
    __device__ __forceinline__ void load_twiddles(const IBPM_GLOBAL double* g) {
        if constexpr (S < Q.n) {
            constexpr int Ns = ns(S), R = Q.r[S], step = M / (Ns * R), n = loads(S), at = first_tw(S);
#pragma unroll
            for (int b = 0; b < rounds(S); ++b) {
                const int j = (int)(threadIdx.x + b * BT) % (M / R);
                const int k = j % Ns * step;
#pragma unroll
                for (int p = 0; p < n; ++p)
                    tw[at + b * n + p] = make_double2(g[2 * (k << p)], g[2 * (k << p) + 1]);
            }
            load_twiddles<S + 1>(g);
        }
    }

    // Stage S: v[b][r] is set (stage 0 by load, later stages from LDS).
    template <int S, bool WAIT, class Emit>
    __device__ __forceinline__ void stages(double2* lds, const Emit& emit) {
        constexpr int R = Q.r[S], MR = M / R, n = loads(S), at = first_tw(S);
        double2 v[rounds(S)][R];
#pragma unroll
        for (int b = 0; b < rounds(S); ++b) {
            const int j = threadIdx.x + b * BT;
            if (j >= MR) continue;
            const double2* in = lds + j + j / R1 * PAD;
            constexpr int step = MR + MR / R1 * PAD;   // MR is a multiple of R1 from stage 1 on
            double2 w[R];
            twiddle_powers<R, n>(tw + at + b * n, w);
            v[b][0] = in[0];
#pragma unroll
            for (int r = 1; r < R; ++r) v[b][r] = cmul(in[r * step], w[r]);
            dft_any<R>(v[b]);
        }
        out<S, WAIT>(v, lds, emit);
    }

    template <int S, bool WAIT, class Emit>
    __device__ __forceinline__ void out(double2 (&v)[rounds(S)][Q.r[S]], double2* lds, const Emit& emit) {
        constexpr int R = Q.r[S], MR = M / R, Ns = ns(S);
        if constexpr (S + 1 == Q.n) {   // k = j + r Ns: the half that a DST-I needs
            if constexpr (WAIT) __syncthreads();
#pragma unroll
            for (int b = 0; b < rounds(S); ++b) {
                const int j = threadIdx.x + b * BT;
                if (j >= MR) continue;
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (r * Ns < M / 2) {
                        const int k = j + r * Ns;
                        if (k > 0 && k < M / 2) emit(k, b * R + r, v[b][r]);
                    }
            }
        } else {
            if constexpr (S > 0) __syncthreads();   // the stage's inputs are read
#pragma unroll
            for (int b = 0; b < rounds(S); ++b) {
                const int j = threadIdx.x + b * BT;
                if (j >= MR) continue;
                double2* o;
                int step;
                if constexpr (S == 0) {
                    o = lds + j * (R1 + PAD);
                    step = 1;
                } else {   // Ns is a multiple of R1
                    const int jm = j % Ns, d = j / Ns * (Ns * R) + jm;
                    o = lds + d + d / R1 * PAD;
                    step = Ns + Ns / R1 * PAD;
                }
#pragma unroll
                for (int r = 0; r < R; ++r) o[r * step] = v[b][r];
            }
            __syncthreads();
            stages<S + 1, WAIT>(lds, emit);
        }
    }

    // load(e): z[e] (called for a valid e by every thread, so its reads are
    // under no branch); emit(k, slot, Z[k]) for 0 < k < M / 2.
    // WAIT: a barrier before emit, which may then write the LDS buffer.  The
    // caller puts a barrier between two runs over one buffer.
    template <bool WAIT, class Load, class Emit>
    __device__ __forceinline__ void run(double2* lds, const Load& load, const Emit& emit) {
        constexpr int R = Q.r[0], MR = M / R;
        double2 v[rounds(0)][R];
#pragma unroll
        for (int b = 0; b < rounds(0); ++b) {
            const int j = min((int)threadIdx.x + b * BT, MR - 1);
#pragma unroll
            for (int r = 0; r < R; ++r) v[b][r] = load(j + r * MR);
        }
#pragma unroll
        for (int b = 0; b < rounds(0); ++b) dft_any<R>(v[b]);
        out<0, WAIT>(v, lds, emit);
    }

    // emit's slots: values g[k - 1] of this thread's outputs k, read ahead of
    // the transform so that emit waits on nothing.
    static constexpr int kEmit = rounds(Q.n - 1) * Q.r[Q.n - 1];
    __device__ __forceinline__ void preload(const IBPM_GLOBAL double* g, double* x) {
        constexpr int S = Q.n - 1, R = Q.r[S], MR = M / R, Ns = ns(S);
#pragma unroll
        for (int b = 0; b < rounds(S); ++b) {
            const int j = min((int)threadIdx.x + b * BT, MR - 1);
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r * Ns < M / 2) x[b * R + r] = g[min(max(j + r * Ns, 1), M / 2 - 1) - 1];
        }
    }
};

// Element e of the odd extension: index (0-based unknown) and sign (0 at e = 0, M / 2).
struct Ext {
    int idx;
    double sign;
};
template <int M>
__device__ __forceinline__ Ext ext_at(int e) {
    const bool hi = e > M / 2, zero = e == 0 || e == M / 2;
    return Ext{zero ? 0 : (hi ? M - e - 1 : e - 1), zero ? 0.0 : (hi ? -1.0 : 1.0)};
}

// A kernel of one pass and length; workgroups in xcd_block order.
#define IBPM_DST_KERNEL(NAME, BT)                                                   \
    template <int M>                                                                 \
    __global__ void __launch_bounds__(BT) NAME(const EllJob* __restrict__ jobs)

// ---------------------------------------------------------------- pass 1
// One row pair per workgroup; rows off the right-hand side's support
// [sup_lo, sup_hi] are left out (pass 2 takes them as 0).
IBPM_DST_KERNEL(k_dst_pass1, dst_threads(M)) {
    constexpr int BT = dst_threads(M), N2 = M / 2 - 1;
    typedef LdsFft<M, BT> F;
    __shared__ double2 lds[F::kSlots];
    const int2 blk = xcd_block();
    const EllJob& J = jobs[blk.y];
    if (skipped(J.skip)) return;
    const int N1 = J.nx - 1, ra = 2 * blk.x;
    if (ra >= N1 || ra + 1 > J.sup_hi || ra + 2 < J.sup_lo) return;
    const bool hb = ra + 1 < N1;
    const int rb = hb ? ra + 1 : ra;
    const int ex = nx_ext(J.nx), ey = nx_ext(J.ny), jc1 = J.ny / 2 + ey;
    const bool ca = J.lev >= 1 && ra + 1 > ex && ra + 1 < J.nx / 2 + ex;
    const bool cb = J.lev >= 1 && rb + 1 > ex && rb + 1 < J.nx / 2 + ex;
    const bool ina = ra + 1 >= J.rb_i0 && ra + 1 <= J.rb_i1, inb = rb + 1 >= J.rb_i0 && rb + 1 <= J.rb_i1;
    const IBPM_GLOBAL double *fa = gin(J.f) + (long)ra * N2, *fb = gin(J.f) + (long)rb * N2;
    const IBPM_GLOBAL double *Ra = gin(J.R) + (long)ra * N2, *Rb = gin(J.R) + (long)rb * N2;
    const int rj0 = J.rb_j0, rj1 = J.rb_j1;
    const double sc = J.in_scale, scb = hb ? sc : 0.0;
    F f;
    IBPM_GLOBAL double* oa = gout(J.T1) + (long)ra * J.ld1;
    IBPM_GLOBAL double* ob = oa + J.ld1;
    if ((N2 & 1) && threadIdx.x == 0) {   // the pad column that pass 2's last pair reads
        oa[N2] = 0.0;
        if (hb) ob[N2] = 0.0;
    }
    bool first = true;
    f.template run<false>(lds, [&](int e) {
        const Ext x = ext_at<M>(e);
        const int j = x.idx + 1;
        // R in the central region of a coarse level (0 off its box, where the
        // boxed coarsify chain left other solves' values), else f
        const bool colc = j > ey && j < jc1, colr = j >= rj0 && j <= rj1;
        const double la = ((ca && colc) ? Ra : fa)[x.idx], lb = ((cb && colc) ? Rb : fb)[x.idx];
        const double sa = (ca && colc && !(ina && colr)) ? 0.0 : x.sign * sc;
        const double sb = (cb && colc && !(inb && colr)) ? 0.0 : x.sign * scb;
        if (first) {   // the twiddles' loads go out behind the first of the rows'
            f.load_twiddles(gin((const double*)J.pj.tw));
            first = false;
        }
        return make_double2(la * sa, lb * sb);
    }, [&](int k, int, double2 z) {
        oa[k - 1] = -z.y;
        if (hb) ob[k - 1] = z.x;
    });
}

// ---------------------------------------------------------------- pass 2
// One column pair per workgroup, in place.  (Two pairs, 32-byte pieces, measured
// the same on batches of 400^2 to 1000^2 levels and slower on one flow: 8.2
// against 7.7 us at 400^2.)
// BOTH: of a Helmholtz solve u = A^-1 f and the Poisson solve L^-1(s u) of its
// result on the same level, from the one forward transform: u's rows to T1,
// the other's to T1b (EllJob::T1b).
template <int M, bool BOTH>
__device__ __forceinline__ void dst_pass2(const EllJob& J, int bx, double2* lds, double2* y) {
    constexpr int BT = dst_threads(M), N1 = M / 2 - 1;
    typedef LdsFft<M, BT> F;
    const int N2 = J.ny - 1, la = 2 * bx;
    if (la >= N2) return;
    typedef double Pair __attribute__((ext_vector_type(2)));
    const long ld = J.ld1;
    IBPM_GLOBAL double* T = gout(J.T1);
    const IBPM_GLOBAL double* bcv = gin(J.bcv);
    const int lo = J.sup_lo, hi = J.sup_hi;
    // the columns, each row's piece read once, into y[row + 1]
    Pair sn = {0, 0}, left = {0, 0}, right = {0, 0};
    if (J.bcv) {
        const IBPM_GLOBAL double* side = bcv + 2 * t1_ld(N1) + la;
        sn = *(const IBPM_GLOBAL Pair*)(gin(J.pj.sin1) + la);
        left = *(const IBPM_GLOBAL Pair*)side;
        right = *(const IBPM_GLOBAL Pair*)(side + ld);
    }
    constexpr int kIn = (N1 + BT - 1) / BT;
    Pair t[kIn], bt[kIn];
#pragma unroll
    for (int b = 0; b < kIn; ++b) {
        const int idx = min((int)threadIdx.x + b * BT, N1 - 1);
        const int row = min(max(idx + 1, lo), hi) - 1;   // rows off the support hold nothing
        t[b] = *(const IBPM_GLOBAL Pair*)(T + row * ld + la);
        bt[b] = J.bcv ? *(const IBPM_GLOBAL Pair*)(bcv + 2 * idx) : Pair{0, 0};   // c (bottom + top), c (bottom - top)
    }
    F f;
    f.load_twiddles(gin((const double*)J.pi.tw));
    double cx[F::kEmit];   // read with the rows, used between the transforms
    f.preload(gin(J.pi.cosn), cx);
    const double ca = gin(J.pj.cosn)[la], cb = gin(J.pj.cosn)[min(la + 1, N2 - 1)];
    const int kind = J.kind, t2_lo = J.t2_lo, t2_hi = J.t2_hi;
    const double bydx2 = J.bydx2, alpha = J.alpha;
#pragma unroll
    for (int b = 0; b < kIn; ++b) {
        const int idx = threadIdx.x + b * BT;
        if (idx >= N1) continue;
        const bool in = idx + 1 >= lo && idx + 1 <= hi;
        double2 v = make_double2(in ? t[b].x : 0.0, in ? t[b].y : 0.0);
        v.x -= sn.x * bt[b].x + (idx == 0 ? left.x : 0.0) + (idx == N1 - 1 ? right.x : 0.0);
        v.y -= sn.y * bt[b].y + (idx == 0 ? left.y : 0.0) + (idx == N1 - 1 ? right.y : 0.0);
        y[idx + 1] = v;
    }
    __syncthreads();
    IBPM_GLOBAL double* Tb = BOTH ? gout(J.T1b) : T;
    const double sb = BOTH ? J.scale_b : 0.0;
    // all transforms by one copy of the code: what bounds a small launch is
    // the time a workgroup takes, its instruction fetch among it
#pragma unroll 1
    for (int it = 0; it < (BOTH ? 3 : 2); ++it) {
        f.template run<F::Q.n == 1>(lds, [&](int e) {
            const Ext x = ext_at<M>(e);
            const double2 v = y[x.idx + 1];
            return make_double2(v.x * x.sign, v.y * x.sign);
        }, [&](int k, int slot, double2 z) {
            if (it == 0 && kind != 2) {
                // spectral scaling, EllipticSolver2d.cc:42-54 (eigenvalues), :89-93 (scale)
                const double l1 = 2. * (cx[slot] + ca - 2.) * bydx2, l2 = 2. * (cx[slot] + cb - 2.) * bydx2;
                const double d1 = kind == 0 ? l1 : 1 + alpha * l1, d2 = kind == 0 ? l2 : 1 + alpha * l2;
                y[k] = make_double2(-z.y * (1. / d1), z.x * (1. / d2));
            } else if (kind == 2) {   // forward transform alone: rows of N2 values to u (ibpm_dst2d)
                gout(J.u)[(long)(k - 1) * N2 + la] = -z.y;
                if (la + 1 < N2) gout(J.u)[(long)(k - 1) * N2 + la + 1] = z.x;
            } else if (k - 1 >= t2_lo && k - 1 <= t2_hi) {   // rows outside are not read
                *(IBPM_GLOBAL Pair*)((it == 1 ? T : Tb) + (k - 1) * ld + la) = Pair{-z.y, z.x};
            }
            if (BOTH && it == 1) {   // (every thread has read y: the transform's barriers lie between)
                const double l1 = 2. * (cx[slot] + ca - 2.) * bydx2, l2 = 2. * (cx[slot] + cb - 2.) * bydx2;
                y[k] = make_double2(sb * y[k].x * (1. / l1), sb * y[k].y * (1. / l2));
            }
        });
        if (kind == 2) return;
        __syncthreads();
    }
}

#define IBPM_DST_PASS2(NAME, BOTH)                                                      \
    IBPM_DST_KERNEL(NAME, dst_threads(M)) {                                             \
        __shared__ double2 lds[LdsFft<M, dst_threads(M)>::kSlots], y[M / 2];            \
        const int2 blk = xcd_block();                                                   \
        const EllJob& J = jobs[blk.y];                                                  \
        if (skipped(J.skip)) return;                                                    \
        dst_pass2<M, BOTH>(J, blk.x, lds, y);                                           \
    }
IBPM_DST_PASS2(k_dst_pass2, false)
IBPM_DST_PASS2(k_dst_pass2_both, true)

// ---------------------------------------------------------------- pass 3
IBPM_DST_KERNEL(k_dst_pass3, dst_threads(M)) {
    constexpr int BT = dst_threads(M), N2 = M / 2 - 1;
    typedef LdsFft<M, BT> F;
    __shared__ double2 lds[F::kSlots];
    const int2 blk = xcd_block();
    const EllJob& J = jobs[blk.y];
    if (skipped(J.skip)) return;
    const int N1 = J.nx - 1, ra = 2 * blk.x;
    if (ra >= N1 || blk.x < J.full_lo || blk.x > J.full_hi) return;
    const bool hb = ra + 1 < N1;
    const IBPM_GLOBAL double* ta = gin(J.T1) + (long)ra * J.ld1;
    const IBPM_GLOBAL double* tb = hb ? ta + J.ld1 : ta;
    const long o = (long)ra * N2;
    const double norm = J.norm;
    F f;
    bool first = true;
    double wa[F::kEmit], wb[F::kEmit];
    f.template run<false>(lds, [&](int e) {
        const Ext x = ext_at<M>(e);
        const double a = ta[x.idx], b = tb[x.idx];
        if (first) {
            f.load_twiddles(gin((const double*)J.pj.tw));
            if (J.epilogue) {
                f.preload(gin(J.W) + o, wa);
                f.preload(gin(J.W) + (hb ? o + N2 : o), wb);
            }
            first = false;
        }
        return make_double2(a * x.sign, b * x.sign);
    }, [&](int k, int slot, double2 z) {
        // sinTransformInv normalisation, EllipticSolver2d.cc:80-83
        const double va = -z.y * norm, vb = z.x * norm;
        const double ua = J.epilogue ? wa[slot] - va : va, ub = J.epilogue ? wb[slot] - vb : vb;
        gout(J.u)[o + k - 1] = ua;
        if (hb) gout(J.u)[o + N2 + k - 1] = ub;
    });
}

// ------------------------------------------------------------ bc (getBC)
// From T after pass 2 of a level lev >= 1: the next finer level's bcv
// (Scalar.cc:91-127; layout in EllJob), which the fine level's pass 2
// subtracts.  Workgroup 0: left and right, u along the two ring rows (the
// inverse transform of their pair), refined to the fine spacing, transformed
// again.  The others: bottom and top, u at the two ring columns of the rows
// between, direct sums over the row's modes, kBcRows coarse rows a wave (each
// also needs the next: 5 rows read for 4).  With explicit boundary values (bcring, one level) both come from those.
constexpr int kBcRows = 4;
IBPM_DST_KERNEL(k_dst_bc, dst_threads(M)) {
    constexpr int BT = dst_threads(M), N2 = M / 2 - 1;
    typedef LdsFft<M, BT> F;
    const EllJob& J = jobs[blockIdx.y];
    const bool given = J.bcring != nullptr;
    if (!J.bc_out || skipped(J.skip)) return;
    const int nx = J.nx, ny = J.ny, ex = nx_ext(nx), ey = nx_ext(ny);
    const double c = J.bc_out_coef, norm = J.norm;
    IBPM_GLOBAL double* out = gout(J.bc_out);
    typedef double Pair __attribute__((ext_vector_type(2)));
    if (blockIdx.x > 0) {
        if (given) {
            const int i = (blockIdx.x - 1) * BT + threadIdx.x + 1;
            if (i >= nx) return;
            const double b = c * bc_bottom(J, i), t = c * bc_top(J, i);
            *(IBPM_GLOBAL Pair*)(out + 2 * (i - 1)) = Pair{b + t, b - t};
            return;
        }
        const int m0 = ((blockIdx.x - 1) * (BT / 64) + threadIdx.x / 64) * kBcRows, lane = threadIdx.x % 64;
        if (m0 >= nx / 2) return;
        // u(ex + m, .) at the two columns for m = m0 .. m0 + kBcRows (past nx / 2: that row again)
        const IBPM_GLOBAL double* r = gin(J.T1) + (long)(ex - 1 + m0) * J.ld1;
        const IBPM_GLOBAL double* s = gin(J.pj.ring);
        double b[kBcRows + 1], t[kBcRows + 1];
#pragma unroll
        for (int q = 0; q <= kBcRows; ++q) b[q] = t[q] = 0.0;
#pragma unroll 2
        for (int l = lane; l < N2; l += 64) {
            const double sb = s[l], st = s[N2 + l];
#pragma unroll
            for (int q = 0; q <= kBcRows; ++q) {
                const double x = r[(long)min(q, nx / 2 - m0) * J.ld1 + l];
                b[q] += x * sb;
                t[q] += x * st;
            }
        }
#pragma unroll
        for (int q = 0; q <= kBcRows; ++q)
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                b[q] += __shfl_xor(b[q], off, 64);
                t[q] += __shfl_xor(t[q], off, 64);
            }
        if (lane != 0) return;
        const double cn = c * norm;
#pragma unroll
        for (int q = 0; q < kBcRows; ++q) {   // fine i = 2 m (none for m = 0) and, halfway to the next row, 2 m + 1
            const int m = m0 + q;
            if (m >= nx / 2) break;
            const double bh = 0.5 * (b[q] + b[q + 1]), th = 0.5 * (t[q] + t[q + 1]);
            if (m > 0) *(IBPM_GLOBAL Pair*)(out + 2 * (2 * m - 1)) = Pair{cn * (b[q] + t[q]), cn * (b[q] - t[q])};
            *(IBPM_GLOBAL Pair*)(out + 2 * (2 * m)) = Pair{cn * (bh + th), cn * (bh - th)};
        }
        return;
    }
    __shared__ double2 lds[F::kSlots], y[M / 2];
    F f;
    f.load_twiddles(gin((const double*)J.pj.tw));
    const int o1 = 2 * t1_ld(nx - 1), ld = J.ld1;
    if (given) {
        for (int j = threadIdx.x + 1; j < ny; j += BT) y[j] = make_double2(bc_left(J, j), bc_right(J, j));
    } else {
        const IBPM_GLOBAL double* ta = gin(J.T1) + (long)(ex - 1) * J.ld1;
        const IBPM_GLOBAL double* tb = ta + (long)(nx / 2) * J.ld1;
        for (int j = threadIdx.x + 1; j < ny; j += BT) y[j] = make_double2(ta[j - 1] * norm, tb[j - 1] * norm);
    }
    __syncthreads();
    // inverse transform of the two rows, then forward of the refined values,
    // by one copy of the code (the given values need the second alone)
#pragma unroll 1
    for (int it = given ? 1 : 0; it < 2; ++it) {
        const bool refine = it == 1 && !given;
        f.template run<F::Q.n == 1>(lds, [&](int e) {
            const Ext x = ext_at<M>(e);
            const int j = x.idx + 1, a = refine ? j / 2 + ey : j, b = refine ? a + (j & 1) : j;
            const double h = 0.5 * x.sign;
            return make_double2((y[a].x + y[b].x) * h, (y[a].y + y[b].y) * h);
        }, [&](int k, int, double2 z) {
            if (it == 0) {
                y[k] = make_double2(-z.y, z.x);
            } else {
                out[o1 + k - 1] = -z.y * c;
                out[o1 + ld + k - 1] = z.x * c;
            }
        });
        __syncthreads();
    }
    if ((N2 & 1) && threadIdx.x == 0) out[o1 + N2] = out[o1 + ld + N2] = 0.0;
}

// ------------------------------------------------------------------ host
// Launches of one pass (4: bc, 5: pass 2 of two solves) over jobs of one length
// (none without jobs); false for a length that is not among the instantiated
// ones (dst_f64.hip).
struct DstLaunch {
    int M, pass, blocks, njobs;
    const EllJob* jobs;
    hipStream_t s;
};

template <int M>
inline void launch_dst_len(const DstLaunch& L) {
    const dim3 grid(L.blocks, L.njobs);
    switch (L.pass) {
    case 1: hipLaunchKernelGGL(k_dst_pass1<M>, grid, dim3(dst_threads(M)), 0, L.s, L.jobs); break;
    case 2: hipLaunchKernelGGL(k_dst_pass2<M>, grid, dim3(dst_threads(M)), 0, L.s, L.jobs); break;
    case 3: hipLaunchKernelGGL(k_dst_pass3<M>, grid, dim3(dst_threads(M)), 0, L.s, L.jobs); break;
    case 5: hipLaunchKernelGGL(k_dst_pass2_both<M>, grid, dim3(dst_threads(M)), 0, L.s, L.jobs); break;
    default: hipLaunchKernelGGL(k_dst_bc<M>, grid, dim3(dst_threads(M)), 0, L.s, L.jobs); break;
    }
}

}  // namespace ibpmg
