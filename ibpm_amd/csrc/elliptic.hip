// elliptic.hip -- batched multi-domain DST-I Poisson/Helmholtz solves.
//
// Replaces EllipticSolver2d::solve (reference EllipticSolver2d.cc:57-185) and
// the multi-domain driver EllipticSolver::solve (EllipticSolver.cc:47-73).
//
// One level solve u = S diag(e) S f * norm (S = DST-I matrix) is three passes,
// each reading and writing the level once (6 words per grid point):
//   pass 1: rows of the right-hand side (coarsify select and sign fused in) ->
//           DST along j -> rows of T
//   pass 2: columns of T, two neighbouring ones a pair, plus the boundary values'
//           share (getRHS) -> DST along i -> eigenvalue scaling -> DST along i ->
//           the same columns of T
//   pass 3: rows of T -> DST along j -> * 1/(4 nx ny) -> u (or u = W - .)
// T keeps the level's (i, j) layout throughout, so passes 1 and 3 read and
// write whole rows and pass 2 works in place.
// Each DST-I of length N is the imaginary part of a complex FFT of length
// M = 2(N+1) of the odd extension; two rows share one FFT (real part row a,
// imaginary part row b).  The FP64 passes are compiled per length in
// dst_passes.h, through LDS; here are those of M = 1024 and 2048 as a radix
// 16 x 16 x M/256 transform held in registers (exchanges through LDS), and the FP32
// passes: a mixed-radix (2, 3, 4, 5, 8) Stockham transform held in LDS, each
// stage staged through registers so that one buffer suffices, with lengths that
// have no compiled plan read from a plan at run time, and the boundary values in
// pass 1, level by level.  Passes may run over part of a level when only part of
// the result is read (EllJob's partial-pass fields; not the FP32 ones).  The file
// also holds the coarsify chain and the local Jacobi solves of the force solve's
// A^-1 (k_fs_helm).
#include "dst_passes.h"

#include <algorithm>

namespace ibpmg {

// FFT lengths whose FP32 passes have a compiled plan (M = 2(N+1) for N = 199, 255,
// 383, 399, 511, 1023: the configured grids); any other length uses the runtime
// plan.
__host__ __device__ constexpr bool compiled_len(int M) {
    return M == 400 || M == 512 || M == 768 || M == 800 || M == 1024 || M == 2048;
}

// Twiddle w^k = exp(-2 pi i k / M), k < M.  The longest compiled length
// keeps only the first quarter in LDS, w^(q M/4 + r) = (-i)^q w^r, which
// halves its LDS footprint and doubles the workgroups per CU; shorter
// lengths are not LDS-limited and read the full table.
__host__ __device__ constexpr bool quarter_twiddles(int M) { return M >= 2048 && M % 4 == 0; }

template <int CM, class C>
__device__ inline C twiddle(const C* tw, int k) {
    if constexpr (CM != 0 && quarter_twiddles(CM)) {
        typedef typename RealOf<C>::T T;
        constexpr int Q = CM / 4;
        const int q = k / Q, r = k - q * Q;
        const C t = tw[r];
        T x = t.x, y = t.y;
        if (q & 1) {   // times -i
            const T u = x;
            x = y;
            y = -u;
        }
        if (q & 2) {   // times -1
            x = -x;
            y = -y;
        }
        return cpx<C>(x, y);
    } else {
        return tw[k];
    }
}

// LDS slot of element e when the buffer is held swizzled: the low 3 bits
// are XORed with bits 3..5.  This permutes each aligned group of 8 complex
// values (128 B, one sweep of the 32 banks; compiled lengths are multiples
// of 8), so 8 lanes whose elements share their low 3 bits -- the first
// stage's radix-R writes, R apart -- land on distinct banks, while contiguous
// runs stay conflict-free.  Only the layout between the first and second
// stage is swizzled (the first stage's writes were the conflicting ones).
template <bool SW>
__device__ inline int lds_slot(int e) {
    if constexpr (SW) return e ^ ((e >> 3) & 7);
    else return e;
}

// The 2048-point transforms (largest grids, bandwidth-bound batches) keep the
// whole buffer swizzled, which measured faster there; the shorter compiled
// lengths swizzle only between the first two stages.
template <int CM>
constexpr bool kSwizzleAll = CM >= 2048;

// One Stockham radix-R stage over np FFTs of length M stored back to back in
// LDS; inputs are staged through registers so the stage runs in place.
// Twiddles come from the LDS table (see twiddle()).  Template
// arguments that are 0 are taken from the runtime values.
template <int R, int CM, int CNP, int CNS, bool SWIN, bool SWOUT, class C>
__device__ inline void fft_stage(C* buf, const C* tw, int Mr, int npr, int Nsr) {
    const int M = CM ? CM : Mr;
    const int np = CM ? CNP : npr;
    const int Ns = CM ? CNS : Nsr;
    constexpr int MAXB = CM ? (CNP * CM / R + kFftThreads - 1) / kFftThreads
                            : (kFftLds / R + kFftThreads - 1) / kFftThreads;
    const int MR = M / R;
    const int total = np * MR;
    const int tstep = M / (Ns * R);
    C v[MAXB][R];
#pragma unroll
    for (int b = 0; b < MAXB; ++b) {
        const int g = threadIdx.x + b * kFftThreads;
        if (g < total) {
            const int p = g / MR;
            const int j = g - p * MR;
            const int jm = j % Ns;
            const int x = p * M;
            v[b][0] = buf[lds_slot<SWIN>(x + j)];
            if constexpr (CM != 0 && CNS == 1) {
#pragma unroll
                for (int r = 1; r < R; ++r) v[b][r] = buf[lds_slot<SWIN>(x + j + r * MR)];
            } else {
                // w^r by binary splitting, w^r = w^(r/2) w^(r - r/2): at most
                // 3 dependent products for R <= 8
                C pw[R];
                pw[1] = twiddle<CM>(tw, jm * tstep);
#pragma unroll
                for (int r = 2; r < R; ++r) pw[r] = cmul(pw[r / 2], pw[r - r / 2]);
#pragma unroll
                for (int r = 1; r < R; ++r) v[b][r] = cmul(buf[lds_slot<SWIN>(x + j + r * MR)], pw[r]);
            }
            dft<R>(v[b]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < MAXB; ++b) {
        const int g = threadIdx.x + b * kFftThreads;
        if (g < total) {
            const int p = g / MR;
            const int j = g - p * MR;
            const int jm = j % Ns;
            const int d = p * M + (j / Ns) * Ns * R + jm;
#pragma unroll
            for (int r = 0; r < R; ++r) buf[lds_slot<SWOUT>(d + r * Ns)] = v[b][r];
        }
    }
    __syncthreads();
}

__host__ __device__ constexpr int pick_radix(int rem) {
    return rem % 8 == 0 ? 8 : rem % 4 == 0 ? 4 : rem % 2 == 0 ? 2 : rem % 5 == 0 ? 5 : 3;
}

// Compile-time stage list: radix 8 first, then 4, 2, 5, 3.
template <int M, int NP, int Ns, class C>
__device__ inline void fft_ct(C* buf, const C* tw) {
    if constexpr (Ns < M) {
        constexpr int R = pick_radix(M / Ns);
        constexpr bool first = Ns == 1, second = Ns > 1 && Ns == pick_radix(M);
        constexpr bool all = kSwizzleAll<M>;
        fft_stage<R, M, NP, Ns, all || second, all || (first && R < M), C>(buf, tw, 0, 0, 0);
        fft_ct<M, NP, Ns * R, C>(buf, tw);
    }
}

// Runtime stage list of a host-built plan (any 2(N+1) with factors 2,3,5).
template <class C>
__device__ inline void fft_rt(C* buf, const C* tw, const FftPlan& P) {
    int Ns = 1;
    for (int s = 0; s < P.nst; ++s) {
        const int R = P.rad[s];
        switch (R) {
        case 8: fft_stage<8, 0, 0, 0, false, false, C>(buf, tw, P.M, P.np, Ns); break;
        case 4: fft_stage<4, 0, 0, 0, false, false, C>(buf, tw, P.M, P.np, Ns); break;
        case 2: fft_stage<2, 0, 0, 0, false, false, C>(buf, tw, P.M, P.np, Ns); break;
        case 3: fft_stage<3, 0, 0, 0, false, false, C>(buf, tw, P.M, P.np, Ns); break;
        default: fft_stage<5, 0, 0, 0, false, false, C>(buf, tw, P.M, P.np, Ns); break;
        }
        Ns *= R;
    }
}

__host__ __device__ constexpr int np_of(int M) {
    return kFftLds / M < 1 ? 1 : (kFftLds / M > kFftNpMax ? kFftNpMax : kFftLds / M);
}

template <int CM, class C>
__device__ inline void fft_any(C* buf, const C* tw, const FftPlan& P) {
    if constexpr (CM != 0) fft_ct<CM, np_of(CM), 1, C>(buf, tw);
    else fft_rt<C>(buf, tw, P);
}

// ------------------------------------- 1024- and 2048-point transforms in registers
// The 511- and 1023-point grids (M = 1024, 2048) run one row pair per
// workgroup of T = M/16 threads as three radix stages 16 x 16 x R3 (R3 =
// M/256) held in registers: the first stage's inputs z[t + T r] come straight
// from global memory, the two exchanges between stages go through LDS, and
// the last stage hands Z[t + T m], m < 8 -- the half of the spectrum a DST-I
// needs -- to the caller as it is ready.
// A launch at M = 1024 runs only a quarter wave per CU when it holds few rows
// (one 511-row level: 256 workgroups of one wave), where the LDS passes'
// larger workgroups hide latency better; it takes the register-held
// transform from kRegMinPairs row pairs on.  The pairs are those of one level,
// summed over the flows that share its length, as they were when a launch was
// one level: a small batch's passes 1 and 3 over all levels at once hold more (five
// levels of one 512^2 flow: 1280 pairs) and stay with the LDS passes, as its pass 2
// does.  The line has not been measured again for those launches.  M = 2048
// always takes the register-held transform.
constexpr long kRegMinPairs = 1024;

// Row pairs per workgroup of the register-held passes: pass 2 reads and writes
// 2 G neighbouring columns, 16 G bytes of a row per piece.
#ifndef IBPM_R16_GROUP2
#define IBPM_R16_GROUP2 2
#endif
__host__ __device__ constexpr int r16_group(int pass) { return pass == 2 ? IBPM_R16_GROUP2 : 1; }

// Waves per SIMD asked of the compiler.  Pass 2 at M = 2048 took 130 registers,
// which leaves three waves where its LDS has room for four; held to 128, 16
// tandem flows' levels of 1023 x 1023 take 110 us instead of 116.  The same
// bound made the compiler take 96 for pass 1, 57 us instead of 52.
__host__ __device__ constexpr int r16_waves(int pass) { return pass == 2 ? 4 : 1; }

// LDS slot of element e: one pad slot after every 16, so the first stage's
// writes (16 consecutive elements per lane) spread over the banks, and every
// access of a stage is a per-lane base plus a compile-time offset.  The
// exchanges move real and imaginary parts in two rounds through a buffer of
// M + M/16 doubles, half the footprint of a buffer of complex values, so
// twice as many workgroups share a CU.  r16_buf counts it in complex slots.
__host__ __device__ constexpr int r16_buf(int M) { return (M + M / 16) / 2; }
__device__ inline int pad16(int e) { return e + (e >> 4); }

// A workgroup of G pairs keeps them interleaved: element e of pair g is
// slot pad16(e) G + g, so neighbouring lanes (pair fastest) stay on
// neighbouring banks.
// One exchange: every lane writes its 16 values at wr[k * ws], reads 16 at
// rd[k * rs] (per-lane bases, compile-time strides), real parts then
// imaginary parts.
template <int WS, int RS>
__device__ __forceinline__ void exchange16(double2* v, double* wr, const double* rd) {
#pragma unroll
    for (int r = 0; r < 16; ++r) wr[WS * r] = v[r].x;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r].x = rd[RS * r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) wr[WS * r] = v[r].y;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r].y = rd[RS * r];
    __syncthreads();
}

// Second half of the odd extension from the first: v[r] = z[t + T r] is set
// for r < 8; z[e] = -z[M - e] (another lane's) for e > M/2 comes through LDS,
// z[M/2] = 0.  The buffer is free again on return.
template <int M, int G>
__device__ __forceinline__ void mirror_second_half(double2* v, double2* buf, int t) {
    constexpr int T = M / 16;
#pragma unroll
    for (int r = 0; r < 8; ++r) buf[(t + T * r) * G] = v[r];
    __syncthreads();
#pragma unroll
    for (int r = 8; r < 16; ++r) {
        const int e = t + T * r;
        if (e == M / 2) {
            v[r] = make_double2(0.0, 0.0);
        } else {
            const double2 y = buf[(M - e) * G];
            v[r] = make_double2(-y.x, -y.y);
        }
    }
    __syncthreads();
}

// The whole odd extension from its first half z[e], e < M/2, left in buf by
// the caller: v[r] = z[t + T r], with z[e] = -z[M - e] for e > M/2 and
// z[M/2] = 0.  The buffer is free again on return.
template <int M, int G>
__device__ __forceinline__ void extension_from_lds(double2* v, double2* buf, int t) {
    constexpr int T = M / 16;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = buf[(t + T * r) * G];
#pragma unroll
    for (int r = 8; r < 16; ++r) {
        const int e = t + T * r;
        if (e == M / 2) {
            v[r] = make_double2(0.0, 0.0);
        } else {
            const double2 y = buf[(M - e) * G];
            v[r] = make_double2(-y.x, -y.y);
        }
    }
    __syncthreads();
}

// First half of the odd extension of two rows a, b (b absent: zeros):
// v[r] = (a, b)[e - 1] at e = t + T r, r < 8, and 0 at e = 0.  Row b is read
// from row a when absent and multiplied by 0.  A select of the loaded value
// would be compiled as a branch around the load, and a load under a branch
// gets a wait for every load before it: the row pair's sixteen loads would
// then complete one after another.
template <int M>
__device__ __forceinline__ void load_first_half(double2* v, const IBPM_GLOBAL double* a,
                                                const IBPM_GLOBAL double* b, bool hb) {
    constexpr unsigned T = M / 16;
    const unsigned t = threadIdx.x & (T - 1);
    const IBPM_GLOBAL double* bb = hb ? b : a;
    const double keep = hb ? 1.0 : 0.0;   // a product, not a select: see above
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const unsigned e = t + T * r, k = e == 0 ? 0u : e - 1;
        const double nz = e == 0 ? 0.0 : 1.0;   // e = 0 holds the extension's zero, also a product
        v[r] = make_double2(a[k] * nz, bb[k] * keep * nz);
    }
}

// In: v[r] = z[t + T r], r < 16.  Out: emit(m, Z[t + T m]) for m < 8, called
// as each output is ready (so callers write results without holding all
// eight).  Twiddles, w = exp(-2 pi i / M), come from global memory (cached):
// the second stage's w^(R3 jm r) from the plan's 256-entry table at 16 r + jm,
// so 16 lanes with consecutive jm read consecutive entries; the third
// stage's w^j (j < 256) from the full table.  The buffer is free again on
// return (the last LDS access precedes the last barrier).
template <int M, int G, class Emit>
__device__ __forceinline__ void fft_regs(double2* v, double* bd, int t, const IBPM_GLOBAL double* tw,
                                         const IBPM_GLOBAL double* twg, const Emit& emit) {
    constexpr int T = M / 16, R3 = M / 256, H = 256 / T, RS = 17 * T / 16;
    dft16(v);   // stage 1 (Ns = 1): outputs 16 t + r to slots 17 t + r; reads
                // t + T r from slots pad16(t) + RS r
    exchange16<G, RS * G>(v, bd + 17 * t * G, bd + pad16(t) * G);
    const int jm = t & 15;   // stage 2 (Ns = 16): twiddles w^(R3 jm r) from the table
#pragma unroll
    for (int r = 1; r < 16; ++r) v[r] = cmul(v[r], make_double2(tw[2 * (16 * r + jm)], tw[2 * (16 * r + jm) + 1]));
    dft16(v);
    // outputs (t/16) 256 + jm + 16 r to slots (t/16) 272 + jm + 17 r; stage 3
    // reads j + 256 r (j = t + T h, h < H) = t + T (h + H r), the exchange16
    // read pattern: lane t reads pad16(t) + RS k for k = 0..15
    exchange16<17 * G, RS * G>(v, bd + ((t >> 4) * 272 + jm) * G, bd + pad16(t) * G);
#pragma unroll
    for (int h = 0; h < H; ++h) {   // stage 3 (Ns = 256): butterflies j = t + T h
        const int j = t + T * h;
        double2 u[R3];
#pragma unroll
        for (int r = 0; r < R3; ++r) u[r] = v[h + H * r];
        const double2 w1 = make_double2(twg[2 * j], twg[2 * j + 1]);
        const double2 w2 = cmul(w1, w1), w3 = cmul(w2, w1);
        u[1] = cmul(u[1], w1);
        u[2] = cmul(u[2], w2);
        u[3] = cmul(u[3], w3);
        if constexpr (R3 == 8) {
            const double2 w4 = cmul(w2, w2);
            u[4] = cmul(u[4], w4);
            u[5] = cmul(u[5], cmul(w4, w1));
            u[6] = cmul(u[6], cmul(w4, w2));
            u[7] = cmul(u[7], cmul(w4, w3));
        }
        dft<R3>(u);
#pragma unroll
        for (int r = 0; r < R3 / 2; ++r) emit(h + H * r, u[r]);   // Z[j + 256 r] with j + 256 r < M/2
    }
}

// The FP32 passes are written once over a template length CM (0: runtime
// plan).  Row length N, FFT length M and rows per block follow from the plan,
// so with CM != 0 every index computation folds to constants.
template <int CM, class C>
__device__ inline void load_twiddles(C* tw, const FftPlan& P) {
    typedef typename RealOf<C>::T T;
    const int M = (CM && quarter_twiddles(CM)) ? CM / 4 : (CM ? CM : P.M);
    const IBPM_GLOBAL double* g = gin((const double*)P.tw);
    for (int k = threadIdx.x; k < M; k += kFftThreads) tw[k] = cpx<C>(T(g[2 * k]), T(g[2 * k + 1]));
}

// Instanced over C = float2: FP32 transforms and scratch T, with the right-hand
// side, boundary terms, eigenvalue scaling and output in FP64.
template <int CM, class C>
__device__ __forceinline__ void pass1_lds(const EllJob& J, C* smem, int bx) {
    typedef typename RealOf<C>::T T;
    const FftPlan& P = J.pj;
    const int M = CM ? CM : P.M, np = CM ? np_of(CM) : P.np;
    const int N1 = J.nx - 1, N2 = M / 2 - 1;
    const int rows = 2 * np;
    const int r0 = bx * rows;
    if (r0 >= N1) return;
    C* buf = smem;
    C* tw = smem + np * M;
    load_twiddles<CM>(tw, P);
    const int n = N2 + 1;
    for (int idx = threadIdx.x; idx < np * N2; idx += kFftThreads) {
        const int p = idx / N2, k = idx - p * N2;
        const int ra = r0 + 2 * p, rb = ra + 1;
        const T va = (ra < N1) ? T(rhs_value(J, ra + 1, k + 1)) : T(0);
        const T vb = (rb < N1) ? T(rhs_value(J, rb + 1, k + 1)) : T(0);
        buf[lds_slot<kSwizzleAll<CM>>(p * M + k + 1)] = cpx<C>(va, vb);
        buf[lds_slot<kSwizzleAll<CM>>(p * M + M - 1 - k)] = cpx<C>(-va, -vb);
    }
    for (int p = threadIdx.x; p < np; p += kFftThreads) {
        buf[lds_slot<kSwizzleAll<CM>>(p * M)] = cpx<C>(T(0), T(0));
        buf[lds_slot<kSwizzleAll<CM>>(p * M + n)] = cpx<C>(T(0), T(0));
    }
    __syncthreads();
    fft_any<CM>(buf, tw, P);
    IBPM_GLOBAL T* out = tout<T>(J.T1);
    for (int idx = threadIdx.x; idx < np * n; idx += kFftThreads) {
        const int p = idx / n, k = idx - p * n;   // k = N2: the pad column of an odd N2, read by pass 2's last pair
        const int ra = r0 + 2 * p, rb = ra + 1;
        if (k == N2) {
            if (!(N2 & 1)) continue;
            if (ra < N1) out[(long)ra * J.ld1 + k] = T(0);
            if (rb < N1) out[(long)rb * J.ld1 + k] = T(0);
            continue;
        }
        const C z = buf[lds_slot<kSwizzleAll<CM>>(p * M + k + 1)];
        if (ra < N1) out[(long)ra * J.ld1 + k] = -z.y;
        if (rb < N1) out[(long)rb * J.ld1 + k] = z.x;
    }
}

template <int CM, class C>
__device__ __forceinline__ void pass2_lds(const EllJob& J, C* smem, int bx) {
    typedef typename RealOf<C>::T T;
    typedef T Pair __attribute__((ext_vector_type(2)));
    const FftPlan& P = J.pi;
    const int M = CM ? CM : P.M, np = CM ? np_of(CM) : P.np;
    const int N1 = M / 2 - 1, N2 = J.ny - 1;
    const int rows = 2 * np;
    const int r0 = bx * rows;   // rows are l = 0..N2-1
    if (r0 >= N2) return;
    C* buf = smem;
    C* tw = smem + np * M;
    load_twiddles<CM>(tw, P);
    const int n = N1 + 1;
    for (int idx = threadIdx.x; idx < np * N1; idx += kFftThreads) {
        const int p = idx / N1, k = idx - p * N1;
        const int la = r0 + 2 * p;
        if (la >= N2) continue;   // (a pair past the last column: its buffer is not written out)
        // both columns of the pair at once; the pad column of an odd N2 holds 0 (pass 1)
        const Pair y = *(const IBPM_GLOBAL Pair*)(tin<T>(J.T1) + (long)k * J.ld1 + la);
        buf[lds_slot<kSwizzleAll<CM>>(p * M + k + 1)] = cpx<C>(y.x, y.y);
        buf[lds_slot<kSwizzleAll<CM>>(p * M + M - 1 - k)] = cpx<C>(-y.x, -y.y);
    }
    for (int p = threadIdx.x; p < np; p += kFftThreads) {
        buf[lds_slot<kSwizzleAll<CM>>(p * M)] = cpx<C>(T(0), T(0));
        buf[lds_slot<kSwizzleAll<CM>>(p * M + n)] = cpx<C>(T(0), T(0));
    }
    __syncthreads();
    fft_any<CM>(buf, tw, P);
    // spectral scaling, EllipticSolver2d.cc:42-54 (eigenvalues), :89-93 (scale)
    for (int idx = threadIdx.x; idx < np * N1; idx += kFftThreads) {
        const int p = idx / N1, k = idx - p * N1;
        const int la = r0 + 2 * p, lb = la + 1;
        const C z = buf[lds_slot<kSwizzleAll<CM>>(p * M + k + 1)];
        double ya = -z.y, yb = z.x;
        const double cx = gin(P.cosn)[k];
        if (la < N2) {
            const double lam = 2. * (cx + gin(J.pj.cosn)[la] - 2.) * J.bydx2;
            ya *= (J.kind == 0) ? 1. / lam : 1. / (1 + J.alpha * lam);
        }
        if (lb < N2) {
            const double lam = 2. * (cx + gin(J.pj.cosn)[lb] - 2.) * J.bydx2;
            yb *= (J.kind == 0) ? 1. / lam : 1. / (1 + J.alpha * lam);
        }
        buf[lds_slot<kSwizzleAll<CM>>(p * M + k + 1)] = cpx<C>(T(ya), T(yb));
        buf[lds_slot<kSwizzleAll<CM>>(p * M + M - 1 - k)] = cpx<C>(T(-ya), T(-yb));
    }
    for (int p = threadIdx.x; p < np; p += kFftThreads) {
        buf[lds_slot<kSwizzleAll<CM>>(p * M)] = cpx<C>(T(0), T(0));
        buf[lds_slot<kSwizzleAll<CM>>(p * M + n)] = cpx<C>(T(0), T(0));
    }
    __syncthreads();
    fft_any<CM>(buf, tw, P);
    for (int idx = threadIdx.x; idx < np * N1; idx += kFftThreads) {
        const int p = idx / N1, k = idx - p * N1;
        const int la = r0 + 2 * p;
        if (la >= N2) continue;
        const C z = buf[lds_slot<kSwizzleAll<CM>>(p * M + k + 1)];
        *(IBPM_GLOBAL Pair*)(tout<T>(J.T1) + (long)k * J.ld1 + la) = Pair{-z.y, z.x};   // (pass 3 reads no pad column)
    }
}

template <int CM, class C>
__device__ __forceinline__ void pass3_lds(const EllJob& J, C* smem, int bx) {
    typedef typename RealOf<C>::T T;
    const FftPlan& P = J.pj;
    const int M = CM ? CM : P.M, np = CM ? np_of(CM) : P.np;
    const int N1 = J.nx - 1, N2 = M / 2 - 1;
    const int rows = 2 * np;
    const int r0 = bx * rows;
    if (r0 >= N1) return;
    C* buf = smem;
    C* tw = smem + np * M;
    load_twiddles<CM>(tw, P);
    const int n = N2 + 1;
    for (int idx = threadIdx.x; idx < np * N2; idx += kFftThreads) {
        const int p = idx / N2, k = idx - p * N2;
        const int ra = r0 + 2 * p, rb = ra + 1;
        const T va = (ra < N1) ? tin<T>(J.T1)[(long)ra * J.ld1 + k] : T(0);
        const T vb = (rb < N1) ? tin<T>(J.T1)[(long)rb * J.ld1 + k] : T(0);
        buf[lds_slot<kSwizzleAll<CM>>(p * M + k + 1)] = cpx<C>(va, vb);
        buf[lds_slot<kSwizzleAll<CM>>(p * M + M - 1 - k)] = cpx<C>(-va, -vb);
    }
    for (int p = threadIdx.x; p < np; p += kFftThreads) {
        buf[lds_slot<kSwizzleAll<CM>>(p * M)] = cpx<C>(T(0), T(0));
        buf[lds_slot<kSwizzleAll<CM>>(p * M + n)] = cpx<C>(T(0), T(0));
    }
    __syncthreads();
    fft_any<CM>(buf, tw, P);
    for (int idx = threadIdx.x; idx < np * N2; idx += kFftThreads) {
        const int p = idx / N2, k = idx - p * N2;
        const C z = buf[lds_slot<kSwizzleAll<CM>>(p * M + k + 1)];
        const int ra = r0 + 2 * p, rb = ra + 1;
        // sinTransformInv normalisation, EllipticSolver2d.cc:80-83
        // with the epilogue, the finer level's BCs must come from v itself
        // (EllipticSolver.cc:62-66 solves c = A^-1 c before omega = omega* - c)
        if (ra < N1) {
            const long o = (long)ra * N2 + k;
            const double v = -(double)z.y * J.norm;
            const double uv = J.epilogue ? gin(J.W)[o] - v : v;
            gout(J.u)[o] = uv;
            if (J.vside && on_bc_ring(J, ra + 1, k + 1)) gout(J.vside)[o] = v;
        }
        if (rb < N1) {
            const long o = (long)rb * N2 + k;
            const double v = (double)z.x * J.norm;
            const double uv = J.epilogue ? gin(J.W)[o] - v : v;
            gout(J.u)[o] = uv;
            if (J.vside && on_bc_ring(J, rb + 1, k + 1)) gout(J.vside)[o] = v;
        }
    }
}

// The three passes for M = 1024, 2048 (N = M/2 - 1), the same arithmetic as those
// of dst_passes.h around a register-held transform.  Passes 1 and 3 run one
// row pair per workgroup of T = M/16 threads, pass 2 G = r16_group(2) column
// pairs (see pass2_r16).

template <int M>
__device__ __forceinline__ void pass1_r16(const EllJob& J, double2* smem, int bx) {
    constexpr int T = M / 16;
    const int N1 = J.nx - 1, ra = 2 * bx, rb = ra + 1;
    if (ra >= N1 || ra + 1 > J.sup_hi || rb + 1 < J.sup_lo) return;
    const int t = threadIdx.x;
    const IBPM_GLOBAL double* tw = gin((const double*)J.pj.tw16);
    const IBPM_GLOBAL double* twg = gin((const double*)J.pj.tw);
    const int ey = nx_ext(J.ny), ex = nx_ext(J.nx);
    const int jc0 = ey, jc1 = J.ny / 2 + ey;   // central columns: jc0 < j < jc1
    const double sc = J.in_scale;
    // the first half of the odd extension, e = t + T r (r < 8) at column j = e
    const bool hb = rb < N1;
    const bool cra = J.lev >= 1 && ra + 1 > ex && ra + 1 < J.nx / 2 + ex;
    const bool crb = hb && J.lev >= 1 && rb + 1 > ex && rb + 1 < J.nx / 2 + ex;
    const IBPM_GLOBAL double* fa = gin(J.f) + sidx(J.nx, J.ny, ra + 1, 1);
    const IBPM_GLOBAL double* fb = gin(J.f) + sidx(J.nx, J.ny, hb ? rb + 1 : ra + 1, 1);
    const IBPM_GLOBAL double* Ra = gin(J.R) + sidx(J.nx, J.ny, ra + 1, 1);
    const IBPM_GLOBAL double* Rb = gin(J.R) + sidx(J.nx, J.ny, hb ? rb + 1 : ra + 1, 1);
    const double keep = hb ? 1.0 : 0.0;
    const bool ina = ra + 1 >= J.rb_i0 && ra + 1 <= J.rb_i1, inb = rb + 1 >= J.rb_i0 && rb + 1 <= J.rb_i1;
    double2 v[16];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const int e = t + T * r, kk = e == 0 ? 0 : e - 1;
        const bool colc = e > jc0 && e < jc1, colr = e >= J.rb_j0 && e <= J.rb_j1;
        // row b absent: read row a, times 0; e = 0, the extension's zero:
        // times 0; R off its box: times 0 (products, as in load_first_half,
        // so that the sixteen loads are in flight together)
        const double nz = e == 0 ? 0.0 : 1.0;
        const double la = ((cra && colc) ? Ra : fa)[kk], lb = ((crb && colc) ? Rb : fb)[kk];
        const double ma = (cra && colc && !(ina && colr)) ? 0.0 : 1.0;
        const double mb = (crb && colc && !(inb && colr)) ? 0.0 : 1.0;
        v[r] = make_double2(la * sc * nz * ma, lb * sc * keep * nz * mb);
    }
    mirror_second_half<M, 1>(v, smem, t);
    // modes kk = t + T m go to column kk - 1; lane 0's kk = 0 instead clears
    // the pad column N = M/2 - 1 that pass 2's last column pair reads
    IBPM_GLOBAL double* oa = gout(J.T1) + (long)ra * J.ld1;
    IBPM_GLOBAL double* ob = oa + J.ld1;
    fft_regs<M, 1>(v, (double*)smem, t, tw, twg, [&](int m, double2 z) {
        const int kk = t + T * m;
        const int c = kk > 0 ? kk - 1 : M / 2 - 1;
        oa[c] = kk > 0 ? -z.y : 0.0;
        if (hb) ob[c] = kk > 0 ? z.x : 0.0;
    });
}

// Pass 2: a workgroup transforms G neighbouring column pairs, lane (t, g) with
// the pair g fastest, in place.  Lane (t, g) loads rows t + T r of its pair as
// one 16-byte value, the complex number of the odd extension itself, so the G
// lanes of a row read one piece of 16 G bytes.  A lane past the last pair
// transforms the last pair again and writes nothing, so every thread reaches
// every barrier (and the pair's owner writes only after the workgroup's reads).
template <int M>
__device__ __forceinline__ void pass2_r16(const EllJob& J, double2* smem, int bx) {
    constexpr int T = M / 16, G = r16_group(2);
    const int N2 = J.ny - 1, npairs = (N2 + 1) / 2;
    if (G * bx >= npairs) return;
    const int g = threadIdx.x % G, t = threadIdx.x / G;
    const int q = min(G * bx + g, npairs - 1);
    const bool own = G * bx + g < npairs;
    double2* buf = smem + g;
    const IBPM_GLOBAL double* tw = gin((const double*)J.pi.tw16);
    const IBPM_GLOBAL double* twg = gin((const double*)J.pi.tw);
    const IBPM_GLOBAL double* gcx = gin(J.pi.cosn);
    const int la = 2 * q, lb = la + 1;
    const bool hb = lb < N2;
    const long ld = J.ld1;
    typedef double Pair __attribute__((ext_vector_type(2)));
    IBPM_GLOBAL double* col = gout(J.T1) + la;
    const int lo = J.sup_lo, hi = J.sup_hi;
    double2 v[16];
#pragma unroll
    for (int r = 0; r < 8; ++r) {   // rows off the support [lo, hi], and e = 0, hold nothing
        const int e = t + T * r, row = min(max(e, lo), hi);
        const Pair y = *(const IBPM_GLOBAL Pair*)(col + (row - 1) * ld);   // a pad column holds 0 (pass 1)
        v[r] = make_double2(row == e ? y.x : 0.0, row == e ? y.y : 0.0);
    }
    if (J.bcv) {   // the boundary values' share (EllJob::bcv)
        const IBPM_GLOBAL double* bcv = gin(J.bcv);
        const IBPM_GLOBAL double* side = bcv + 2 * t1_ld(M / 2 - 1) + la;
        const Pair sn = *(const IBPM_GLOBAL Pair*)(gin(J.pj.sin1) + la);
        const Pair left = *(const IBPM_GLOBAL Pair*)side, right = *(const IBPM_GLOBAL Pair*)(side + ld);
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int e = t + T * r;
            const Pair bt = *(const IBPM_GLOBAL Pair*)(bcv + 2 * (e == 0 ? 0 : e - 1));
            const double nz = e == 0 ? 0.0 : 1.0;
            v[r].x -= nz * (sn.x * bt.x) + (e == 1 ? left.x : 0.0) + (e == M / 2 - 1 ? right.x : 0.0);
            v[r].y -= nz * (sn.y * bt.y) + (e == 1 ? left.y : 0.0) + (e == M / 2 - 1 ? right.y : 0.0);
        }
    }
    mirror_second_half<M, G>(v, buf, t);
    // spectral scaling, EllipticSolver2d.cc:42-54 (eigenvalues), :89-93 (scale),
    // into the first half of the odd extension for the second transform,
    // kept in the (free) LDS buffer rather than in registers beside the
    // transform's own
    const double cya = gin(J.pj.cosn)[la], cyb = hb ? gin(J.pj.cosn)[lb] : 0.0;
    const bool forward_only = J.kind == 2;   // ibpm_dst2d: rows of N2 values to u
    fft_regs<M, G>(v, (double*)smem + g, t, tw, twg, [&](int m, double2 z) {
        const int kk = t + T * m;
        double ya = 0.0, yb = 0.0;
        if (forward_only) {
            if (kk > 0 && own) {
                gout(J.u)[(long)(kk - 1) * N2 + la] = -z.y;
                if (hb) gout(J.u)[(long)(kk - 1) * N2 + lb] = z.x;
            }
            return;
        }
        if (kk > 0) {
            const double cx = gcx[kk - 1];
            ya = -z.y;
            yb = z.x;
            const double lama = 2. * (cx + cya - 2.) * J.bydx2;
            ya *= (J.kind == 0) ? 1. / lama : 1. / (1 + J.alpha * lama);
            if (hb) {
                const double lamb = 2. * (cx + cyb - 2.) * J.bydx2;
                yb *= (J.kind == 0) ? 1. / lamb : 1. / (1 + J.alpha * lamb);
            }
        }
        buf[kk * G] = make_double2(ya, yb);
    });
    if (forward_only) return;
    extension_from_lds<M, G>(v, buf, t);
    fft_regs<M, G>(v, (double*)smem + g, t, tw, twg, [&](int m, double2 z) {
        const int kk = t + T * m;
        if (kk > 0 && own && kk - 1 >= J.t2_lo && kk - 1 <= J.t2_hi)   // rows outside are not read
            *(IBPM_GLOBAL Pair*)(col + (kk - 1) * ld) = Pair{-z.y, z.x};
    });
}

template <int M>
__device__ __forceinline__ void pass3_r16(const EllJob& J, double2* smem, int bx) {
    constexpr int T = M / 16;
    const int N1 = J.nx - 1, N2 = M / 2 - 1, npairs = (N1 + 1) / 2;
    if (bx >= npairs || bx < J.full_lo || bx > J.full_hi) return;
    double2* buf = smem;
    const IBPM_GLOBAL double* tw = gin((const double*)J.pj.tw16);
    const IBPM_GLOBAL double* twg = gin((const double*)J.pj.tw);
    const int t = threadIdx.x;
    const int ra = 2 * bx, rb = ra + 1;
    const bool hb = rb < N1;
    double2 v[16];
    load_first_half<M>(v, gin(J.T1) + (long)ra * J.ld1, gin(J.T1) + (long)rb * J.ld1, hb);
    mirror_second_half<M, 1>(v, buf, t);
    fft_regs<M, 1>(v, (double*)buf, t, tw, twg, [&](int m, double2 z) {
        const int kk = t + T * m;
        if (kk == 0) return;
        const int k = kk - 1;
        // sinTransformInv normalisation, EllipticSolver2d.cc:80-83
        {
            const long o2 = (long)ra * N2 + k;
            const double val_a = -z.y * J.norm;
            const double ua = J.epilogue ? gin(J.W)[o2] - val_a : val_a;
            gout(J.u)[o2] = ua;
        }
        if (hb) {
            const long o2 = (long)rb * N2 + k;
            const double val_b = z.x * J.norm;
            const double ub = J.epilogue ? gin(J.W)[o2] - val_b : val_b;
            gout(J.u)[o2] = ub;
        }
    });
}

// Register-held passes, one kernel per pass and length (dst_passes.h has the
// other lengths' passes and the launch order).  A job whose flow has finished
// its force solve does nothing (skipped()).
#define IBPM_REG_KERNEL(NAME, BODY, PASS)                                        \
    template <int M>                                                             \
    __global__ void __launch_bounds__(r16_group(PASS) * (M / 16), r16_waves(PASS)) NAME(const EllJob* __restrict__ jobs) { \
        extern __shared__ double2 smem[];                                        \
        const int2 blk = xcd_block();                                            \
        const EllJob& J = jobs[blk.y];                                           \
        if (skipped(J.skip)) return;                                             \
        BODY<M>(J, smem, blk.x);                                                 \
    }
IBPM_REG_KERNEL(k_reg_pass1, pass1_r16, 1)
IBPM_REG_KERNEL(k_reg_pass2, pass2_r16, 2)
IBPM_REG_KERNEL(k_reg_pass3, pass3_r16, 3)

// FP32 instances of the LDS passes (every length, runtime plan for lengths
// without a compiled one): the step's own solves (k32_ell_pass*) and those
// inside the force solve (k32_fs_pass*).
#define IBPM_PASS32_KERNEL(NAME, LDSFN)                                                        \
    template <int CM>                                                                          \
    __global__ void __launch_bounds__(kFftThreads) NAME(const EllJob* __restrict__ jobs) {    \
        extern __shared__ float2 smem32[];                                                     \
        const int2 blk = xcd_block();                                                          \
        const EllJob& J = jobs[blk.y];                                                         \
        if (skipped(J.skip)) return;                                                           \
        LDSFN<CM, float2>(J, smem32, blk.x);                                                   \
    }
IBPM_PASS32_KERNEL(k32_ell_pass1, pass1_lds)
IBPM_PASS32_KERNEL(k32_ell_pass2, pass2_lds)
IBPM_PASS32_KERNEL(k32_ell_pass3, pass3_lds)
IBPM_PASS32_KERNEL(k32_fs_pass1, pass1_lds)
IBPM_PASS32_KERNEL(k32_fs_pass2, pass2_lds)
IBPM_PASS32_KERNEL(k32_fs_pass3, pass3_lds)

// --------------------------------------------------------------- coarsify
// Scalar::coarsify (reference Scalar.cc:46-63) for one level, writing only
// the central region into R; neighbours at level lev-1 come from R where the
// finer level is itself coarsified (central region of a level >= 1) and from
// the original field elsewhere.
// One workgroup per coarse row i of the central region; each thread makes two
// neighbouring points (j, j + 1) from the 3 x 5 fine values they share, with
// the same sums in the same order as Scalar::coarsify.
__device__ inline void coarsify_body(const CoarsifyJob& J) {
    if (skipped(J.skip)) return;
    const int nx = J.nx, ny = J.ny;
    const int ex = nx_ext(nx), ey = nx_ext(ny);
    const int wi = nx / 2 - 1, wj = ny / 2 - 1;
    const int row = blockIdx.x;
    if (row >= wi) return;
    const int i = ex + 1 + row, ii = (i - ex) * 2;   // Grid::c2f
    const int lf = J.lev - 1;
    const long lofs = (long)lf * (nx - 1) * (ny - 1);
    // fine rows ii - 1, ii, ii + 1: base pointers (value at column c is [c]) and
    // whether the row crosses the finer level's own central region
    const IBPM_GLOBAL double* fr[3];
    const IBPM_GLOBAL double* Rr[3];
    bool crow[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int r = ii - 1 + d;
        fr[d] = gin(J.f) + lofs + sidx(nx, ny, r, 1) - 1;
        Rr[d] = gin(J.R) + lofs + sidx(nx, ny, r, 1) - 1;
        crow[d] = lf >= 1 && r > ex && r < nx / 2 + ex;
    }
    IBPM_GLOBAL double* out = gout(J.R) + (long)J.lev * (nx - 1) * (ny - 1) + sidx(nx, ny, i, 1) - 1;
    const int npairs = (wj + 1) / 2;
    for (int q = threadIdx.x; q < npairs; q += blockDim.x) {
        const int j0 = ey + 1 + 2 * q;
        const bool two = j0 + 1 <= ey + wj;
        const int jj = (j0 - ey) * 2;
        double x[3][5];   // fine (ii - 1 + d, jj - 1 + c)
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                const int col = jj - 1 + c;
                if (c >= 3 && !two) {
                    x[d][c] = 0.0;
                    continue;
                }
                const bool central = crow[d] && col > ey && col < ny / 2 + ey;
                x[d][c] = central ? Rr[d][col] : fr[d][col];
            }
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            if (o == 1 && !two) break;
            const int c = 1 + 2 * o;   // centre column of this output
            const double v = 0.25 * x[1][c]
                + 0.125 * (x[2][c] + x[1][c + 1] + x[0][c] + x[1][c - 1])
                + 0.0625 * (x[2][c + 1] + x[2][c - 1] + x[0][c + 1] + x[0][c - 1]);
            out[j0 + o] = v;
        }
    }
}

__global__ void __launch_bounds__(kThreads) k_coarsify(const CoarsifyJob* __restrict__ jobs) {
    coarsify_body(jobs[blockIdx.y]);
}
__global__ void __launch_bounds__(kThreads) k_fs_coarsify(const CoarsifyJob* __restrict__ jobs) {
    coarsify_body(jobs[blockIdx.y]);
}

// ------------------------------------------------- local Helmholtz sweeps
// Jacobi sweeps of A u = r, A = 1 + alpha Lap, over a job's box, for the
// force solve's A^-1.  With |alpha| / dx^2 small the solution decays by a
// factor 4|c| / (1 - 4c) per cell away from the right-hand side, so a box
// around the body's smeared force holds it to rounding and the host chooses
// the sweep count for an error below 1e-18 of the solution; it uses the DST
// solve wherever the box would reach a level's boundary ring.  The first
// sweep starts from u = 0, u is 0 off the box, and the right-hand side is
// rhs_value's without boundary terms, which the box keeps away from.
//
// One launch runs up to kHelmDepth sweeps on tiles of kHelmTile^2 points:
// a workgroup loads its tile with a kHelmDepth-point halo into LDS and
// sweeps there, the valid region shrinking by one point a sweep, then writes
// the tile.  Each point's update is the same arithmetic in the same order as
// a sweep over global memory, so the result does not depend on the blocking.
// Launches alternate between tmp and out so that the last writes out.
//
// Small boxes are bound by latency: a launch's descriptor, one round of loads,
// a barrier per sweep.  So a thread's few points are loaded all at once and
// their right-hand side stays in registers.  Plate at 128^2 x 3 (8 to 11
// sweeps, a box of about 60 by 30 cells): two launches of 12.9 us with 256 threads walking eight
// points each in turn; unrolled, six sweeps a launch, 8.2 us with 256 threads,
// 5.9 with 512, 5.1 with 1024; twelve sweeps, 9.3 with 1024 (11.4 with 512),
// one launch.  16 tandem flows, per step: 698 us before, 273 with six sweeps
// and 512 threads, 306 as it is.
#ifndef IBPM_HELM_DEPTH
#define IBPM_HELM_DEPTH 12
#endif
constexpr int kHelmTile = 32, kHelmDepth = IBPM_HELM_DEPTH, kHelmReg = kHelmTile + 2 * kHelmDepth;
constexpr int kHelmThreads = 1024, kHelmPer = (kHelmReg * kHelmReg + kHelmThreads - 1) / kHelmThreads;
static_assert(kHelmDepth >= 1 && kHelmDepth <= 12, "sweeps per launch: 1..12 (LDS tiles with the halo)");

constexpr int kHelmChainPts = kHelmReg * kHelmReg;   // the sweeps' LDS tiles hold it
int helm_chain_points() { return kHelmChainPts; }

// The coarsify chain of the local solves' right-hand side over each job's
// support: Scalar::coarsify's weights and order (as coarsify_body) with the
// finer level's value taken as 0 in its central region off its support (R
// holds other solves' values there) and from f outside the central region.
// Point p of the support; fineR(fi, fj) is R on the finer level's support.
template <class FineR>
__device__ inline double helm_coarse_value(const HelmJob& J, int i, int j, const FineR& fineR) {
    const int ex = nx_ext(J.nx), ey = nx_ext(J.ny);
    const int ii = (i - ex) * 2, jj = (j - ey) * 2;   // Grid::c2f
    const int lf = J.lev - 1;
    auto fine = [&](int fi, int fj) {
        const bool central = lf >= 1 && fi > ex && fi < J.nx / 2 + ex && fj > ey && fj < J.ny / 2 + ey;
        if (!central) return gin(J.f_fine)[sidx(J.nx, J.ny, fi, fj)];
        const bool sup = fi >= J.fs0 && fi <= J.fs1 && fj >= J.ft0 && fj <= J.ft1;
        return sup ? fineR(fi, fj) : 0.0;
    };
    double x[3][3];   // fine (ii - 1 + d, jj - 1 + c)
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int c = 0; c < 3; ++c) x[d][c] = fine(ii - 1 + d, jj - 1 + c);
    return 0.25 * x[1][1] + 0.125 * (x[2][1] + x[1][2] + x[0][1] + x[1][0])
        + 0.0625 * (x[2][2] + x[2][0] + x[0][2] + x[0][0]);
}

// One level of it in a launch over the whole support.
__global__ void __launch_bounds__(kThreads) k_fs_helm_coarsify(const HelmJob* __restrict__ jobs, int lev) {
    const HelmJob& J = jobs[blockIdx.y];
    if (J.lev != lev || skipped(J.skip)) return;
    const int w = J.t1 - J.t0 + 1, h = J.s1 - J.s0 + 1;
    const int p = blockIdx.x * kThreads + threadIdx.x;
    if (w <= 0 || h <= 0 || p >= w * h) return;
    const int i = J.s0 + p / w, j = J.t0 + p % w;
    const double v = helm_coarse_value(J, i, j, [&](int fi, int fj) {
        return gin(J.R_fine)[sidx(J.nx, J.ny, fi, fj)];
    });
    gout(J.R)[sidx(J.nx, J.ny, i, j)] = v;
}

// Where every level's support fits a workgroup's LDS (kHelmChainPts), one
// workgroup runs the chain itself, a level's R going to the next through LDS:
// inside k_fs_helm for its own right-hand side, and in one launch
// (k_fs_chain) for the L^-1 solve's.  A launch per level costs 3.9 us however
// small its support is; the whole second chain takes 3.9 us at 128^2 x 3, and
// 9.9 at 512^2 x 5 where four launches took 4.9 each.  Level J's R into cur, row by row of its support.
__device__ inline void helm_chain_level(const HelmJob& J, const double* prev, double* cur) {
    const int w = J.t1 - J.t0 + 1, h = J.s1 - J.s0 + 1, fw = J.ft1 - J.ft0 + 1;
    if (w > 0 && h > 0)
        for (int p = threadIdx.x; p < w * h; p += blockDim.x)
            cur[p] = helm_coarse_value(J, J.s0 + p / w, J.t0 + p % w, [&](int fi, int fj) {
                return prev[(fi - J.fs0) * fw + (fj - J.ft0)];
            });
    __syncthreads();
}

// CHAIN: the coarse levels' right-hand sides come from the chain run here
// (jobs hold a flow's levels one after another, level 0 first).
template <bool CHAIN>
__global__ void __launch_bounds__(kHelmThreads) k_fs_helm(const HelmJob* __restrict__ jobs, int sweep0, int nsw,
                                                          bool to_out) {
    const HelmJob& J = jobs[blockIdx.y];
    if (skipped(J.skip)) return;
    const int i0 = J.i0, i1 = J.i1, j0 = J.j0, j1 = J.j1, ny = J.ny;
    const int w = j1 - j0 + 1, h = i1 - i0 + 1;
    if (w <= 0 || h <= 0) return;
    const int tw = (w + kHelmTile - 1) / kHelmTile, th = (h + kHelmTile - 1) / kHelmTile;
    if ((int)blockIdx.x >= tw * th) return;
    const int bi = (int)blockIdx.x / tw, bj = (int)blockIdx.x - bi * tw;
    const int ti0 = i0 + bi * kHelmTile - kHelmDepth;   // region origin
    const int tj0 = j0 + bj * kHelmTile - kHelmDepth;
    __shared__ double ua[kHelmReg * kHelmReg], ub[kHelmReg * kHelmReg];
    const int ex = nx_ext(J.nx), ey = nx_ext(ny);
    const int ci1 = J.lev >= 1 ? J.nx / 2 + ex : 0, cj1 = ny / 2 + ey;   // central region's ends
    const IBPM_GLOBAL double* src = gin(to_out ? J.tmp : J.out);
    const IBPM_GLOBAL double* f = gin(J.f);
    const IBPM_GLOBAL double* Rc = !CHAIN && J.lev >= 1 ? gin(J.R) : f;
    const double in_scale = J.in_scale, inv_diag = J.inv_diag, c = J.c;
    // a thread's points: all loads issued together, from the box's nearest
    // point where the point is off the box and the value is not used
    double r[kHelmPer], u[kHelmPer];
    bool inbox[kHelmPer];
#pragma unroll
    for (int p = 0; p < kHelmPer; ++p) {
        const int q = threadIdx.x + p * kHelmThreads;
        const int i = ti0 + q / kHelmReg, j = tj0 + q % kHelmReg;
        inbox[p] = i >= i0 && i <= i1 && j >= j0 && j <= j1;
        const int k = (int)sidx(J.nx, ny, min(max(i, i0), i1), min(max(j, j0), j1));
        const bool central = i > ex && i < ci1 && j > ey && j < cj1;
        r[p] = (central ? Rc : f)[k];
        u[p] = sweep0 > 0 ? src[k] : 0.0;
    }
    const double* chain = ua;
    if (CHAIN) {
        double *prev = ub, *cur = ua;
        for (int lev = 1; lev <= J.lev; ++lev) {
            helm_chain_level(jobs[(int)blockIdx.y - J.lev + lev], prev, cur);
            chain = cur;
            cur = prev;
            prev = (double*)chain;
        }
    }
#pragma unroll
    for (int p = 0; p < kHelmPer; ++p) {
        const int q = threadIdx.x + p * kHelmThreads;
        const int i = ti0 + q / kHelmReg, j = tj0 + q % kHelmReg;
        const bool support = i >= J.s0 && i <= J.s1 && j >= J.t0 && j <= J.t1;
        const bool central = i > ex && i < ci1 && j > ey && j < cj1;
        if (CHAIN && support && central) r[p] = chain[(i - J.s0) * (J.t1 - J.t0 + 1) + (j - J.t0)];
        r[p] = inbox[p] && support ? r[p] * in_scale : 0.0;
    }
    if (CHAIN) __syncthreads();   // chain is one of the tiles
#pragma unroll
    for (int p = 0; p < kHelmPer; ++p) {
        const int q = threadIdx.x + p * kHelmThreads;
        if (q < kHelmReg * kHelmReg) ua[q] = inbox[p] ? u[p] : 0.0;
    }
    __syncthreads();
    double* cur = ua;
    double* nxt = ub;
    for (int d = 0; d < nsw; ++d) {
        const int m = d + 1;   // points within m of the region's edge are no longer valid
#pragma unroll
        for (int p = 0; p < kHelmPer; ++p) {
            const int q = threadIdx.x + p * kHelmThreads;
            const int a = q / kHelmReg, b = q % kHelmReg;
            if (a < m || b < m || a >= kHelmReg - m || b >= kHelmReg - m) continue;
            double v = 0.0;
            if (sweep0 + d == 0) {
                v = r[p] * inv_diag;
            } else {
                const double s4 = (cur[q - kHelmReg] + cur[q + kHelmReg]) + (cur[q - 1] + cur[q + 1]);
                v = (r[p] - c * s4) * inv_diag;
            }
            nxt[q] = inbox[p] ? v : 0.0;
        }
        __syncthreads();
        double* t = cur;
        cur = nxt;
        nxt = t;
    }
    IBPM_GLOBAL double* dst = gout(to_out ? J.out : J.tmp);
    for (int q = threadIdx.x; q < kHelmTile * kHelmTile; q += kHelmThreads) {
        const int a = kHelmDepth + q / kHelmTile, b = kHelmDepth + q % kHelmTile;
        const int i = ti0 + a, j = tj0 + b;
        if (i > i1 || j > j1) continue;
        dst[sidx(J.nx, ny, i, j)] = cur[a * kHelmReg + b];
    }
}

// The chain of each flow's jobs, levels 1, 2, ... one after another, in the
// workgroup of its level-1 job.
__global__ void __launch_bounds__(kHelmThreads) k_fs_chain(const HelmJob* __restrict__ jobs, int njobs) {
    __shared__ double buf[2][kHelmChainPts];
    const int first = blockIdx.x;
    if (jobs[first].lev != 1 || skipped(jobs[first].skip)) return;
    for (int q = first; q < njobs && jobs[q].lev == 1 + q - first; ++q) {
        const HelmJob& J = jobs[q];
        double* cur = buf[(q - first) & 1];
        helm_chain_level(J, buf[(q - first + 1) & 1], cur);
        const int w = J.t1 - J.t0 + 1, h = J.s1 - J.s0 + 1;
        if (w <= 0 || h <= 0) continue;
        for (int p = threadIdx.x; p < w * h; p += kHelmThreads)
            gout(J.R)[sidx(J.nx, J.ny, J.s0 + p / w, J.t0 + p % w)] = cur[p];
    }
}

// u = W - v over each job's box, v the local result (J.out): the epilogue of
// the step's omega = omega* - A^-1 c in place (W and u are one field, which off
// the boxes holds omega* already).
__global__ void __launch_bounds__(kThreads) k_helm_epilogue(const HelmJob* __restrict__ jobs) {
    const HelmJob& J = jobs[blockIdx.y];
    const int w = J.j1 - J.j0 + 1, h = J.i1 - J.i0 + 1;
    const int p = blockIdx.x * kThreads + threadIdx.x;
    if (w <= 0 || h <= 0 || p >= w * h) return;
    const long k = sidx(J.nx, J.ny, J.i0 + p / w, J.j0 + p % w);
    gout(J.eo)[k] = gin(J.ei)[k] - gin(J.out)[k];
}

// ------------------------------------------------ dense sine-matrix GEMM on MFMA
// A level solve as four dense products with the DST-I matrix S (S[a][b] =
// 2 sin(pi (a+1)(b+1) / n), symmetric), each C = A S of an Np x Np operand A
// (Np = N rounded up to 64, zero padded) held as two bf16 planes, hi =
// bf16(x) and lo = bf16(x - hi): C = Ah Sh + Ah Sl + Al Sh accumulated in FP32
// on the 16x16x32 bf16 MFMA (split-BF16 compensated products; the dropped
// Al Sl term and FP32 accumulation leave a relative error near 1e-6).
//   prep: F = the level's right-hand side (rhs_value) -> planes X0
//   G1: X1^T = (X0 S)^T              along j, written transposed
//   G2: X2^T = X1^T S, / eigenvalue  along i, the spectral scaling
//   G3: X3 = (X2^T S)^T              inverse along i, written transposed
//   G4: u = norm X3 S                inverse along j, FP64 output (pass 3's epilogue)
// A and S fragments are read straight from global memory (16 bytes per lane:
// 8 consecutive bf16 along k, as the MFMA takes them; S symmetric makes its
// columns rows); one wave computes a 32 x 64 tile of C.
typedef __bf16 Bf16x8 __attribute__((ext_vector_type(8)));
typedef float FloatX4 __attribute__((ext_vector_type(4)));

__host__ __device__ constexpr int gemm_np(int n) { return (n + 63) / 64 * 64; }

// The two planes of a level's operand inside the job's scratch:
// plane pair 0 in T1, pair 1 in T2 (each 2 Np^2 bf16 <= the FP64 scratch).
__device__ inline __bf16* gemm_plane(const EllJob& J, int pair, int lohi) {
    const int Np = gemm_np(J.nx - 1);
    __bf16* base = (__bf16*)(pair == 0 ? J.T1 : J.T2);
    return base + (size_t)lohi * Np * Np;
}

__device__ inline void split_bf16(float x, __bf16& hi, __bf16& lo) {
    hi = (__bf16)x;
    lo = (__bf16)(x - (float)hi);
}

// prep: X0 = rhs (FP64 -> FP32 -> hi, lo), zero in the padding.
__global__ void __launch_bounds__(kThreads) k_gemm_prep(const EllJob* __restrict__ jobs) {
    const EllJob& J = jobs[blockIdx.y];
    if (skipped(J.skip)) return;
    const int N1 = J.nx - 1, N2 = J.ny - 1, Np = gemm_np(N1);
    const long t = (long)blockIdx.x * kThreads + threadIdx.x;
    if (t >= (long)Np * Np) return;
    const int i = (int)(t / Np), j = (int)(t % Np);
    const float v = (i < N1 && j < N2) ? (float)rhs_value(J, i + 1, j + 1) : 0.0f;
    __bf16 hi, lo;
    split_bf16(v, hi, lo);
    gemm_plane(J, 0, 0)[t] = hi;
    gemm_plane(J, 0, 1)[t] = lo;
}

// One C = A S product of every job (stage 1..4 as above).  Grid: (Np / 64
// column tiles, Np / 32 row tiles, jobs); one wave per workgroup.
template <int STAGE>
__global__ void __launch_bounds__(64) k_gemm_dst(const EllJob* __restrict__ jobs, const __bf16* __restrict__ Sh,
                                                 const __bf16* __restrict__ Sl, int Np_max) {
    const EllJob& J = jobs[blockIdx.z];
    if (skipped(J.skip)) return;
    const int N1 = J.nx - 1, N2 = J.ny - 1, Np = gemm_np(N1);
    const int c0 = blockIdx.x * 64, r0 = blockIdx.y * 32;
    if (c0 >= Np || r0 >= Np) return;
    const int in_pair = (STAGE == 1 || STAGE == 3) ? 0 : 1;
    const __bf16* Ah = gemm_plane(J, in_pair, 0);
    const __bf16* Al = gemm_plane(J, in_pair, 1);
    const int l = threadIdx.x, lr = l & 15, lk = (l >> 4) * 8;
    FloatX4 acc[2][4];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = FloatX4{0.f, 0.f, 0.f, 0.f};
    // fragments of step k0 are loaded while step k0 - 32 multiplies
    Bf16x8 ah[2], al[2], sh[4], sl[4];
    auto load = [&](int k0, Bf16x8* xh, Bf16x8* xl, Bf16x8* yh, Bf16x8* yl) {
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            const size_t o = (size_t)(r0 + 16 * a + lr) * Np + k0 + lk;
            xh[a] = *(const Bf16x8*)(Ah + o);
            xl[a] = *(const Bf16x8*)(Al + o);
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {   // S[k][c] = S[c][k]: row c, 8 consecutive k
            const size_t o = (size_t)(c0 + 16 * b + lr) * Np_max + k0 + lk;
            yh[b] = *(const Bf16x8*)(Sh + o);
            yl[b] = *(const Bf16x8*)(Sl + o);
        }
    };
    load(0, ah, al, sh, sl);
    for (int k0 = 0; k0 < Np; k0 += 32) {
        Bf16x8 nah[2], nal[2], nsh[4], nsl[4];
        const int kn = k0 + 32 < Np ? k0 + 32 : k0;   // the last step reloads its own (in bounds)
        load(kn, nah, nal, nsh, nsl);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[a], sh[b], acc[a][b], 0, 0, 0);
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[a], sl[b], acc[a][b], 0, 0, 0);
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[a], sh[b], acc[a][b], 0, 0, 0);
            }
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            ah[a] = nah[a];
            al[a] = nal[a];
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            sh[b] = nsh[b];
            sl[b] = nsl[b];
        }
    }
    // C[r][c] of block (a, b): r = r0 + 16 a + 4 (l / 16) + e, c = c0 + 16 b + l % 16
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = r0 + 16 * a + 4 * (l >> 4) + e, c = c0 + 16 * b + lr;
                float v = acc[a][b][e];
                if constexpr (STAGE == 4) {   // u = norm X3 S (+ pass 3's epilogue), rows i = r, columns j = c
                    if (r < N1 && c < N2) {
                        const long o = (long)r * N2 + c;
                        const double vv = (double)v * J.norm;
                        const double uv = J.epilogue ? gin(J.W)[o] - vv : vv;
                        gout(J.u)[o] = uv;
                                    if (J.vside && on_bc_ring(J, r + 1, c + 1)) gout(J.vside)[o] = vv;
                    }
                } else {
                    if constexpr (STAGE == 2) {   // X2^T[l][k] / eigenvalue (EllipticSolver2d.cc:42-54, 89-93)
                        if (r < N2 && c < N1) {
                            const double lam = 2. * (gin(J.pi.cosn)[c] + gin(J.pj.cosn)[r] - 2.) * J.bydx2;
                            v = (float)((double)v * ((J.kind == 0) ? 1. / lam : 1. / (1 + J.alpha * lam)));
                        } else {
                            v = 0.0f;
                        }
                    }
                    __bf16 hi, lo;
                    split_bf16(v, hi, lo);
                    const size_t o = (STAGE == 2) ? (size_t)r * Np + c : (size_t)c * Np + r;   // 1, 3 transposed
                    gemm_plane(J, 1 - in_pair, 0)[o] = hi;
                    gemm_plane(J, 1 - in_pair, 1)[o] = lo;
                }
            }
}

// GEMM-DST of every job of one group (N1 = N2 = N of the plan, <= 511).
// Sh, Sl: the split sine matrix of that N, Np_max columns per row.
void launch_gemm_dst(const EllJob* d_jobs, int njobs, int n, const __bf16* Sh, const __bf16* Sl, hipStream_t s) {
    const int Np = gemm_np(n);
    hipLaunchKernelGGL(k_gemm_prep, dim3((unsigned)(((long)Np * Np + kThreads - 1) / kThreads), njobs),
                       dim3(kThreads), 0, s, d_jobs);
    const dim3 grid(Np / 64, Np / 32, njobs);
    hipLaunchKernelGGL(k_gemm_dst<1>, grid, dim3(64), 0, s, d_jobs, Sh, Sl, Np);
    hipLaunchKernelGGL(k_gemm_dst<2>, grid, dim3(64), 0, s, d_jobs, Sh, Sl, Np);
    hipLaunchKernelGGL(k_gemm_dst<3>, grid, dim3(64), 0, s, d_jobs, Sh, Sl, Np);
    hipLaunchKernelGGL(k_gemm_dst<4>, grid, dim3(64), 0, s, d_jobs, Sh, Sl, Np);
}

// ------------------------------------------------------------ host launch
bool pass_in_registers(int M, long row_pairs) {
    return M == 2048 || (M == 1024 && row_pairs >= kRegMinPairs);
}

bool launch_dst_0(const DstLaunch& L);
bool launch_dst_1(const DstLaunch& L);
bool launch_dst_2(const DstLaunch& L);
bool launch_dst_3(const DstLaunch& L);
bool launch_dst_4(const DstLaunch& L);
bool launch_dst_5(const DstLaunch& L);
bool launch_dst_6(const DstLaunch& L);
bool launch_dst_7(const DstLaunch& L);

static bool launch_dst(const DstLaunch& L) {
    return launch_dst_0(L) || launch_dst_1(L) || launch_dst_2(L) || launch_dst_3(L) || launch_dst_4(L) ||
           launch_dst_5(L) || launch_dst_6(L) || launch_dst_7(L);
}

bool dst_length_built(int M) { return launch_dst(DstLaunch{M, 1, 0, 0, nullptr, nullptr}); }

int blocks_for_pass(const EllJob& J, int pass, bool regs) {
    const int M = pass == 2 ? J.pi.M : J.pj.M, bt = dst_threads(M);
    if (pass == 4) return 1 + (J.bcring ? (J.nx - 1 + bt - 1) / bt : (J.nx / 2 + bt / 64 * kBcRows - 1) / (bt / 64 * kBcRows));
    const int pairs = ((pass == 2 ? J.ny - 1 : J.nx - 1) + 1) / 2;
    const int per = pass == 2 && regs ? r16_group(2) : 1;
    return (pairs + per - 1) / per;
}

int lds_for_pass32(const EllJob& J, int pass) {
    const FftPlan& P = (pass == 2) ? J.pi : J.pj;
    const int ntw = (compiled_len(P.M) && quarter_twiddles(P.M)) ? P.M / 4 : P.M;
    return (int)sizeof(float2) * (P.np * P.M + ntw);
}

#define IBPM_LAUNCH32_LEN(KER)                                                                    \
    switch (M) {                                                                                  \
    case 400: hipLaunchKernelGGL(KER<400>, grid, dim3(kFftThreads), lds_bytes, s, d_jobs); break;   \
    case 512: hipLaunchKernelGGL(KER<512>, grid, dim3(kFftThreads), lds_bytes, s, d_jobs); break;   \
    case 768: hipLaunchKernelGGL(KER<768>, grid, dim3(kFftThreads), lds_bytes, s, d_jobs); break;   \
    case 800: hipLaunchKernelGGL(KER<800>, grid, dim3(kFftThreads), lds_bytes, s, d_jobs); break;   \
    case 1024: hipLaunchKernelGGL(KER<1024>, grid, dim3(kFftThreads), lds_bytes, s, d_jobs); break; \
    case 2048: hipLaunchKernelGGL(KER<2048>, grid, dim3(kFftThreads), lds_bytes, s, d_jobs); break; \
    default: hipLaunchKernelGGL(KER<0>, grid, dim3(kFftThreads), lds_bytes, s, d_jobs); break;      \
    }

int blocks_for_pass32(const EllJob& J, int pass) {
    const int rows_total = (pass == 2) ? J.ny - 1 : J.nx - 1;
    const int rows = 2 * ((pass == 2) ? J.pi : J.pj).np;
    return (rows_total + rows - 1) / rows;
}

// FP32 passes (LDS transforms); max_blocks from blocks_for_pass32, lds_bytes
// from lds_for_pass32.
void launch_ell_pass32(int pass, const EllJob* d_jobs, int njobs, int max_blocks, int lds_bytes, hipStream_t s,
                       bool force_solve, int M) {
    dim3 grid(max_blocks, njobs);
    if (pass == 1) {
        if (force_solve) { IBPM_LAUNCH32_LEN(k32_fs_pass1) } else { IBPM_LAUNCH32_LEN(k32_ell_pass1) }
    } else if (pass == 2) {
        if (force_solve) { IBPM_LAUNCH32_LEN(k32_fs_pass2) } else { IBPM_LAUNCH32_LEN(k32_ell_pass2) }
    } else {
        if (force_solve) { IBPM_LAUNCH32_LEN(k32_fs_pass3) } else { IBPM_LAUNCH32_LEN(k32_ell_pass3) }
    }
}

// Pass 1..3, bc (4) or pass 2 of two solves (5) of jobs of one FFT length M
// (J.pi.M for passes 2 and 5, J.pj.M for the others); regs: pass_in_registers for the launch, with max_blocks
// sized for that choice (bc runs the LDS transform at every length).
void launch_ell_pass(int pass, const EllJob* d_jobs, int njobs, int max_blocks, hipStream_t s, int M, bool regs) {
    const dim3 grid(max_blocks, njobs);
    if (regs && pass < 4) {
        const int lds = (int)sizeof(double2) * r16_group(pass) * r16_buf(M), bt = r16_group(pass) * (M / 16);
        if (M == 2048) {
            if (pass == 1) hipLaunchKernelGGL(k_reg_pass1<2048>, grid, dim3(bt), lds, s, d_jobs);
            else if (pass == 2) hipLaunchKernelGGL(k_reg_pass2<2048>, grid, dim3(bt), lds, s, d_jobs);
            else hipLaunchKernelGGL(k_reg_pass3<2048>, grid, dim3(bt), lds, s, d_jobs);
        } else {
            if (pass == 1) hipLaunchKernelGGL(k_reg_pass1<1024>, grid, dim3(bt), lds, s, d_jobs);
            else if (pass == 2) hipLaunchKernelGGL(k_reg_pass2<1024>, grid, dim3(bt), lds, s, d_jobs);
            else hipLaunchKernelGGL(k_reg_pass3<1024>, grid, dim3(bt), lds, s, d_jobs);
        }
        return;
    }
    (void)launch_dst(DstLaunch{M, pass, max_blocks, njobs, d_jobs, s});   // (plans are of built lengths)
}

void launch_helm_coarsify(const HelmJob* d_jobs, int njobs, int max_blocks, int lev, hipStream_t s) {
    hipLaunchKernelGGL(k_fs_helm_coarsify, dim3(max_blocks, njobs), dim3(kThreads), 0, s, d_jobs, lev);
}

// out = tmp = 0 over each job's box.
__global__ void __launch_bounds__(kThreads) k_helm_clear(const HelmJob* __restrict__ jobs) {
    const HelmJob& J = jobs[blockIdx.y];
    const int w = J.j1 - J.j0 + 1, h = J.i1 - J.i0 + 1;
    const int p = blockIdx.x * kThreads + threadIdx.x;
    if (w <= 0 || h <= 0 || p >= w * h) return;
    const long k = sidx(J.nx, J.ny, J.i0 + p / w, J.j0 + p % w);
    gout(J.out)[k] = 0.0;
    gout(J.tmp)[k] = 0.0;
}

void launch_helm_clear(const HelmJob* d_jobs, int njobs, int max_blocks, hipStream_t s) {
    hipLaunchKernelGGL(k_helm_clear, dim3(max_blocks, njobs), dim3(kThreads), 0, s, d_jobs);
}

void launch_helm_epilogue(const HelmJob* d_jobs, int njobs, int max_blocks, hipStream_t s) {
    hipLaunchKernelGGL(k_helm_epilogue, dim3(max_blocks, njobs), dim3(kThreads), 0, s, d_jobs);
}

int helm_launches(int nsweeps) { return (nsweeps + kHelmDepth - 1) / kHelmDepth; }

int helm_tiles(int h, int w) { return ((h + kHelmTile - 1) / kHelmTile) * ((w + kHelmTile - 1) / kHelmTile); }

void launch_helm_chain(const HelmJob* d_jobs, int njobs, hipStream_t s) {
    hipLaunchKernelGGL(k_fs_chain, dim3(njobs), dim3(kHelmThreads), 0, s, d_jobs, njobs);
}
void launch_helm_sweeps(const HelmJob* d_jobs, int njobs, int max_tiles, int nsweeps, bool chain, hipStream_t s,
                        const std::function<void(const std::function<void()>&)>& timed_launch) {
    const int nl = (nsweeps + kHelmDepth - 1) / kHelmDepth;
    for (int n = 0; n < nl; ++n) {
        const int s0 = n * kHelmDepth, nsw = std::min(kHelmDepth, nsweeps - s0);
        const bool to_out = ((nl - 1 - n) & 1) == 0;
        timed_launch([&] {
            hipLaunchKernelGGL(chain ? k_fs_helm<true> : k_fs_helm<false>, dim3(max_tiles, njobs), dim3(kHelmThreads), 0, s,
                               d_jobs, s0, nsw, to_out);
        });
    }
}

void launch_coarsify(const CoarsifyJob* d_jobs, int njobs, int max_rows, hipStream_t s, bool force_solve) {
    dim3 grid(max_rows, njobs);
    hipLaunchKernelGGL(force_solve ? k_fs_coarsify : k_coarsify, grid, dim3(kThreads), 0, s, d_jobs);
}

}  // namespace ibpmg
