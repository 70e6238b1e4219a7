// advect.h -- index rules of a batch's stencils (k_advect_rim, k_advect in
// ops.hip): which nodes, node values, fluxes and field values each lane reads.
// Host and device, so that every offset can be checked against its field's
// size on the CPU for every grid.
#pragma once
#include "common.h"

namespace ibpmg {

struct Lay {
    int nx, ny, L;
    __host__ __device__ long ns() const { return (long)(nx - 1) * (ny - 1); }
    __host__ __device__ long nf() const { return 2L * nx * ny + nx + ny; }
    __host__ __device__ long nfx() const { return (long)(nx + 1) * ny; }
    __host__ __device__ long s(int lev, int i, int j) const { return lev * ns() + (long)(i - 1) * (ny - 1) + (j - 1); }
    __host__ __device__ long fx(int lev, int i, int j) const { return lev * nf() + (long)i * ny + j; }
    __host__ __device__ long fy(int lev, int i, int j) const { return lev * nf() + nfx() + (long)i * (ny + 1) + j; }
};

constexpr int kAdvI = 8, kAdvJ = 64, kRimLanes = 32;

struct AdvShape {
    int ti, tj, tiles;   // tiles per level
    int rim, edge;       // rim nodes of a coarse level, edge values of a level below the coarsest
};
__host__ __device__ inline AdvShape adv_shape(int nx, int ny) {
    AdvShape s;
    s.ti = (nx - 1 + kAdvI - 1) / kAdvI;
    s.tj = (ny - 1 + kAdvJ - 1) / kAdvJ;
    s.tiles = s.ti * s.tj;
    s.edge = 2 * (ny / 2 + 1) + 2 * (nx / 2 + 1);
    s.rim = nx + ny + 8;
    return s;
}

// Rim node m of a coarse level: rows ex and ex + nx/2 from column ey to ey +
// ny/2, those columns of the rows between, then the two nodes outside each
// corner.  False for one that is not of the level (on 4 cells the nodes outside
// a corner lie on the level's boundary), and (i, j) = (1, 1) then: the caller
// forms addresses from it all the same.
__host__ __device__ inline bool rim_node(const Lay& g, int m, int& i, int& j) {
    const int ex = nx_ext(g.nx), ey = nx_ext(g.ny), hx = ex + g.nx / 2, hy = ey + g.ny / 2;
    const int wide = g.ny / 2 + 1, tall = g.nx / 2 - 1;
    if (m < 2 * wide) {
        i = m < wide ? ex : hx;
        j = ey + m % wide;
    } else if (m < 2 * wide + 2 * tall) {
        m -= 2 * wide;
        j = m < tall ? ey : hy;
        i = ex + 1 + m % tall;
    } else {
        m -= 2 * wide + 2 * tall;   // 0..7: past the corner along i, then along j
        const bool e = m & 1, n = m & 2;
        i = (e ? hx : ex) + (m < 4 ? (e ? 1 : -1) : 0);
        j = (n ? hy : ey) + (m < 4 ? 0 : (n ? 1 : -1));
    }
    const bool in = i >= 1 && i <= g.nx - 1 && j >= 1 && j <= g.ny - 1;
    if (!in) i = j = 1;
    return in;
}
__host__ __device__ inline bool is_rim(const Lay& g, int i, int j) {
    const int ex = nx_ext(g.nx), ey = nx_ext(g.ny), hx = ex + g.nx / 2, hy = ey + g.ny / 2;
    const bool oni = i == ex || i == hx, onj = j == ey || j == hy;
    const bool ini = i >= ex && i <= hx, inj = j >= ey && j <= hy;
    return (oni && inj) || (onj && ini) || ((i == ex - 1 || i == hx + 1) && onj) || ((j == ey - 1 || j == hy + 1) && oni);
}

// A node value in a flux or at an edge: coef times U (u) or V at (lev, i, j).
struct NodeTerm {
    int lev, i, j;
    bool u;
    double coef;   // 0: no term
};

// Term t (0..2) of an X (x) or Y flux outside region G, i in 1..nx-1 of an X
// flux and j in 1..ny-1 of a Y flux (the rules of xflux_from / yflux_from).
__host__ __device__ inline NodeTerm flux_term(const Lay& g, double dx0, bool x, int lev, int i, int j, int t) {
    const double dx = dx0 * (1 << lev);
    const int along = x ? i : j, across = x ? j : i, n = x ? g.ny : g.nx;
    if (across == 0 || across == n - 1) {   // next to the edge: the node inside, and the coarser level's
        const int ea = nx_ext(x ? g.nx : g.ny), ec = nx_ext(n);
        if (t == 0) {
            const int in = across == 0 ? 1 : n - 1;
            return NodeTerm{lev, x ? i : in, x ? in : j, !x, 0.5 * dx};
        }
        const int a = along / 2 + ea + (t - 1), c = across == 0 ? ec : n / 2 + ec;
        const double coef = lev == g.L - 1 || (t == 2 && !(along & 1)) ? 0.0 : (along & 1) ? 0.25 * dx : 0.5 * dx;
        return NodeTerm{lev + 1, x ? a : c, x ? c : a, !x, coef};
    }
    return NodeTerm{lev, x ? i : i + t, x ? j + t : j, !x, t < 2 ? 0.5 * dx : 0.0};
}

// Region G of a coarse level: the fluxes that are the sum of two of the finer
// level, (2 (i - ex), 2 (j - ey) + 0, 1) of an X flux (VectorOperations.cc:669-915).
__host__ __device__ inline bool flux_central(const Lay& g, bool x, int lev, int i, int j) {
    const int ex = nx_ext(g.nx), ey = nx_ext(g.ny), hx = ex + g.nx / 2, hy = ey + g.ny / 2;
    return lev > 0 && (x ? i > ex && i < hx && j >= ey && j < hy : j > ey && j < hy && i >= ex && i < hx);
}

// Number of terms of a rim node's curl: a flux of region G is two of the finer
// level, next to that level's edge, three node values each. With four cells
// across the pair, one of the two lies in the finer level's own region G, so that the
// pairs go on down to level 0.
__host__ __device__ inline int rim_terms(const Lay& g, int lev) {
    return g.nx == 4 || g.ny == 4 ? 12 * (lev + 1) : 24;
}

// Term m (0 .. rim_terms - 1) of fy(i, j) - fy(i - 1, j) + fx(i, j - 1) - fx(i, j).
__host__ __device__ inline NodeTerm rim_term(const Lay& g, double dx0, int lev, int i, int j, int m) {
    const int per = rim_terms(g, lev) / 4, f = m / per, t = m % per;
    const bool x = f >= 2;
    int l = lev, ii = f == 1 ? i - 1 : i, jj = f == 2 ? j - 1 : j, d = t / 3;
    NodeTerm r{0, 1, 1, false, 0.0};
    if (f > 3) return r;
    // flux d of the chain: a pair's member outside region G, then on with the other
    for (; flux_central(g, x, l, ii, jj); --d) {
        ii = 2 * (ii - nx_ext(g.nx));
        jj = 2 * (jj - nx_ext(g.ny));
        --l;
        const bool first = !flux_central(g, x, l, ii, jj);   // the member that the chain ends at
        if ((d == 0) != first) (x ? jj : ii) += 1;
        if (d == 0) break;
    }
    if (d == 0) r = flux_term(g, dx0, x, l, ii, jj, t % 3);
    if (f & 1) r.coef = -r.coef;
    return r;
}

// Offsets of the two values whose mean a level's field has at (i, j), 0 <= i <=
// nx, 0 <= j <= ny, off its corners: its own value twice inside, getBC's of the
// coarser level (Scalar.cc:91-127) on the boundary.  False (offsets of the
// nearest node): 0 on the coarsest level's boundary.
__host__ __device__ inline bool halo_at(const Lay& g, int lev, int i, int j, unsigned& a, unsigned& b) {
    const unsigned ny1 = (unsigned)(g.ny - 1), base = (unsigned)(lev * g.ns());
    const int ci = min(max(i, 1), g.nx - 1), cj = min(max(j, 1), g.ny - 1);
    a = b = base + (unsigned)(ci - 1) * ny1 + (unsigned)(cj - 1);
    if (ci == i && cj == j) return true;
    if (lev == g.L - 1) return false;
    const bool side = ci != i;   // on left or right, else on bottom or top
    const int ii = nx_ext(g.nx) + i / 2, jj = nx_ext(g.ny) + j / 2;
    a = base + (unsigned)g.ns() + (unsigned)(min(max(ii, 1), g.nx - 1) - 1) * ny1 + (unsigned)(min(max(jj, 1), g.ny - 1) - 1);
    b = a + (side ? (unsigned)(j & 1) : (i & 1) * ny1);
    return true;
}

// The fluxes whose weighted sum is a node's velocity times dx (the rules of
// xvel and yvel): X fluxes of U, Y fluxes of V, at (lev, i, j), at most four.
struct NodeFluxes {
    int lev[4], i[4], j[4];
    double co[4];
};
__host__ __device__ inline NodeFluxes node_fluxes(const Lay& g, const NodeTerm& t) {
    const int lev = t.lev, na = t.u ? g.nx : g.ny, nc = t.u ? g.ny : g.nx;   // along and across the flux pair
    const int al = t.u ? t.i : t.j, ac = t.u ? t.j : t.i;
    const int alo = nx_ext(na), ahi = alo + na / 2, clo = nx_ext(nc), chi = clo + nc / 2;
    const bool rim = lev >= 1 && (ac == clo || ac == chi) && al >= alo && al <= ahi;
    const bool corner = rim && (al == alo || al == ahi), face = rim && !corner;
    const int c0 = ac == clo ? ac - 1 : ac, c1 = ac == clo ? ac : ac - 1;   // outside the rim, inside it
    const int cf = ac == clo ? 0 : nc - 1, af = face ? 2 * (al - alo) : al == alo ? 1 : na - 1;
    // fluxes (level, along, across) and coefficients
    const int fl[4] = {lev, (face ? lev - 1 : lev), rim ? lev - 1 : lev, rim ? lev - 1 : lev};
    const int fa[4] = {al, face ? af : al, face ? af - 1 : corner ? af : al, face ? af + 1 : al};
    const int fc[4] = {rim ? c0 : ac, face ? cf : corner ? c1 : ac - 1, rim ? cf : ac, rim ? cf : ac};
    NodeFluxes f{{}, {}, {}, {face ? 2. / 3 : corner ? 8. / 15 : 0.5, face ? 1. / 3 : corner ? 6. / 15 : 0.5,
                             face ? 1. / 6 : corner ? 2. / 15 : 0.0, face ? 1. / 6 : 0.0}};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        f.lev[k] = fl[k] < 0 ? 0 : fl[k];
        f.i[k] = t.u ? fa[k] : fc[k];
        f.j[k] = t.u ? fc[k] : fa[k];
    }
    return f;
}

// Lane idx of k_advect_rim: kRimLanes lanes per rim node, which share its terms
// (first, first + kRimLanes, .. below n), then one lane per edge value (slot at of
// FlowOps::edge, the one term t).  (lev, i, j) is the rim node; every lane's is a
// node of the grid, since the kernel's loads at it are under no branch.
struct RimLane {
    bool used, rim, node;   // node: a rim node of the level
    int lev, i, j, at;
    int first, n;
    NodeTerm t;
};
__host__ __device__ inline RimLane rim_lane(const Lay& g, const AdvShape& S, int idx) {
    RimLane r{true, false, false, 0, 1, 1, 0, 0, 1, NodeTerm{0, 1, 1, false, 0.0}};
    const int nrim = (g.L - 1) * S.rim * kRimLanes;
    r.rim = idx < nrim;
    if (r.rim) {
        const int k = idx / kRimLanes;
        r.lev = k / S.rim + 1;
        r.node = rim_node(g, k % S.rim, r.i, r.j);
        r.first = idx % kRimLanes;
        r.n = r.node ? rim_terms(g, r.lev) : 0;
        return r;
    }
    // U at the coarser level's nodes along left and right, V along bottom and top
    r.at = idx - nrim;
    r.used = r.at < (g.L - 1) * S.edge;
    if (!r.used) return r;
    const int l = r.at / S.edge, wide = g.ny / 2 + 1, tall = g.nx / 2 + 1;
    const int ex = nx_ext(g.nx), ey = nx_ext(g.ny);
    int m = r.at % S.edge;
    const bool u = m < 2 * wide;
    if (!u) m -= 2 * wide;
    if (u) r.t = NodeTerm{l + 1, m < wide ? ex : ex + g.nx / 2, ey + m % wide, true, 1.0};
    else r.t = NodeTerm{l + 1, ex + m % tall, m < tall ? ey : ey + g.ny / 2, false, 1.0};
    return r;
}

// Node (lev, i, j) + neighbour k (0..3: i + 1, i - 1, j + 1, j - 1) of a five-point stencil.
__host__ __device__ inline bool neighbour_at(const Lay& g, int lev, int i, int j, int k, unsigned& a, unsigned& b) {
    return halo_at(g, lev, i + (k == 0) - (k == 1), j + (k == 2) - (k == 3), a, b);
}

}  // namespace ibpmg
