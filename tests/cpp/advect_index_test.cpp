// Every offset that k_advect_rim and k_advect's halo loads form (advect.h), for
// every grid of 4..24 cells a side (multiples of 4) and some thin ones, two to
// four levels: inside its field, and the rim list is what k_advect leaves out.
// Host code only.
#include <cstdio>
#include <vector>

#include "advect.h"

using namespace ibpmg;

static long bad = 0;

static void need(bool ok, const char* what, const Lay& g, int lev, int i, int j) {
    if (ok) return;
    if (++bad <= 10) std::printf("%d x %d x %d: %s out of range at level %d (%d, %d)\n", g.nx, g.ny, g.L, what, lev, i, j);
}

static void point(const Lay& g, int lev, int i, int j, const char* what) {
    need(lev >= 0 && lev < g.L && i >= 1 && i < g.nx && j >= 1 && j < g.ny, what, g, lev, i, j);
    const long k = g.s(lev, i, j);
    need(k >= 0 && k < g.L * g.ns(), what, g, lev, i, j);
}

static void halo(const Lay& g, int lev, int i, int j, const char* what) {
    unsigned a, b;
    halo_at(g, lev, i, j, a, b);
    need(a < (unsigned long)(g.L * g.ns()) && b < (unsigned long)(g.L * g.ns()), what, g, lev, i, j);
}

static void node(const Lay& g, const NodeTerm& t) {
    point(g, t.lev, t.i, t.j, "omega of a node value");
    const NodeFluxes f = node_fluxes(g, t);
    for (int k = 0; k < 4; ++k) {
        const int l = f.lev[k], i = f.i[k], j = f.j[k];
        halo(g, l, t.u ? i : i + 1, t.u ? j + 1 : j, "psi of a flux");
        halo(g, l, i, j, "psi of a flux");
        const bool in = t.u ? i >= 0 && i <= g.nx && j >= 0 && j < g.ny : i >= 0 && i < g.nx && j >= 0 && j <= g.ny;
        need(in && l >= 0 && l < g.L, "flux", g, l, i, j);
    }
}

static void grid(int nx, int ny, int L) {
    const Lay g{nx, ny, L};
    const AdvShape S = adv_shape(nx, ny);
    std::vector<int> seen((size_t)(L * g.ns()), 0);
    const int lanes = (L - 1) * (S.rim * kRimLanes + S.edge);
    for (int idx = 0; idx < (lanes + kThreads - 1) / kThreads * kThreads; ++idx) {
        const RimLane r = rim_lane(g, S, 0.1, idx);
        if (!r.used) continue;
        point(g, r.lev, r.i, r.j, "omega and N_prev of a lane");   // loaded whether the node exists or not
        for (int k = 0; k < 4; ++k) {
            unsigned a, b;
            neighbour_at(g, r.lev, r.i, r.j, k, a, b);
            need(a < (unsigned long)(L * g.ns()) && b < (unsigned long)(L * g.ns()), "neighbour", g, r.lev, r.i, r.j);
        }
        if (r.t.coef != 0.0) node(g, r.t);
        if (!r.rim) need(r.at >= 0 && (size_t)r.at < (size_t)L * S.edge, "edge value", g, r.lev, r.at, 0);
        else if (r.node && idx % kRimLanes == 0) seen[g.s(r.lev, r.i, r.j)] += 1;
    }
    for (int lev = 0; lev < L; ++lev)
        for (int i = 1; i < nx; ++i)
            for (int j = 1; j < ny; ++j)
                need(seen[g.s(lev, i, j)] == (lev >= 1 && is_rim(g, i, j) ? 1 : 0), "rim list", g, lev, i, j);
    for (int lev = 0; lev < L; ++lev)
        for (int i = 0; i <= nx; ++i)
            for (int j = 0; j <= ny; ++j) halo(g, lev, i, j, "tile halo");
}

int main() {
    for (int L = 2; L <= 4; ++L) {
        for (int nx = 4; nx <= 24; nx += 4)
            for (int ny = 4; ny <= 24; ny += 4) grid(nx, ny, L);
        grid(4, 200, L);
        grid(200, 4, L);
        grid(8, 160, L);
        grid(160, 8, L);
    }
    std::printf("%ld offsets out of range\n", bad);
    return bad != 0;
}
