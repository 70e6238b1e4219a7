// Every offset that k_advect_rim and k_advect's halo loads form (advect.h), for
// every grid of 4..24 cells a side (multiples of 4) and some thin ones, two to
// six levels: inside its field, and the rim list is what k_advect leaves out.
// Host code only.
#include <cmath>
#include <cstdio>
#include <map>
#include <tuple>
#include <vector>

#include "advect.h"

using namespace ibpmg;

static long bad = 0;

static void need(bool ok, const char* what, const Lay& g, int lev, int i, int j) {
    if (ok) return;
    if (++bad <= 10) std::printf("%d x %d x %d: %s wrong at level %d (%d, %d)\n", g.nx, g.ny, g.L, what, lev, i, j);
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

typedef std::map<std::tuple<bool, int, int, int>, double> Sum;   // (U or V, level, i, j) -> coefficient

// sign times the X (x) or Y flux (i, j) of level lev as node values, dx of level 0 being 1
static void flux(const Lay& g, bool x, int lev, int i, int j, double sign, Sum& out) {
    const int ex = nx_ext(g.nx), ey = nx_ext(g.ny), hx = ex + g.nx / 2, hy = ey + g.ny / 2;
    const double h = 0.5 * sign * (1 << lev);
    const bool region = lev > 0 && (x ? i > ex && i < hx && j >= ey && j < hy : j > ey && j < hy && i >= ex && i < hx);
    if (region) {
        for (int k = 0; k < 2; ++k) flux(g, x, lev - 1, 2 * (i - ex) + (x ? 0 : k), 2 * (j - ey) + (x ? k : 0), sign, out);
        return;
    }
    auto add = [&](int l, int a, int b, double c) { out[{!x, l, a, b}] += c; };
    if (x && (j == 0 || j == g.ny - 1)) {   // the node inside, and the coarser level's half way
        add(lev, i, j == 0 ? 1 : j, h);
        if (lev == g.L - 1) return;
        const int b = j == 0 ? ey : hy, a = i / 2 + ex;
        if (i % 2 == 0) { add(lev + 1, a, b, h); return; }
        add(lev + 1, a, b, 0.5 * h);
        add(lev + 1, a + 1, b, 0.5 * h);
    } else if (!x && (i == 0 || i == g.nx - 1)) {
        add(lev, i == 0 ? 1 : i, j, h);
        if (lev == g.L - 1) return;
        const int a = i == 0 ? ex : hx, b = j / 2 + ey;
        if (j % 2 == 0) { add(lev + 1, a, b, h); return; }
        add(lev + 1, a, b, 0.5 * h);
        add(lev + 1, a, b + 1, 0.5 * h);
    } else {
        add(lev, i, j, h);
        add(lev, x ? i : i + 1, x ? j + 1 : j, h);
    }
}

static void rim_sum(const Lay& g, int lev, int i, int j) {
    Sum want, got;
    flux(g, false, lev, i, j, 1, want);
    flux(g, false, lev, i - 1, j, -1, want);
    flux(g, true, lev, i, j - 1, 1, want);
    flux(g, true, lev, i, j, -1, want);
    for (int m = 0; m < rim_terms(g, lev); ++m) {
        const NodeTerm t = rim_term(g, 1.0, lev, i, j, m);
        if (t.coef != 0.0) got[{t.u, t.lev, t.i, t.j}] += t.coef;
    }
    bool same = true;
    for (auto& k : want) same = same && std::fabs(got[k.first] - k.second) <= 1e-12;
    for (auto& k : got) same = same && std::fabs(want[k.first] - k.second) <= 1e-12;
    need(same, "terms of a rim node", g, lev, i, j);
}

static void grid(int nx, int ny, int L) {
    const Lay g{nx, ny, L};
    const AdvShape S = adv_shape(nx, ny);
    std::vector<int> seen((size_t)(L * g.ns()), 0);
    const int lanes = (L - 1) * (S.rim * kRimLanes + S.edge);
    for (int idx = 0; idx < (lanes + kThreads - 1) / kThreads * kThreads; ++idx) {
        const RimLane r = rim_lane(g, S, idx);
        if (!r.used) continue;
        point(g, r.lev, r.i, r.j, "omega and N_prev of a lane");   // loaded whether the node exists or not
        for (int k = 0; k < 4; ++k) {
            unsigned a, b;
            neighbour_at(g, r.lev, r.i, r.j, k, a, b);
            need(a < (unsigned long)(L * g.ns()) && b < (unsigned long)(L * g.ns()), "neighbour", g, r.lev, r.i, r.j);
        }
        for (int m = r.first; m < r.n; m += kRimLanes) {
            const NodeTerm t = r.rim ? rim_term(g, 0.1, r.lev, r.i, r.j, m) : r.t;
            if (t.coef != 0.0) node(g, t);
        }
        if (!r.rim) need(r.at >= 0 && (size_t)r.at < (size_t)L * S.edge, "edge value", g, r.lev, r.at, 0);
        else if (r.node && idx % kRimLanes == 0) seen[g.s(r.lev, r.i, r.j)] += 1;
    }
    for (int lev = 1; lev < L; ++lev)
        for (int i = 1; i < nx; ++i)
            for (int j = 1; j < ny; ++j)
                if (is_rim(g, i, j)) rim_sum(g, lev, i, j);
    for (int lev = 0; lev < L; ++lev)
        for (int i = 1; i < nx; ++i)
            for (int j = 1; j < ny; ++j)
                need(seen[g.s(lev, i, j)] == (lev >= 1 && is_rim(g, i, j) ? 1 : 0), "rim list", g, lev, i, j);
    for (int lev = 0; lev < L; ++lev)
        for (int i = 0; i <= nx; ++i)
            for (int j = 0; j <= ny; ++j) halo(g, lev, i, j, "tile halo");
}

int main() {
    for (int L = 2; L <= 6; ++L) {
        for (int nx = 4; nx <= 24; nx += 4)
            for (int ny = 4; ny <= 24; ny += 4) grid(nx, ny, L);
        grid(4, 200, L);
        grid(200, 4, L);
        grid(8, 160, L);
        grid(160, 8, L);
    }
    std::printf("%ld faults\n", bad);
    return bad != 0;
}
