// Checks of the multigrid kernels on the host, one per command-line name; see
// tests/test_multigrid_cpu.py.
#include <memory>
#include <string>
#include <vector>

#include "k_sort.host.inc"
#include "k_multigrid.host.inc"

namespace flipmi {
template <class T>
static hipError_t fill(T *p, size_t n, T v) {
    std::fill(p, p + n, v);
    return hipSuccess;
}
hipError_t launch_fill_f64(double *p, size_t n, double v, hipStream_t) { return fill(p, n, v); }
hipError_t launch_fill_f32(float *p, size_t n, float v, hipStream_t) { return fill(p, n, v); }
hipError_t launch_fill_i32(int *p, size_t n, int v, hipStream_t) { return fill(p, n, v); }
}  // namespace flipmi

using namespace flipmi;

#define CHECK(c)                                                        \
    do {                                                                \
        if (!(c)) {                                                     \
            std::printf("line %d: %s\n", __LINE__, #c);                 \
            std::exit(1);                                               \
        }                                                               \
    } while (0)

// The projection's inputs on an I x J x K grid with closed walls one cell
// inside it, air everywhere.
struct System {
    GridGeom g{};
    double dt = 1.0 / 60;
    std::vector<float> liquid, wU, wV, wW, wC, u, v, w, sU, sV, sW;
    size_t cell(int i, int j, int k) const { return (size_t)i + (size_t)g.I * ((size_t)j + (size_t)g.J * k); }
    size_t fu(int i, int j, int k) const { return (size_t)i + (size_t)(g.I + 1) * ((size_t)j + (size_t)g.J * k); }
    size_t fv(int i, int j, int k) const { return (size_t)i + (size_t)g.I * ((size_t)j + (size_t)(g.J + 1) * k); }
    size_t fw(int i, int j, int k) const { return cell(i, j, k); }
    System(int I, int J, int K) {
        g.I = I; g.J = J; g.K = K;
        g.dx = 1.0 / std::max(I, std::max(J, K));
        g.invdx = 1.0 / g.dx;
        const size_t nc = (size_t)I * J * K;
        liquid.assign(nc, (float)(3 * g.dx));
        wC.assign(nc, 1.0f);
        wU.assign((size_t)(I + 1) * J * K, 1.0f);
        wV.assign((size_t)I * (J + 1) * K, 1.0f);
        wW.assign((size_t)I * J * (K + 1), 1.0f);
        for (int k = 0; k < K; k++)
            for (int j = 0; j < J; j++)
                for (int i = 0; i < I; i++) {
                    if (i < 2) wU[fu(i, j, k)] = 0.0f;
                    if (j < 2) wV[fv(i, j, k)] = 0.0f;
                    if (k < 2) wW[fw(i, j, k)] = 0.0f;
                    if (i > I - 3) wU[fu(i + 1, j, k)] = 0.0f;
                    if (j > J - 3) wV[fv(i, j + 1, k)] = 0.0f;
                    if (k > K - 3) wW[fw(i, j, k + 1)] = 0.0f;
                }
        u.assign(wU.size(), 0.0f); v.assign(wV.size(), 0.0f); w.assign(wW.size(), 0.0f);
        sU = u; sV = v; sW = w;
    }
    // A pool up to row `rows`, its surface 0.3 cells above the last centre.
    void pool(int rows) {
        for (int k = 0; k < g.K; k++)
            for (int j = 0; j < g.J; j++)
                for (int i = 0; i < g.I; i++)
                    liquid[cell(i, j, k)] = (float)std::min(3.0 * g.dx, (j + 0.7 - rows) * g.dx);
    }
    // Liquid in n^3 cells from (i0, j0, k0) whose outer faces are closed.
    void pocket(int i0, int j0, int k0, int n) {
        for (int a = 0; a < n; a++)
            for (int b = 0; b < n; b++)
                for (int c = 0; c < n; c++) liquid[cell(i0 + a, j0 + b, k0 + c)] = (float)(-0.5 * g.dx);
        for (int a = 0; a < n; a++)
            for (int b = 0; b < n; b++) {
                wU[fu(i0, j0 + a, k0 + b)] = wU[fu(i0 + n, j0 + a, k0 + b)] = 0.0f;
                wV[fv(i0 + a, j0, k0 + b)] = wV[fv(i0 + a, j0 + n, k0 + b)] = 0.0f;
                wW[fw(i0 + a, j0 + b, k0)] = wW[fw(i0 + a, j0 + b, k0 + n)] = 0.0f;
            }
    }
    void stir(unsigned seed) {
        auto next = [&]() {
            seed = seed * 1664525u + 1013904223u;
            return (float)((seed >> 8) * (1.0 / 16777216.0) - 0.5);
        };
        for (auto *f : {&u, &v, &w})
            for (float &x : *f) x = next();
    }
    PressureFields fields() const {
        return PressureFields{liquid.data(), wU.data(), wV.data(), wW.data(), wC.data(), u.data(),
                              v.data(),      w.data(),  sU.data(), sV.data(), sW.data()};
    }
};

struct Solver {
    MgPlan plan;
    std::vector<double> d[6], part;
    std::vector<float> f;
    std::vector<int> ints;
    std::vector<int4> bricks;
    MgScalars sc{};
    MgCoarse coarse{};
    MgSolver mg;
    explicit Solver(const System &s) : plan(make_mg_plan(s.g.I, s.g.J, s.g.K)) {
        CHECK(plan.usable());
        size_t nf = 2 * plan.cells[0], nb = 0;
        for (int l = 0; l < plan.nlevels; l++) nf += 8 * plan.cells[l];
        for (int l = 0; l < plan.nglobal; l++) nb += plan.bricks[l];
        double *dp[6];
        for (int q = 0; q < 6; q++) {
            d[q].assign(plan.cells[0], 0.0);
            dp[q] = d[q].data();
        }
        f.assign(nf, 0.0f);
        part.assign(kMgPartials, 0.0);
        ints.assign(2 * nb + 2 * kMgMaxLevels + scan_scratch_elems((int)nb), 0);
        bricks.assign(nb, int4{});
        mg.bind(plan, dp, f.data(), nf, part.data(), ints.data(), bricks.data(), &sc, &coarse);
        coarse = mg.coarse_host;
    }
    // A solve as the host runs it, from setup to the end or `cap` iterations.
    void solve(const System &s, double tol = 1e-9, int cap = 60) {
        mg.setup(s.g, s.dt, s.fields(), tol, cap, nullptr);
        mg.start(false, nullptr);
        for (int it = 0; it <= 2 * cap && !sc.done; it++) {
            mg.iterate(nullptr, nullptr);
            mg.verify(nullptr);
            if (sc.restart) mg.start(true, nullptr);
        }
    }
    double x(int i, int j, int k) const { return mg.fine.x[(i - 1) + mg.lv[0].px * (j - 1) + mg.lv[0].pxy * (k - 1)]; }
};

// One launch of the restriction in which the solve's end is announced while a
// workgroup's first wave is past its look at it and the others are not: every
// sum that reaches the coarse level is either left out or whole.
static void late_end() {
    System s(20, 20, 20);
    s.pool(14);
    s.stir(3);
    Solver a(s);
    a.mg.setup(s.g, s.dt, s.fields(), 1e-9, 60, nullptr);
    a.mg.start(false, nullptr);
    MgSolver &mg = a.mg;
    const MgLevel &C = mg.lv[1];
    const size_t n = (size_t)C.pxy * C.nz;
    double *norm = mg.part + 2 * kMgBlocks;
    const int blocks = grid_for(mg.lv[0]);
    auto restriction = [&]() {
        for (size_t q = 0; q < n; q++) C.r[q] = -7.0f;
        a.sc.done = 0;
        a.sc.iters = 0;
        cpu::launch((unsigned)blocks, kMgThreads, 0,
                    [&] { k_mg_restrict(mg.lv[0], mg.lists, C, (const double *)norm, blocks, &a.sc); });
        return std::vector<float>(C.r, C.r + n);
    };
    for (int q = 0; q < blocks; q++) norm[q] = 1.0;  // no convergence by itself
    const std::vector<float> whole = restriction();
    for (unsigned late = 0; late < (unsigned)blocks; late += 5) {
        cpu::on_yield = [&] {
            if (cpu::block_idx.x == late && cpu::thread_idx.x == 63) a.sc.done = 1;
        };
        const std::vector<float> got = restriction();
        cpu::on_yield = nullptr;
        for (size_t q = 0; q < n; q++) CHECK(got[q] == -7.0f || got[q] == whole[q]);
    }
}

// A right-hand side that is not a number anywhere is no solved system, though
// the rest of it is below the tolerance.
static void not_a_number() {
    for (float bad : {NAN, -NAN, INFINITY}) {
        System s(20, 20, 20);
        s.pool(14);
        s.u[s.fu(9, 6, 11)] = bad;
        Solver a(s);
        a.solve(s);
        CHECK(a.sc.done && !a.sc.converged && a.sc.failed);
    }
    System still(20, 20, 20);
    still.pool(14);
    Solver a(still);
    a.solve(still);
    CHECK(a.sc.done && a.sc.converged && a.sc.iters == 0);
}

// Regions that border no air: cubes that fall into one cell of some level, and
// others, with faces partly open.  The pressure in them is fixed up to a
// constant.
static void pockets() {
    struct Place {
        int i, j, k, n;
        double dt;
    };
    // Interior cell (1, 1, 1) is the first of its aggregates.
    for (const Place &p : {Place{9, 9, 5, 2, 1.0 / 60}, Place{9, 9, 5, 4, 0.013}, Place{5, 9, 1, 8, 1.0 / 60},
                           Place{10, 9, 7, 3, 0.013}}) {
        System s(19, 19, 12);
        s.dt = p.dt;
        s.stir(5);
        for (size_t q = 0; q < s.wU.size(); q++) s.wU[q] *= 0.6f + 0.7f * s.u[q];
        for (size_t q = 0; q < s.wV.size(); q++) s.wV[q] *= 0.6f + 0.7f * s.v[q];
        for (size_t q = 0; q < s.wW.size(); q++) s.wW[q] *= 0.6f + 0.7f * s.w[q];
        s.pool(6);
        s.pocket(p.i, p.j, p.k, p.n);
        s.stir(11);
        Solver a(s);
        a.solve(s, 1e-9, 40);
        std::printf("pocket %d at %d %d %d, dt %g: %d iterations, failed %d\n", p.n, p.i, p.j, p.k, p.dt, a.sc.iters,
                    a.sc.failed);
        CHECK(a.sc.converged && a.sc.iters <= 30);
    }
}

// A solve's result does not depend on what the same store solved before.  The
// pocket's cell of level 1 has no couplings and lies in a brick that holds
// nothing else in the second system, and rows in the first.
static void history() {
    System first(36, 36, 20), second(36, 36, 20);
    first.pool(33);
    first.stir(2);
    second.pool(6);
    second.pocket(9, 29, 9, 2);
    second.stir(11);
    Solver used(first), fresh(second);
    CHECK(used.plan.nglobal >= 2);
    used.solve(first, 1e-2, 4);
    used.solve(second, 1e-3, 8);
    fresh.solve(second, 1e-3, 8);
    CHECK(used.sc.iters == fresh.sc.iters && used.sc.converged && fresh.sc.converged);
    for (int k = 1; k < 19; k++)
        for (int j = 1; j < 35; j++)
            for (int i = 1; i < 35; i++)
                if (second.liquid[second.cell(i, j, k)] < 0) CHECK(used.x(i, j, k) == fresh.x(i, j, k));
}

int main(int argc, char **argv) {
    const std::string name = argc > 1 ? argv[1] : "";
    if (name == "late_end") late_end();
    else if (name == "not_a_number") not_a_number();
    else if (name == "pockets") pockets();
    else if (name == "history") history();
    else return 2;
    std::printf("ok\n");
    return 0;
}
