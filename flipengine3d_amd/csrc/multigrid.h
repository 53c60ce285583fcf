// The mixed-precision pressure solve (k_multigrid.hip): conjugate gradients
// with a multigrid preconditioner.
#pragma once

#include <hip/hip_runtime.h>

#include "flipmi_kernels.h"

namespace flipmi {

constexpr int kMgMaxLevels = 24;
constexpr int kMgCoarseCells = 2048;  // cells of the first level done by one workgroup, at most

struct MgScalars {
    double bnorm, tol, resid, mf;
    double rho[2];  // z.r of this and the last iteration, by turn
    long long rows;
    int done, failed, converged, restart, iters, maxiter, refinements;
};

// Level sizes of an I x J x K grid: level 0 holds its interior cells.
struct MgPlan {
    int nlevels = 0, nglobal = 0;  // nglobal: levels done by bricks; the others by one workgroup
    int dims[kMgMaxLevels][3] = {};
    size_t cells[kMgMaxLevels] = {};  // floats per array, padding and guards included
    size_t guard[kMgMaxLevels] = {};  // floats before cell (0, 0, 0)
    size_t bricks[kMgMaxLevels] = {};
    bool usable() const { return nglobal > 0; }
    size_t device_bytes() const;
};
MgPlan make_mg_plan(int I, int J, int K);

// One level.  Couplings towards +x/+y/+z, inverse diagonal, excess of the
// diagonal over the couplings, right-hand side and two solution buffers; the
// pointers are at cell (0, 0, 0).
struct MgLevel {
    int index, nx, ny, nz, nbx, nby, nbz;
    int px, pxy;  // signed: a neighbour of the first cells lies before them
    float *wx, *wy, *wz, *inv, *e, *r, *z, *y;
};
struct MgFine {
    double *rhs, *diag, *x, *q;
};
struct MgLists {
    int4 *bricks;  // first cell (x, y, z) and its flat index
    int *range;    // per level: first entry, number of entries
};
struct MgBrickMap {
    int nlevels, total;
    int first[kMgMaxLevels + 1], nbx[kMgMaxLevels], nby[kMgMaxLevels];
    int px[kMgMaxLevels], pxy[kMgMaxLevels];
};
struct MgCoarseLevel {
    int n, nx, ny, nxy;  // cells, and their unpadded layout in LDS
    int ex, ey;          // layout of the residuals, even sizes
    int gpx, gpxy;       // global layout
    int wx, wy, wz, inv, r, z, y, res, at;  // LDS offsets
    const float *gwx, *gwy, *gwz, *ginv, *gr;
    float *gz;
};
struct MgCoarse {
    int nlevels, lds_floats;
    MgCoarseLevel lv[kMgMaxLevels];
};

struct PressureFields {
    const float *liquid, *wU, *wV, *wW, *wC, *u, *v, *w, *sU, *sV, *sW;
};

// Launches of one solve over buffers it does not own.  setup() assembles the
// system and its levels; start() begins from x = 0 (restart: from the true
// residual verify() left); iterate() runs one iteration; verify() tests the
// true residual once the recursion has stopped.  Nothing waits on the host.
struct MgSolver {
    MgPlan plan;
    MgLevel lv[kMgMaxLevels];
    MgFine fine{};
    MgLists lists{};
    MgBrickMap map{};
    MgCoarse *coarse = nullptr;  // device copy of coarse_host
    MgCoarse coarse_host{};
    MgScalars *sc = nullptr;
    double *d64[6] = {};
    float *f32 = nullptr;
    size_t nf32 = 0;
    double *ra = nullptr, *rb = nullptr, *part = nullptr;
    float *sa = nullptr, *sb = nullptr;
    int *flags = nullptr, *pos = nullptr, *scan_tmp = nullptr;
    int turn = 0;        // which of the two s and r buffers the next iteration reads
    bool first = false;  // the next iteration takes s = z

    // coarse_dev: the caller copies coarse_host there afterwards.
    void bind(const MgPlan &p, double *const d[6], float *f, size_t nf, double *partials, int *ints,
              int4 *brick_list, MgScalars *scalars, MgCoarse *coarse_dev);
    hipError_t clear(hipStream_t s);
    hipError_t setup(const GridGeom &g, double dt, const PressureFields &p, double tol, int maxiter, hipStream_t s);
    hipError_t start(bool restart, hipStream_t s);
    // kt: kPcgPieces timings (those with a start event are recorded), or null.
    hipError_t iterate(hipStream_t s, const KernelTiming *kt);
    hipError_t verify(hipStream_t s);

private:
    double *r_now() const { return turn ? rb : ra; }
    double *r_next() const { return turn ? ra : rb; }
    hipError_t cycle(bool count, hipStream_t s, const KernelTiming *kt);
};
constexpr size_t kMgPartials = 4 * 1024;  // doubles
// Lets the multigrid kernel use its LDS on `device` (current), once.
hipError_t mg_allow_lds(int device);

}  // namespace flipmi
