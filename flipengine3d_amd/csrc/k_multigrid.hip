// The mixed-precision pressure solve: conjugate gradients preconditioned by
// one multigrid V-cycle.
//
// Same system and same stopping rule as PressureSolver / PCGSolver
// (pressuresolver.cpp:44-1047, pcgsolver/pcgsolver.h:248-302): the rows are
// assembled with the reference's arithmetic (assemble_row), and the solve has
// converged when the FP64 true residual satisfies |b - A x|_inf <= tol |b|_inf.
// x, r, q = A s and every dot product are FP64 and q is formed with the FP64
// matrix, so the recursive residual stays the true one; the direction s and
// everything inside the preconditioner are FP32.
//
// The preconditioner.  Rows are aggregated 2 x 2 x 2, level after level, and
// the coarse matrix is half the Galerkin product of the piecewise constant
// prolongation (the product alone overestimates a smooth error's energy by a
// factor of two), which keeps the 7-point stencil: coarse couplings are sums
// of the four fine ones across a face.  Each level smooths with a Chebyshev
// pair of Jacobi steps (damping 1.5 and 0.6) before and after its coarse
// correction.  Restriction is the prolongation's transpose and the pairs are
// polynomials in D^-1 A, so the cycle is symmetric positive definite.
//
// Why not the reference's MIC(0) here: its triangular solves are a chain of
// I + J + K dependent steps (about 75 us each way on a 256x128x128 grid, 30
// tile hand-offs deep), and it takes about 115 iterations to 1e-9 there; the
// V-cycle has no such chain and takes 10 to 22 iterations to 1e-9 at
// 16^3 to 320x160x160 (20 there).
// 256x128x128 double dam break, 1.23 M rows: 21.8 -> 3.2 ms per solve (factor
// included).
// The FP64 path keeps MIC(0), bit for bit, and so do mixed scenes of request
// size; a solve that does not converge here is redone with the FP32 MIC(0)
// iteration.
//
// Layout.  Levels are dense grids of the interior cells, x fastest, with
// zero padding that serves as the halo: a row of nx cells has pitch px > nx,
// a plane ny + 1 rows, and a plane of guard cells lies before and after, so
// every neighbour is a constant offset and no access needs a bounds test.
// Work goes by bricks of 64 x 2 x 2 cells (one 256-thread workgroup; its
// 2 x 2 x 2 aggregates are whole); the bricks with a row in them are listed
// once per solve.  Levels of at most 2048 cells are done by one workgroup in
// LDS.
#include <algorithm>
#include <cstring>
#include <mutex>
#include <set>

#include <hip/hip_ext.h>

#include "multigrid.h"
#include "pressure_device.h"

namespace flipmi {

constexpr int kMgThreads = 256;
constexpr int kBrickX = 64, kBrickY = 2, kBrickZ = 2;
// Grid of the kernels that walk bricks, a multiple of kXcds.  Fixed, so that
// the order of the dot products' partial sums does not depend on anything
// but the system.
constexpr int kMgBlocks = 1024;
static_assert(4 * kMgBlocks <= (int)kMgPartials, "z.r, s.q, the recursive norm and the true one");
constexpr float kDampA = 1.5f, kDampB = 0.6f;
// Least excess of a row's diagonal over its couplings, relative to their sum,
// that is more than rounding (six products and sums in FP64, under 1e-14).  A
// cell of some level that holds a whole region without air has no coupling, and
// an inverse of 1e15 made of such rounding broke the iteration down.
constexpr double kLeastExcess = 1e-12;

// ---------------------------------------------------------------------------
// Shared pieces
// ---------------------------------------------------------------------------

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double o = __shfl_xor(v, off, 64);
        v = o > v ? o : v;
    }
    return v;
}
// The maximum m with a further magnitude.  A NaN counts as infinite, so it can
// pass neither for a right-hand side below the tolerance nor for convergence.
__device__ __forceinline__ double larger(double m, double a) { return a <= m ? m : (a == a ? a : INFINITY); }
// Sum (MAX: maximum) over the workgroup in a fixed order, to every thread.
template <bool MAX>
__device__ __forceinline__ double block_total(double v) {
    __shared__ double sh[kMgThreads / 64];
    v = MAX ? wave_max(v) : wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = sh[0];
#pragma unroll
    for (int w = 1; w < kMgThreads / 64; w++) t = MAX ? (sh[w] > t ? sh[w] : t) : t + sh[w];
    return t;
}
// The total of a kernel's n per-block partials.  Every block of the next
// kernel forms it (n <= kMgBlocks, four loads a thread), which costs less
// than a last block's tickets at the end of the first one.
template <bool MAX>
__device__ __forceinline__ double partials_total(const double *__restrict__ part, int n) {
    double v = 0.0;
    for (int q = (int)threadIdx.x; q < n; q += kMgThreads) {
        const double o = part[q];
        v = MAX ? (o > v ? o : v) : v + o;
    }
    return block_total<MAX>(v);
}

// Whether the solve has ended, the same for every wave of the workgroup: in
// the kernels that may end it, another workgroup of the same launch can do so
// between two waves' reads, and a wave that went on alone would take the sums
// of those that left from LDS nobody wrote.
__device__ __forceinline__ bool ended(const MgScalars *sc) {
    __shared__ int done;
    if (threadIdx.x == 0) done = __hip_atomic_load(&sc->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    return done != 0;
}
__device__ __forceinline__ void end_solve(MgScalars *sc) {
    __hip_atomic_store(&sc->done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Calls f(q, x, y, z, in) for this block's share of the level's active
// bricks: cell (x, y, z) at flat index q, or (in = false) a lane outside the
// level, whose q is the brick's first cell.  The call is uniform over the
// workgroup.
template <class F>
__device__ __forceinline__ void for_bricks(const MgLevel &L, const MgLists &ls, F &&f) {
    const int begin = ls.range[2 * L.index], count = ls.range[2 * L.index + 1];
    const ListRange lr = xcd_list(count);
    const int lx = (int)(threadIdx.x & 63u), ly = (int)((threadIdx.x >> 6) & 1u), lz = (int)(threadIdx.x >> 7);
    for (int e = lr.begin; e < lr.end; e += lr.step) {
        const int4 b = ls.bricks[begin + e];
        const int x = b.x + lx, y = b.y + ly, z = b.z + lz;
        const bool in = x < L.nx && y < L.ny && z < L.nz;
        const int q = in ? b.w + lx + L.px * ly + L.pxy * lz
                              : b.w;
        f(q, x, y, z, in);
    }
}

// Sum of the six neighbours of q weighted by the couplings; at(n) gives the
// value of cell n.
template <class At>
__device__ __forceinline__ float coupled_sum(const MgLevel &L, int q, At &&at) {
    const float *__restrict__ wx = L.wx, *__restrict__ wy = L.wy, *__restrict__ wz = L.wz;
    const int px = L.px, pz = L.pxy;
    float s = wz[q - pz] * at(q - pz);
    s = __builtin_fmaf(wy[q - px], at(q - px), s);
    s = __builtin_fmaf(wx[q - 1], at(q - 1), s);
    s = __builtin_fmaf(wx[q], at(q + 1), s);
    s = __builtin_fmaf(wy[q], at(q + px), s);
    s = __builtin_fmaf(wz[q], at(q + pz), s);
    return s;
}

// One Jacobi step, z + damp D^-1 (r - A z), from the neighbours' weighted sum.
__device__ __forceinline__ float jacobi(float damp, float inv, float r, float z, float coupled) {
    return z + damp * (inv * (r + coupled) - z);
}

// ---------------------------------------------------------------------------
// Setup
// ---------------------------------------------------------------------------

__global__ void k_mg_reset(MgScalars *sc, int maxiter) {
    sc->done = 0;
    sc->failed = 0;
    sc->converged = 0;
    sc->restart = 0;
    sc->iters = 0;
    sc->maxiter = maxiter;
    sc->refinements = 0;
    sc->rho[0] = sc->rho[1] = 0.0;
}

// The rows (assemble_row) of level 0, brick by brick over the whole grid,
// with each block's share of max |rhs| and of the row count.  Every cell of
// the level is written.  inv = mf / diag and the excess e = diag / mf - sum of
// couplings are those of A / mf (mf = dt / dx^2), whose couplings are the face
// weights themselves; scaling a preconditioner changes nothing.
__global__ __launch_bounds__(kMgThreads) void k_mg_assemble(GridGeom g, double dt, AssembleInputs in, MgFine f,
                                                            MgLevel L, int *flags, double *part_max,
                                                            double *part_rows, MgScalars *sc) {
    const double mf = dt / (g.dx * g.dx);
    if (blockIdx.x == 0 && threadIdx.x == 0) sc->mf = mf;
    double bmax = 0.0, rows = 0.0;
    const ListRange lr = xcd_list(L.nbx * L.nby * L.nbz);
    const int lx = (int)(threadIdx.x & 63u), ly = (int)((threadIdx.x >> 6) & 1u), lz = (int)(threadIdx.x >> 7);
    for (int e = lr.begin; e < lr.end; e += lr.step) {
        const int bx = e % L.nbx, t = e / L.nbx, by = t % L.nby, bz = t / L.nby;
        const int x = bx * kBrickX + lx, y = by * kBrickY + ly, z = bz * kBrickZ + lz;
        int row_here = 0;
        if (x < L.nx && y < L.ny && z < L.nz) {
            const int q = x + L.px * y + L.pxy * z;
            PressureRow row;
            float inv = 0.0f, excess = 0.0f;
            if (is_row_cell(g, in.liquid, x + 1, y + 1, z + 1)) {
                row = assemble_row(g, mf, in, x + 1, y + 1, z + 1);
                bmax = larger(bmax, fabs(row.rhs));
                rows += 1.0;
                row_here = 1;
                if (row.diag > 0.0) {
                    inv = (float)(mf / row.diag);
                    const double e = row.diag / mf - row.coupled;
                    excess = e > kLeastExcess * row.coupled ? (float)e : 0.0f;
                }
            }
            f.rhs[q] = row.rhs;
            f.diag[q] = row.diag;
            L.wx[q] = row.wx;
            L.wy[q] = row.wy;
            L.wz[q] = row.wz;
            L.inv[q] = inv;
            L.e[q] = excess;
        }
        const int any = __syncthreads_or(row_here);
        if (threadIdx.x == 0) flags[e] = any ? 1 : 0;
    }
    const double m = block_total<true>(bmax), n = block_total<false>(rows);
    if (threadIdx.x == 0) {
        part_max[blockIdx.x] = m;
        part_rows[blockIdx.x] = n;
    }
}

// Combines the shares; a right-hand side below the absolute tolerance ends
// the solve before it starts (pressuresolver.cpp:52-62).
__global__ __launch_bounds__(kMgThreads) void k_mg_assemble_total(const double *part_max, const double *part_rows,
                                                                  int n, double tol, MgScalars *sc) {
    const double m = partials_total<true>(part_max, n), rows = partials_total<false>(part_rows, n);
    if (threadIdx.x == 0) {
        sc->bnorm = m;
        sc->resid = m;
        sc->rows = (long long)rows;
        sc->tol = (tol < 1e-30 ? 1e-30 : tol) * m;
        if (m < tol) sc->done = sc->converged = 1;
    }
}

// Level l + 1 from level l, brick by brick.  e and the couplings are halves
// of sums over children, so the coarse diagonal e + sum of couplings has no
// cancellation.  A cell above a row counts as active even where that diagonal
// is zero (it holds a whole region without air): the correction reads its z,
// which must be this solve's zero and not what an earlier one left there.
__global__ __launch_bounds__(kMgThreads) void k_mg_coarsen(MgLevel F, MgLevel C, int *flags) {
    const ListRange lr = xcd_list(C.nbx * C.nby * C.nbz);
    const int lx = (int)(threadIdx.x & 63u), ly = (int)((threadIdx.x >> 6) & 1u), lz = (int)(threadIdx.x >> 7);
    for (int b = lr.begin; b < lr.end; b += lr.step) {
        const int bx = b % C.nbx, t = b / C.nbx, by = t % C.nby, bz = t / C.nby;
        const int x = bx * kBrickX + lx, y = by * kBrickY + ly, z = bz * kBrickZ + lz;
        int row_here = 0;
        if (x < C.nx && y < C.ny && z < C.nz) {
            // Children past the level's end are padding and hold zeros, except
            // past its last plane pair, where nothing is allocated.
            const int nz2 = min(2, F.nz - 2 * z), ny2 = min(2, F.ny - 2 * y), nx2 = min(2, F.nx - 2 * x);
            const int f0 = 2 * x + F.px * (2 * y) + F.pxy * (2 * z);
            float e = 0.0f, xm = 0.0f, xp = 0.0f, ym = 0.0f, yp = 0.0f, zm = 0.0f, zp = 0.0f;
            for (int c = 0; c < nz2; c++)
                for (int b2 = 0; b2 < ny2; b2++)
                    for (int a = 0; a < nx2; a++) {
                        const int q = f0 + a + F.px * b2 + F.pxy * c;
                        e += F.e[q];
                        row_here |= F.inv[q] > 0.0f;
                        if (a == 0) xm += F.wx[q - 1]; else xp += F.wx[q];
                        if (b2 == 0) ym += F.wy[q - F.px]; else yp += F.wy[q];
                        if (c == 0) zm += F.wz[q - F.pxy]; else zp += F.wz[q];
                    }
            e *= 0.5f; xm *= 0.5f; xp *= 0.5f; ym *= 0.5f; yp *= 0.5f; zm *= 0.5f; zp *= 0.5f;
            const float d = e + (((xm + xp) + (ym + yp)) + (zm + zp));
            const int q = x + C.px * y + C.pxy * z;
            C.wx[q] = xp;
            C.wy[q] = yp;
            C.wz[q] = zp;
            C.e[q] = e;
            C.inv[q] = d > 0.0f ? 1.0f / d : 0.0f;
            row_here |= d > 0.0f;
        }
        const int any = __syncthreads_or(row_here);
        if (flags && threadIdx.x == 0) flags[b] = any ? 1 : 0;
    }
}

// The active bricks of the levels that are walked by bricks, in order, from
// the scan of their flags; range[2 l], range[2 l + 1] are level l's first
// entry and its number of entries.
__global__ __launch_bounds__(256) void k_mg_lists(MgBrickMap m, const int *__restrict__ flags,
                                                  const int *__restrict__ pos, MgLists ls) {
    const unsigned t = blockIdx.x * 256u + threadIdx.x;
    if (t < (unsigned)m.nlevels) {
        const int b0 = m.first[t], b1 = m.first[t + 1];
        const int total = pos[m.total - 1] + flags[m.total - 1];
        const int begin = b0 < m.total ? pos[b0] : total, end = b1 < m.total ? pos[b1] : total;
        ls.range[2 * t] = begin;
        ls.range[2 * t + 1] = end - begin;
    }
    if (t >= (unsigned)m.total || !flags[t]) return;
    int l = 0;
    while (l + 1 < m.nlevels && (int)t >= m.first[l + 1]) l++;
    const int b = (int)t - m.first[l], bx = b % m.nbx[l], r = b / m.nbx[l], by = r % m.nby[l], bz = r / m.nby[l];
    const int x = bx * kBrickX, y = by * kBrickY, z = bz * kBrickZ;
    ls.bricks[pos[t]] = make_int4(x, y, z, x + m.px[l] * y + m.pxy[l] * z);
}

// ---------------------------------------------------------------------------
// The iteration's kernels on level 0
// ---------------------------------------------------------------------------

// s' = z + beta s and q = A s' (FP64 matrix and sums) with the shares of
// s'.q.  rho = z.r is the total of the last smoothing's shares.  Reads of the
// stencil form s' where they need it; s and s' are two buffers.
template <bool FIRST>
__global__ __launch_bounds__(kMgThreads) void k_mg_spmv(MgFine f, MgLevel L, MgLists ls, const float *__restrict__ s,
                                                        float *s_out, const double *__restrict__ part_zr, int nzr,
                                                        double *part_sq, MgScalars *sc, int turn) {
    if (ended(sc)) return;
    const double rho = partials_total<false>(part_zr, nzr);
    const float beta = FIRST ? 0.0f : (float)(rho / sc->rho[turn ^ 1]);
    const bool bad = !(rho > 0.0) || !(rho <= 1.7976931348623157e308) || !(beta == beta);
    if (bad) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            sc->failed = 1;
            end_solve(sc);
        }
        return;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) sc->rho[turn] = rho;
    const double mf = sc->mf;
    const float *__restrict__ z = L.z;
    const float *__restrict__ wx = L.wx, *__restrict__ wy = L.wy, *__restrict__ wz = L.wz;
    const int px = L.px, pz = L.pxy;
    auto dir = [&](int p) -> float { return FIRST ? z[p] : z[p] + beta * s[p]; };
    double acc = 0.0;
    for_bricks(L, ls, [&](int p, int, int, int, bool in) {
        const float sp = dir(p);
        double v = coupling(wz[p - pz], mf) * (double)dir(p - pz);
        v += coupling(wy[p - px], mf) * (double)dir(p - px);
        v += coupling(wx[p - 1], mf) * (double)dir(p - 1);
        v += f.diag[p] * (double)sp;
        v += coupling(wx[p], mf) * (double)dir(p + 1);
        v += coupling(wy[p], mf) * (double)dir(p + px);
        v += coupling(wz[p], mf) * (double)dir(p + pz);
        if (in) {
            f.q[p] = v;
            s_out[p] = sp;
            acc += (double)sp * v;
        }
    });
    const double t = block_total<false>(acc);
    if (threadIdx.x == 0) part_sq[blockIdx.x] = t;
}

// The axpy x += alpha s, r' = r - alpha q with the shares of |r'|_inf, and
// both steps of the first smoothing on level 0, z = 0 to start with: the
// neighbours' first step needs only their r', formed on the fly, so r and r'
// are two buffers.  kInit starts a solve (r' = b, x = 0), kRestart takes r as
// it is.
enum { kInit = 0, kIterate = 1, kRestart = 2 };
template <int MODE>
__global__ __launch_bounds__(kMgThreads) void k_mg_axpy_smooth(MgFine f, MgLevel L, MgLists ls,
                                                               const double *__restrict__ r, double *r_out,
                                                               const float *__restrict__ s,
                                                               const double *__restrict__ part_sq, int nsq,
                                                               double *part_norm, MgScalars *sc, int turn) {
    if (ended(sc)) return;
    double alpha = 0.0;
    if (MODE == kIterate) {
        const double sq = partials_total<false>(part_sq, nsq);
        alpha = sc->rho[turn] / sq;
        if (!(sq > 0.0) || !(alpha == alpha) || !(alpha <= 1.7976931348623157e308)) {
            if (blockIdx.x == 0 && threadIdx.x == 0) {
                sc->failed = 1;
                end_solve(sc);
            }
            return;
        }
    }
    if (MODE == kRestart && blockIdx.x == 0 && threadIdx.x == 0) sc->restart = 0;
    const double *__restrict__ q = f.q;
    const float *__restrict__ inv = L.inv;
    auto next = [&](int p) -> double { return MODE == kIterate ? r[p] - alpha * q[p] : r[p]; };
    double mx = 0.0;
    for_bricks(L, ls, [&](int p, int, int, int, bool in) {
        const double rp = next(p);
        const float rf = (float)rp, ip = inv[p];
        const float c = coupled_sum(L, p, [&](int n) { return kDampA * (inv[n] * (float)next(n)); });
        if (in) {
            r_out[p] = rp;
            L.r[p] = rf;
            L.z[p] = jacobi(kDampB, ip, rf, kDampA * (ip * rf), c);
            if (MODE == kIterate) f.x[p] += alpha * (double)s[p];
            if (MODE == kInit) f.x[p] = 0.0;
            mx = larger(mx, fabs(rp));
        }
    });
    const double t = block_total<true>(mx);
    if (threadIdx.x == 0) part_norm[blockIdx.x] = t;
}

// The true residual b - A x in FP64 with the shares of its maximum, once the
// recursive one has met the tolerance (or the iterations are used up).
__global__ __launch_bounds__(kMgThreads) void k_mg_true_residual(MgFine f, MgLevel L, MgLists ls, double *r_out,
                                                                 double *part_norm, const MgScalars *sc) {
    if (!sc->done || sc->failed || sc->converged) return;
    const double mf = sc->mf;
    const double *__restrict__ x = f.x;
    const float *__restrict__ wx = L.wx, *__restrict__ wy = L.wy, *__restrict__ wz = L.wz;
    const int px = L.px, pz = L.pxy;
    double mx = 0.0;
    for_bricks(L, ls, [&](int p, int, int, int, bool in) {
        double v = coupling(wz[p - pz], mf) * x[p - pz];
        v += coupling(wy[p - px], mf) * x[p - px];
        v += coupling(wx[p - 1], mf) * x[p - 1];
        v += f.diag[p] * x[p];
        v += coupling(wx[p], mf) * x[p + 1];
        v += coupling(wy[p], mf) * x[p + px];
        v += coupling(wz[p], mf) * x[p + pz];
        const double rp = f.rhs[p] - v;
        if (in) {
            r_out[p] = rp;
            mx = larger(mx, fabs(rp));
        }
    });
    const double t = block_total<true>(mx);
    if (threadIdx.x == 0) part_norm[blockIdx.x] = t;
}

__global__ __launch_bounds__(kMgThreads) void k_mg_verify(const double *part_norm, int n, MgScalars *sc) {
    if (!sc->done || sc->failed || sc->converged) return;
    const double m = partials_total<true>(part_norm, n);
    __syncthreads();  // every thread has read done
    if (threadIdx.x == 0) {
        sc->resid = m;
        sc->refinements += 1;
        if (m <= sc->tol) {
            sc->converged = 1;
        } else if (sc->iters < sc->maxiter && sc->bnorm > 0.0) {
            sc->done = 0;
            sc->restart = 1;  // the host restarts from this residual
        }
    }
}

// ---------------------------------------------------------------------------
// V-cycle
// ---------------------------------------------------------------------------

// Both pre-smoothing steps of a coarser level.
__global__ __launch_bounds__(kMgThreads) void k_mg_smooth_down(MgLevel L, MgLists ls, const MgScalars *sc) {
    if (sc->done) return;
    const float *__restrict__ inv = L.inv, *__restrict__ r = L.r;
    for_bricks(L, ls, [&](int p, int, int, int, bool in) {
        const float rp = r[p], ip = inv[p];
        const float c = coupled_sum(L, p, [&](int n) { return kDampA * (inv[n] * r[n]); });
        if (in) L.z[p] = jacobi(kDampB, ip, rp, kDampA * (ip * rp), c);
    });
}

// The residual r - A z, summed over each 2 x 2 x 2 aggregate.  On level 0 it
// also decides on the norm the axpy left (norm != nullptr).
__global__ __launch_bounds__(kMgThreads) void k_mg_restrict(MgLevel L, MgLists ls, MgLevel C, const double *norm,
                                                            int nnorm, MgScalars *sc) {
    __shared__ float sh[4][64];
    if (ended(sc)) return;
    if (norm) {
        const double m = partials_total<true>(norm, nnorm);
        const bool stop = m <= sc->tol;
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            const int it = sc->iters + 1;
            sc->iters = it;
            sc->resid = m;
            if (stop || it >= sc->maxiter) end_solve(sc);
        }
        if (stop) return;
    }
    const float *__restrict__ z = L.z;
    for_bricks(L, ls, [&](int p, int x, int y, int zc, bool in) {
        const float ip = L.inv[p];
        const float c = coupled_sum(L, p, [&](int n) { return z[n]; });
        // A z = z / inv - coupled; cells that are no rows have inv = 0.
        float v = in && ip > 0.0f ? (L.r[p] - z[p] / ip) + c : 0.0f;
        v += __shfl_xor(v, 1, 64);
        __syncthreads();  // the last brick's sums are read
        sh[threadIdx.x >> 6][threadIdx.x & 63] = v;
        __syncthreads();
        if (threadIdx.x < 64 && (threadIdx.x & 1) == 0 && in) {
            const float t = (sh[0][threadIdx.x] + sh[1][threadIdx.x]) + (sh[2][threadIdx.x] + sh[3][threadIdx.x]);
            C.r[(x >> 1) + C.px * (y >> 1) + C.pxy * (zc >> 1)] = t;
        }
    });
}

// The coarse correction and the first post-smoothing step: y = z' + damp
// D^-1 (r - A z') with z' = z + P z_coarse formed where the stencil reads it.
__global__ __launch_bounds__(kMgThreads) void k_mg_correct(MgLevel L, MgLists ls, MgLevel C, const MgScalars *sc) {
    if (sc->done) return;
    const float *__restrict__ z = L.z, *__restrict__ zc = C.z, *__restrict__ inv = L.inv;
    const int px = L.px, pz = L.pxy;
    const long long cpx = C.px, cpz = C.pxy;
    for_bricks(L, ls, [&](int p, int x, int y, int k, bool in) {
        // Parents of the cell and of its neighbours (level padding is even:
        // the parent of index -1 is the coarse padding at -1).
        auto parent = [&](int a, int b, int c) -> float {
            return zc[(a >> 1) + cpx * (b >> 1) + cpz * (c >> 1)];
        };
        const int x1 = in ? x : 0, y1 = in ? y : 0, k1 = in ? k : 0;
        const float ip = inv[p], own = parent(x1, y1, k1);
        const float *__restrict__ wx = L.wx, *__restrict__ wy = L.wy, *__restrict__ wz = L.wz;
        float c = wz[p - pz] * (z[p - pz] + parent(x1, y1, k1 - 1));
        c = __builtin_fmaf(wy[p - px], z[p - px] + parent(x1, y1 - 1, k1), c);
        c = __builtin_fmaf(wx[p - 1], z[p - 1] + parent(x1 - 1, y1, k1), c);
        c = __builtin_fmaf(wx[p], z[p + 1] + parent(x1 + 1, y1, k1), c);
        c = __builtin_fmaf(wy[p], z[p + px] + parent(x1, y1 + 1, k1), c);
        c = __builtin_fmaf(wz[p], z[p + pz] + parent(x1, y1, k1 + 1), c);
        if (in) L.y[p] = ip > 0.0f ? jacobi(kDampB, ip, L.r[p], z[p] + own, c) : 0.0f;
    });
}

// The last post-smoothing step; on level 0 with the shares of z.r (FP64 r).
template <bool DOT>
__global__ __launch_bounds__(kMgThreads) void k_mg_smooth_up(MgLevel L, MgLists ls, const double *__restrict__ r64,
                                                             double *part_zr, const MgScalars *sc) {
    if (sc->done) return;
    const float *__restrict__ y = L.y;
    double acc = 0.0;
    for_bricks(L, ls, [&](int p, int, int, int, bool in) {
        const float c = coupled_sum(L, p, [&](int n) { return y[n]; });
        const float v = jacobi(kDampA, L.inv[p], L.r[p], y[p], c);
        if (in) {
            const float out = L.inv[p] > 0.0f ? v : 0.0f;
            L.z[p] = out;
            if (DOT) acc += (double)out * r64[p];
        }
    });
    if (DOT) {
        const double t = block_total<false>(acc);
        if (threadIdx.x == 0) part_zr[blockIdx.x] = t;
    }
}

// The V-cycle from the first level of at most kMgCoarseCells cells down, by
// one workgroup.  Everything it needs is brought to LDS at once: couplings,
// inverse diagonals and, per cell, where its aggregate lies, so that each of
// the forty or so dependent passes is a few LDS reads and a barrier.  Bound by
// that chain: 1024 cells of a 256x128x128 grid 19.5 us, 16 on the mean over all
// launches with those past convergence.  (8192 cells with the couplings read
// from the L2 in every pass took 62 us on that mean, more than four launches per
// level cost.)
// Cells lie unpadded: a neighbour beyond the grid is some other cell, and its
// coupling is zero (zero guards stand before and after the arrays).
constexpr int kCoarseThreads = 512;
__global__ __launch_bounds__(kCoarseThreads) void k_mg_coarse(const MgCoarse *__restrict__ a, const MgScalars *sc) {
    extern __shared__ float lds[];
    if (sc->done) return;
    const int tid = (int)threadIdx.x;
    for (int q = tid; q < a->lds_floats; q += kCoarseThreads) lds[q] = 0.0f;
    __syncthreads();
    const int last = a->nlevels - 1;
    for (int l = 0; l <= last; l++) {
        const MgCoarseLevel &C = a->lv[l];
        unsigned short *const at = reinterpret_cast<unsigned short *>(lds + C.at);
        for (int c = tid; c < C.n; c += kCoarseThreads) {
            const int x = c % C.nx, t = c / C.nx, y = t % C.ny, z = t / C.ny;
            const int q = x + C.gpx * y + C.gpxy * z;
            lds[C.wx + c] = C.gwx[q];
            lds[C.wy + c] = C.gwy[q];
            lds[C.wz + c] = C.gwz[q];
            lds[C.inv + c] = C.ginv[q];
            if (l == 0) lds[C.r + c] = C.gr[q];
            // Where the cell's residual goes, its aggregate, and the first of
            // its own children's residuals.
            at[c] = (unsigned short)(x + C.ex * (y + C.ey * z));
            if (l < last) {
                const MgCoarseLevel &D = a->lv[l + 1];
                at[C.n + c] = (unsigned short)((x >> 1) + D.nx * ((y >> 1) + D.ny * (z >> 1)));
            }
            if (l > 0) {
                const MgCoarseLevel &F = a->lv[l - 1];
                at[2 * C.n + c] = (unsigned short)(2 * x + F.ex * (2 * y + F.ey * (2 * z)));
            }
        }
    }
    __syncthreads();
    auto coupled = [&](const MgCoarseLevel &C, const float *z, int c) -> float {
        const float *const wx = lds + C.wx, *const wy = lds + C.wy, *const wz = lds + C.wz;
        float s = wz[c - C.nxy] * z[c - C.nxy];
        s = __builtin_fmaf(wy[c - C.nx], z[c - C.nx], s);
        s = __builtin_fmaf(wx[c - 1], z[c - 1], s);
        s = __builtin_fmaf(wx[c], z[c + 1], s);
        s = __builtin_fmaf(wy[c], z[c + C.nx], s);
        s = __builtin_fmaf(wz[c], z[c + C.nxy], s);
        return s;
    };
    // One Jacobi step from one buffer to the other.
    auto step = [&](const MgCoarseLevel &C, int from, int to, float damp) {
        for (int c = tid; c < C.n; c += kCoarseThreads) {
            const float ip = lds[C.inv + c];
            lds[to + c] = ip > 0.0f ? jacobi(damp, ip, lds[C.r + c], lds[from + c], coupled(C, lds + from, c)) : 0.0f;
        }
        __syncthreads();
    };
    auto first = [&](const MgCoarseLevel &C) {  // the first step, from zero
        for (int c = tid; c < C.n; c += kCoarseThreads) lds[C.z + c] = kDampA * (lds[C.inv + c] * lds[C.r + c]);
        __syncthreads();
    };
    for (int l = 0; l < last; l++) {
        const MgCoarseLevel &C = a->lv[l], &D = a->lv[l + 1];
        first(C);
        step(C, C.z, C.y, kDampB);
        const unsigned short *const at = reinterpret_cast<const unsigned short *>(lds + C.at);
        for (int c = tid; c < C.n; c += kCoarseThreads) {
            const float ip = lds[C.inv + c];
            lds[C.res + at[c]] =
                ip > 0.0f ? (lds[C.r + c] - lds[C.y + c] / ip) + coupled(C, lds + C.y, c) : 0.0f;
        }
        __syncthreads();
        const unsigned short *const dt = reinterpret_cast<const unsigned short *>(lds + D.at);
        for (int c = tid; c < D.n; c += kCoarseThreads) {
            const float *const e = lds + C.res + dt[2 * D.n + c];
            const int py = C.ex, pz = C.ex * C.ey;
            lds[D.r + c] = ((e[0] + e[1]) + (e[py] + e[py + 1])) + ((e[pz] + e[pz + 1]) + (e[pz + py] + e[pz + py + 1]));
        }
        __syncthreads();
    }
    const MgCoarseLevel &E = a->lv[last];
    first(E);
    step(E, E.z, E.y, kDampB);
    for (int q = 0; q < 3; q++) {
        step(E, E.y, E.z, kDampB);
        step(E, E.z, E.y, kDampA);
    }
    for (int l = last - 1; l >= 0; l--) {
        const MgCoarseLevel &C = a->lv[l], &D = a->lv[l + 1];
        const unsigned short *const at = reinterpret_cast<const unsigned short *>(lds + C.at);
        const int zc = l + 1 == last ? D.y : D.z;
        for (int c = tid; c < C.n; c += kCoarseThreads)
            lds[C.z + c] = lds[C.inv + c] > 0.0f ? lds[C.y + c] + lds[zc + at[C.n + c]] : 0.0f;
        __syncthreads();
        step(C, C.z, C.y, kDampB);
        step(C, C.y, C.z, kDampA);
    }
    const MgCoarseLevel &T = a->lv[0];
    const int out = last == 0 ? T.y : T.z;
    for (int c = tid; c < T.n; c += kCoarseThreads) {
        const int x = c % T.nx, t = c / T.nx, y = t % T.ny, z = t / T.ny;
        T.gz[x + T.gpx * y + T.gpxy * z] = lds[out + c];
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

namespace {

int pitch_for(int nx) { return (nx + 1 + 31) & ~31; }

// LDS layout of one level done by one workgroup, from offset `at` on;
// returns the offset after it.
size_t place_coarse(const int d[3], size_t at, MgCoarseLevel &C) {
    const size_t n = (size_t)d[0] * d[1] * d[2], g = (size_t)d[0] * d[1];
    auto take = [&](size_t before, size_t count, size_t after) {
        const size_t o = at + before;
        at = o + count + after;
        return (int)o;
    };
    C.nx = d[0]; C.ny = d[1]; C.nxy = (int)g; C.n = (int)n;
    C.ex = (d[0] + 1) & ~1; C.ey = (d[1] + 1) & ~1;
    C.wx = take(g, n, 0); C.wy = take(g, n, 0); C.wz = take(g, n, 0);
    C.inv = take(0, n, 0);
    C.r = take(0, n, 0);
    C.z = take(g, n, g); C.y = take(g, n, g);
    C.res = take(0, (size_t)C.ex * C.ey * (size_t)((d[2] + 1) & ~1), 0);
    C.at = take(0, (3 * n + 1) / 2, 0);
    return at;
}
constexpr size_t kCoarseLdsLimit = 150 * 1024 / sizeof(float);

size_t coarse_lds_from(const MgPlan &p, int l0) {
    size_t at = 0;
    MgCoarseLevel C{};
    for (int l = l0; l < p.nlevels; l++) at = place_coarse(p.dims[l], at, C);
    return at;
}

template <class K, class... A>
hipError_t launch_timed(K kernel, int blocks, hipStream_t s, const KernelTiming *kt, A... args) {
    if (kt && kt->start) {
        hipExtLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kMgThreads), 0, s, kt->start, kt->stop, 0,
                              args...);
        return hipGetLastError();
    }
    kernel<<<blocks, kMgThreads, 0, s>>>(args...);
    return hipGetLastError();
}

int grid_for(const MgLevel &L) {
    const int n = L.nbx * L.nby * L.nbz;
    return std::min(kMgBlocks, (n + (int)kXcds - 1) / (int)kXcds * (int)kXcds);
}

}  // namespace

MgPlan make_mg_plan(int I, int J, int K) {
    MgPlan p;
    int d[3] = {I - 2, J - 2, K - 2};
    if (d[0] < 1 || d[1] < 1 || d[2] < 1) return p;
    for (int l = 0; l < kMgMaxLevels; l++) {
        for (int a = 0; a < 3; a++) p.dims[l][a] = d[a];
        p.nlevels = l + 1;
        const size_t px = (size_t)pitch_for(d[0]), pxy = px * (size_t)(d[1] + 1);
        p.guard[l] = pxy + px + 32;
        p.guard[l] = (p.guard[l] + 31) & ~(size_t)31;
        p.cells[l] = pxy * (size_t)d[2] + 2 * p.guard[l];
        p.bricks[l] = (size_t)((d[0] + kBrickX - 1) / kBrickX) * ((d[1] + kBrickY - 1) / kBrickY) *
                      ((d[2] + kBrickZ - 1) / kBrickZ);
        if (d[0] <= 2 && d[1] <= 2 && d[2] <= 2 && l >= 1) break;
        for (int a = 0; a < 3; a++) d[a] = (d[a] + 1) / 2;
    }
    // The first level below level 0 that one workgroup can hold.
    p.nglobal = 0;
    for (int l = 1; l < p.nlevels; l++) {
        const size_t n = (size_t)p.dims[l][0] * p.dims[l][1] * p.dims[l][2];
        if (n <= (size_t)kMgCoarseCells && coarse_lds_from(p, l) <= kCoarseLdsLimit) {
            p.nglobal = l;
            break;
        }
    }
    // Cell offsets (negative ones too, into the guards) and brick numbers are
    // ints.
    if (p.cells[0] >= 0x7fffffffull || p.bricks[0] >= 0x3fffffffull) p.nglobal = 0;
    return p;
}

size_t MgPlan::device_bytes() const {
    if (!usable()) return 0;
    size_t b = cells[0] * (6 * sizeof(double) + 2 * sizeof(float));  // rhs, diag, x, q, r twice; s twice
    size_t nb = 0;
    for (int l = 0; l < nlevels; l++) b += cells[l] * 8 * sizeof(float);  // wx, wy, wz, inv, e, r, z, y
    for (int l = 0; l < nglobal; l++) nb += bricks[l];
    b += nb * (2 * sizeof(int) + sizeof(int4)) + sizeof(int) * (2 * kMgMaxLevels + scan_scratch_elems((int)nb));
    return b + sizeof(double) * kMgPartials + sizeof(MgScalars) + sizeof(MgCoarse);
}

hipError_t MgSolver::clear(hipStream_t s) {
    for (int q = 0; q < 6; q++) {
        hipError_t e = launch_fill_f64(d64[q], plan.cells[0], 0.0, s);
        if (e != hipSuccess) return e;
    }
    return launch_fill_f32(f32, nf32, 0.0f, s);
}

void MgSolver::bind(const MgPlan &p, double *const d[6], float *f, size_t nf, double *partials, int *ints,
                    int4 *brick_list, MgScalars *scalars, MgCoarse *coarse_dev) {
    plan = p;
    for (int q = 0; q < 6; q++) d64[q] = d[q];
    f32 = f;
    nf32 = nf;
    sc = scalars;
    part = partials;
    const size_t g0 = p.guard[0];
    fine.rhs = d[0] + g0; fine.diag = d[1] + g0; fine.x = d[2] + g0; fine.q = d[3] + g0;
    ra = d[4] + g0; rb = d[5] + g0;
    sa = f + g0; sb = f + p.cells[0] + g0;
    float *at = f + 2 * p.cells[0];
    map.nlevels = p.nglobal;
    map.total = 0;
    for (int l = 0; l < p.nlevels; l++) {
        MgLevel &L = lv[l];
        L.index = l;
        L.nx = p.dims[l][0]; L.ny = p.dims[l][1]; L.nz = p.dims[l][2];
        L.px = pitch_for(L.nx); L.pxy = L.px * (L.ny + 1);
        L.nbx = (L.nx + kBrickX - 1) / kBrickX;
        L.nby = (L.ny + kBrickY - 1) / kBrickY;
        L.nbz = (L.nz + kBrickZ - 1) / kBrickZ;
        float **arr[8] = {&L.wx, &L.wy, &L.wz, &L.inv, &L.e, &L.r, &L.z, &L.y};
        for (int q = 0; q < 8; q++) {
            *arr[q] = at + p.guard[l];
            at += p.cells[l];
        }
        if (l < p.nglobal) {
            map.first[l] = map.total;
            map.nbx[l] = L.nbx; map.nby[l] = L.nby; map.px[l] = L.px; map.pxy[l] = L.pxy;
            map.total += (int)p.bricks[l];
        }
    }
    map.first[p.nglobal] = map.total;
    flags = ints;
    pos = flags + map.total;
    lists.range = pos + map.total;
    scan_tmp = lists.range + 2 * kMgMaxLevels;
    lists.bricks = brick_list;
    coarse = coarse_dev;
    std::memset(&coarse_host, 0, sizeof(coarse_host));
    coarse_host.nlevels = p.nlevels - p.nglobal;
    size_t lds = 0;
    for (int q = 0; q < coarse_host.nlevels; q++) {
        const MgLevel &L = lv[p.nglobal + q];
        MgCoarseLevel &C = coarse_host.lv[q];
        lds = place_coarse(p.dims[p.nglobal + q], lds, C);
        C.gpx = L.px; C.gpxy = L.pxy;
        C.gwx = L.wx; C.gwy = L.wy; C.gwz = L.wz; C.ginv = L.inv;
        C.gr = L.r; C.gz = L.z;
    }
    coarse_host.lds_floats = (int)lds;
}

hipError_t mg_allow_lds(int device) {
    static std::mutex m;
    static std::set<int> done;
    std::lock_guard<std::mutex> lk(m);
    if (done.count(device)) return hipSuccess;
    // Dynamic LDS above 64 KB is opted into per device.
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_mg_coarse),
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)(kCoarseLdsLimit * sizeof(float)));
    if (e == hipSuccess) done.insert(device);
    return e;
}

hipError_t MgSolver::setup(const GridGeom &g, double dt, const PressureFields &p, double tol, int maxiter,
                           hipStream_t s) {
    const AssembleInputs in{p.liquid, p.wU, p.wV, p.wW, p.wC, p.u, p.v, p.w, p.sU, p.sV, p.sW};
    k_mg_reset<<<1, 1, 0, s>>>(sc, maxiter);
    const int blocks = grid_for(lv[0]);
    k_mg_assemble<<<blocks, kMgThreads, 0, s>>>(g, dt, in, fine, lv[0], flags, part, part + kMgBlocks, sc);
    k_mg_assemble_total<<<1, kMgThreads, 0, s>>>(part, part + kMgBlocks, blocks, tol, sc);
    for (int l = 1; l < plan.nlevels; l++)
        k_mg_coarsen<<<grid_for(lv[l]), kMgThreads, 0, s>>>(lv[l - 1], lv[l],
                                                            l < plan.nglobal ? flags + map.first[l] : nullptr);
    hipError_t e = launch_exclusive_scan(flags, pos, map.total, scan_tmp, s);
    if (e != hipSuccess) return e;
    const int n = std::max(map.total, map.nlevels);
    k_mg_lists<<<(n + 255) / 256, 256, 0, s>>>(map, flags, pos, lists);
    turn = 0;
    return hipGetLastError();
}

hipError_t MgSolver::cycle(bool count, hipStream_t s, const KernelTiming *kt) {
    const int G = plan.nglobal;
    double *norm = part + 2 * kMgBlocks, *zr = part;
    hipError_t e = hipSuccess;
    for (int l = 0; l < G; l++) {
        if (l > 0) k_mg_smooth_down<<<grid_for(lv[l]), kMgThreads, 0, s>>>(lv[l], lists, sc);
        e = launch_timed(k_mg_restrict, grid_for(lv[l]), s, l == 0 && kt ? kt + kPcgForward : nullptr, lv[l], lists,
                         lv[l + 1], (const double *)(l == 0 && count ? norm : nullptr), grid_for(lv[0]), sc);
        if (e != hipSuccess) return e;
    }
    k_mg_coarse<<<1, kCoarseThreads, (size_t)coarse_host.lds_floats * sizeof(float), s>>>(coarse, sc);
    for (int l = G - 1; l >= 0; l--) {
        const bool fine_level = l == 0;
        e = launch_timed(k_mg_correct, grid_for(lv[l]), s, fine_level && kt ? kt + kPcgUpdate : nullptr, lv[l], lists,
                         lv[l + 1], (const MgScalars *)sc);
        if (e != hipSuccess) return e;
        if (fine_level)
            e = launch_timed(k_mg_smooth_up<true>, grid_for(lv[l]), s, kt ? kt + kPcgBackward : nullptr, lv[l], lists,
                             (const double *)r_now(), zr, (const MgScalars *)sc);
        else
            k_mg_smooth_up<false><<<grid_for(lv[l]), kMgThreads, 0, s>>>(lv[l], lists, nullptr, nullptr, sc);
        if (e != hipSuccess) return e;
    }
    return hipGetLastError();
}

hipError_t MgSolver::start(bool restart, hipStream_t s) {
    double *norm = part + 2 * kMgBlocks;
    const int blocks = grid_for(lv[0]);
    if (restart) {
        // The true residual lies in the buffer the next iteration reads.
        k_mg_axpy_smooth<kRestart><<<blocks, kMgThreads, 0, s>>>(fine, lv[0], lists, r_now(), r_next(), nullptr,
                                                                 nullptr, 0, norm, sc, turn);
    } else {
        k_mg_axpy_smooth<kInit><<<blocks, kMgThreads, 0, s>>>(fine, lv[0], lists, fine.rhs, r_next(), nullptr,
                                                              nullptr, 0, norm, sc, turn);
    }
    turn ^= 1;
    first = true;
    return cycle(false, s, nullptr);
}

hipError_t MgSolver::iterate(hipStream_t s, const KernelTiming *kt) {
    double *zr = part, *sq = part + kMgBlocks, *norm = part + 2 * kMgBlocks;
    const int blocks = grid_for(lv[0]);
    const float *s_in = turn ? sb : sa;
    float *s_out = turn ? sa : sb;
    const KernelTiming *k0 = kt ? kt + kPcgSpmv : nullptr, *k1 = kt ? kt + kPcgAxpy : nullptr;
    hipError_t e = first ? launch_timed(k_mg_spmv<true>, blocks, s, k0, fine, lv[0], lists, s_in, s_out,
                                        (const double *)zr, blocks, sq, sc, turn)
                         : launch_timed(k_mg_spmv<false>, blocks, s, k0, fine, lv[0], lists, s_in, s_out,
                                        (const double *)zr, blocks, sq, sc, turn);
    if (e != hipSuccess) return e;
    first = false;
    e = launch_timed(k_mg_axpy_smooth<kIterate>, blocks, s, k1, fine, lv[0], lists, (const double *)r_now(), r_next(),
                     (const float *)s_out, (const double *)sq, blocks, norm, sc, turn);
    if (e != hipSuccess) return e;
    turn ^= 1;
    return cycle(true, s, kt);
}

hipError_t MgSolver::verify(hipStream_t s) {
    double *tr = part + 3 * kMgBlocks;
    const int blocks = grid_for(lv[0]);
    // Over the residual buffer the finished iteration left: it is replaced
    // only when the recursion has stopped.
    k_mg_true_residual<<<blocks, kMgThreads, 0, s>>>(fine, lv[0], lists, r_now(), tr, sc);
    k_mg_verify<<<1, kMgThreads, 0, s>>>(tr, blocks, sc);
    return hipGetLastError();
}

}  // namespace flipmi
