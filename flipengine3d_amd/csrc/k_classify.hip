// Marker/cell classification: the liquid signed distance field and the
// fluid/air labels it defines (phi < 0 is fluid).
//
// Reference: ParticleLevelSet::calculateSignedDistanceField and
// postProcessSignedDistanceField (particlelevelset.cpp:161-196, 299-630).
// The reference bins particles into 10^3 cell blocks and takes, per block,
//     phi(c) = min(3 dx, min_p |c_local - p_local| - r)
// in block-local float coordinates.  Here one workgroup owns one 10^3 block,
// gathers the particles of the cells around it from the arrays sorted into
// half-cell bins,
// replays the reference's particle-to-block assignment and local arithmetic,
// and folds distances into LDS with an order-independent atomic minimum.
// The result is bit-identical to the reference.
#include "device_math.h"
#include "flipmi_kernels.h"
#include "half_cell_rows.h"

namespace flipmi {

constexpr int kBW = 10;            // particlelevelset.h:140 (_blockwidth)
constexpr int kHalo = 2;           // search radius 2r = sqrt(3) dx < 2 dx
constexpr int kSpan = kBW + 2 * kHalo;
constexpr int kSdfThreads = 256;

// Whether the reference assigns point p to block (bi, bj, bk)
// (particlelevelset.cpp:497-536; velocityadvector.cpp:280-320).
__device__ __forceinline__ bool point_in_block(F3 p, float sr, float blockdx, double inv_blockdx,
                                               int bi, int bj, int bk) {
    I3 b = pos_to_index(p, inv_blockdx);
    F3 bp = idx_to_pos(b.i, b.j, b.k, (double)blockdx);
    if (p.x - sr > bp.x && p.y - sr > bp.y && p.z - sr > bp.z && p.x + sr < bp.x + blockdx &&
        p.y + sr < bp.y + blockdx && p.z + sr < bp.z + blockdx) {
        return b.i == bi && b.j == bj && b.k == bk;
    }
    I3 lo = pos_to_index((double)(p.x - sr), (double)(p.y - sr), (double)(p.z - sr), inv_blockdx);
    I3 hi = pos_to_index((double)(p.x + sr), (double)(p.y + sr), (double)(p.z + sr), inv_blockdx);
    return bi >= lo.i && bi <= hi.i && bj >= lo.j && bj <= hi.j && bk >= lo.k && bk <= hi.k;
}

// ParticleLevelSet::postProcessSignedDistanceField (particlelevelset.cpp:
// 172-196) for one cell: cells within half a cell of the surface whose centre
// lies inside the solid become -dx/2 (MeshLevelSet::getDistanceAtCellCenter,
// meshlevelset.cpp:152-162), and |phi| < 0.005 dx is pushed out to 0.005 dx.
__device__ __forceinline__ float postprocess_phi(const GridGeom &g, const float *__restrict__ solid,
                                                 int i, int j, int k, float v) {
    Dims N{g.I + 1, g.J + 1, g.K + 1};
    float eps = (float)(0.005 * g.dx);
    if ((double)v < 0.5 * g.dx) {
        float sc = 0.125f * (solid[N.at(i, j, k)] + solid[N.at(i + 1, j, k)] +
                             solid[N.at(i, j + 1, k)] + solid[N.at(i + 1, j + 1, k)] +
                             solid[N.at(i, j, k + 1)] + solid[N.at(i + 1, j, k + 1)] +
                             solid[N.at(i, j + 1, k + 1)] + solid[N.at(i + 1, j + 1, k + 1)]);
        if (sc < 0) v = (float)(-0.5f * g.dx);
    }
    if (fabsf(v) < eps) v = v > 0 ? eps : -eps;
    return v;
}

constexpr int kRows = 4 * kSpan * kSpan;           // half-cell rows of the candidate box
constexpr int kRowsPerThread = (kRows + kSdfThreads - 1) / kSdfThreads;

__global__ __launch_bounds__(kSdfThreads) void k_liquid_sdf(
    GridGeom g, const float4 *__restrict__ spos, const int *__restrict__ sub_offset, float radius,
    const float *__restrict__ solid, float *phi_out) {
    __shared__ uint32_t phi_ord[kBW * kBW * kBW];
    __shared__ int run_begin[kRows];
    __shared__ int run_prefix[kRows + 1];
    __shared__ int wave_total[kSdfThreads / 64];
    __shared__ float centre[kBW];  // Grid3d::GridIndexToCellCenter of local index c

    int nbi = (g.I + kBW - 1) / kBW, nbj = (g.J + kBW - 1) / kBW;
    int bid = blockIdx.x;
    int bi = bid % nbi, bj = (bid / nbi) % nbj, bk = bid / (nbi * nbj);
    float maxd = (float)(3.0 * g.dx);  // particlelevelset.cpp:295-297
    uint32_t init = f2ord(maxd);
    for (int c = threadIdx.x; c < kBW * kBW * kBW; c += kSdfThreads) phi_ord[c] = init;
    if (threadIdx.x < kBW) centre[threadIdx.x] = idx_to_center1(threadIdx.x, g.dx);

    // Candidate particles: cells [b0 - 2, b0 + 12) per axis.  In the
    // half-cell sort each (sy, sz) row of half-cells over those cells is one
    // contiguous run: 4 rows per (j, k) row of cells.
    int i0 = max(bi * kBW - kHalo, 0), i1 = min(bi * kBW + kBW + kHalo, g.I);
    int j0 = max(bj * kBW - kHalo, 0), j1 = min(bj * kBW + kBW + kHalo, g.J);
    int k0 = max(bk * kBW - kHalo, 0), k1 = min(bk * kBW + kBW + kHalo, g.K);
    int nsy = 2 * (j1 - j0), nsz = 2 * (k1 - k0), nrows = nsy * nsz;
    const size_t SI = 2 * (size_t)g.I, SJ = 2 * (size_t)g.J;
    // Each thread takes kRowsPerThread consecutive rows; a block-wide
    // exclusive scan of the row lengths gives every row's start.
    int len[kRowsPerThread];
    int mine = 0;
#pragma unroll
    for (int q = 0; q < kRowsPerThread; q++) {
        int r = threadIdx.x * kRowsPerThread + q;
        len[q] = 0;
        if (r < nrows) {
            size_t sy = 2 * (size_t)j0 + (size_t)(r % nsy), sz = 2 * (size_t)k0 + (size_t)(r / nsy);
            size_t b0 = 2 * (size_t)i0 + SI * (sy + SJ * sz);
            size_t b1 = b0 + 2 * (size_t)(i1 - i0);
            int s0 = sub_offset[b0];
            run_begin[r] = s0;
            len[q] = sub_offset[b1] - s0;
        }
        mine += len[q];
    }
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int inc = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        int t = __shfl_up(inc, off, 64);
        if (lane >= off) inc += t;
    }
    if (lane == 63) wave_total[wave] = inc;
    __syncthreads();
    int run = inc - mine;
    for (int w = 0; w < wave; w++) run += wave_total[w];
#pragma unroll
    for (int q = 0; q < kRowsPerThread; q++) {
        int r = threadIdx.x * kRowsPerThread + q;
        if (r < nrows) run_prefix[r] = run;
        run += len[q];
    }
    if (threadIdx.x == kSdfThreads - 1) run_prefix[nrows] = run;
    __syncthreads();
    int total = run_prefix[nrows];

    float r = radius;
    float sr = 2.0f * r;  // particlelevelset.h:142 (_searchRadiusFactor)
    float blockdx = (float)(kBW * g.dx);
    double inv_blockdx = 1.0 / (double)blockdx;
    F3 boff = idx_to_pos(bi, bj, bk, kBW * g.dx);
    for (int t = threadIdx.x; t < total; t += kSdfThreads) {
        int lo = 0, hi = nrows - 1;
        while (lo < hi) {  // last row whose prefix <= t
            int mid = (lo + hi + 1) >> 1;
            if (run_prefix[mid] <= t) lo = mid; else hi = mid - 1;
        }
        int q = run_begin[lo] + (t - run_prefix[lo]);
        const float4 p4 = spos[q];
        F3 p0 = f3(p4.x, p4.y, p4.z);
        if (!point_in_block(p0, sr, blockdx, inv_blockdx, bi, bj, bk)) continue;
        F3 p = p0 - boff;
        I3 gmin = pos_to_index((double)(p.x - sr), (double)(p.y - sr), (double)(p.z - sr), g.invdx);
        I3 gmax = pos_to_index((double)(p.x + sr), (double)(p.y + sr), (double)(p.z + sr), g.invdx);
        gmin.i = max(gmin.i, 0); gmin.j = max(gmin.j, 0); gmin.k = max(gmin.k, 0);
        gmax.i = min(gmax.i, kBW - 1); gmax.j = min(gmax.j, kBW - 1); gmax.k = min(gmax.k, kBW - 1);
        for (int k = gmin.k; k <= gmax.k; k++) {
            float cz = centre[k];
            for (int j = gmin.j; j <= gmax.j; j++) {
                float cy = centre[j];
                for (int i = gmin.i; i <= gmax.i; i++) {
                    F3 c = f3(centre[i], cy, cz);
                    F3 dv = c - p;
                    float d2 = dot3(dv, dv);
                    // Values only fall, so a distance no smaller than the
                    // value already there cannot change it.  A squared
                    // distance clearly beyond (value + r)^2 (margins of 2e-5
                    // relative cover every rounding of the exact test) skips
                    // the square root; otherwise the exact distance decides.
                    uint32_t *slot = &phi_ord[i + kBW * (j + kBW * k)];
                    uint32_t cur = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    float lim = ord2f(cur) + r * 1.00002f;
                    if (lim > 0.0f && d2 > lim * lim * 1.00002f) continue;
                    float dist = sqrtf(d2) - r;
                    uint32_t o = f2ord(dist);
                    if (o < cur) atomicMin(slot, o);
                }
            }
        }
    }
    __syncthreads();

    // Write back, fused with the post-processing pass when a solid is given
    // (calculateSignedDistanceField alone otherwise).
    for (int c = threadIdx.x; c < kBW * kBW * kBW; c += kSdfThreads) {
        int li = c % kBW, lj = (c / kBW) % kBW, lk = c / (kBW * kBW);
        int i = bi * kBW + li, j = bj * kBW + lj, k = bk * kBW + lk;
        if (i >= g.I || j >= g.J || k >= g.K) continue;
        float v = ord2f(phi_ord[c]);
        if (solid) v = postprocess_phi(g, solid, i, j, k, v);
        phi_out[(size_t)i + (size_t)g.I * ((size_t)j + (size_t)g.J * k)] = v;
    }
}

// The signed distance by cells, for search radii under two cells (the
// simulation's 2 r = sqrt(3) dx among them): one thread per cell looks for
// its nearest particle among the half-cells around its centre, nearest
// half-cells first, and stops when no half-cell left can hold a nearer one.
// Rounding keeps order (sqrtf and the subtraction of r are monotonic), so
// min_p (|c - p| - r) is formed from the smallest squared distance alone.
//
// A cell of the liquid is settled by the eight half-cells that meet at its
// centre (about eight particles), where the particle-by-particle pass above
// folds every particle into up to 125 cells and a small scene is a handful of
// its blocks.  256x128x128 double dam break (9.4 M particles): 1767 -> 410 us;
// 37x22x30 (8 k cells): 841 -> 62 us.  Bound by the latency of the dependent
// loads (half-cell offsets, then particles), so no LDS limits the wavefronts
// in flight.
constexpr int kTileI = 16, kTileJ = 4, kTileK = 4;  // cells of a workgroup
static_assert(kTileI * kTileJ * kTileK == kSdfThreads, "one thread per cell");
static_assert(4 * (kTileJ + 4) * (kTileK + 4) == kSdfThreads, "one half-cell row per thread");

struct CellSdfArgs {
    GridGeom g;
    const float4 *spos;
    const int *sub_offset;
    const float *solid;
    float *phi;
    float radius;
    // Distances below, in cells: a half-cell `ring` half-cells away holds no
    // particle nearer than ring / 2 - margin (the margin covers every float
    // rounding of positions and distances); a particle nearer than `sure` is
    // in reach of the cell whatever the rounding, and one further along an
    // axis than `possible` is not.
    float margin, sure, possible;
    int nti, ntj;          // workgroup tiles along i and j
    unsigned ntiles, nblocks;
};

__global__ __launch_bounds__(kSdfThreads) void k_cell_sdf(CellSdfArgs a) {
    const GridGeom &g = a.g;
    // The blocks of one XCD take one contiguous eighth of the tiles, so
    // neighbouring cells, which read the same particles, share an L2.
    const unsigned tile = (blockIdx.x & 7u) * (a.nblocks >> 3) + (blockIdx.x >> 3);
    if (tile >= a.ntiles) return;
    const int ti = (int)(tile % (unsigned)a.nti), tjk = (int)(tile / (unsigned)a.nti);
    const int i0 = ti * kTileI, j0 = (tjk % a.ntj) * kTileJ, k0 = (tjk / a.ntj) * kTileK;
    const int SI = 2 * g.I, SJ = 2 * g.J, SK = 2 * g.K;
    const int i = i0 + (int)(threadIdx.x & 15u), j = j0 + (int)((threadIdx.x >> 4) & 3u);
    const int k = k0 + (int)(threadIdx.x >> 6);
    const bool in = i < g.I && j < g.J && k < g.K;

    // A tile with no particle within reach of any of its cells is air.
    int any = 0;
    {
        const int sy = 2 * j0 - 4 + (int)(threadIdx.x & 15u), sz = 2 * k0 - 4 + (int)(threadIdx.x >> 4);
        if (sy >= 0 && sz >= 0 && sy < SJ && sz < SK) {
            const size_t row = (size_t)SI * ((size_t)sy + (size_t)SJ * (size_t)sz);
            any = a.sub_offset[row + (size_t)max(2 * i0 - 4, 0)] <
                  a.sub_offset[row + (size_t)min(2 * (i0 + kTileI) + 4, SI)];
        }
    }
    any = __syncthreads_or(any);
    if (!in) return;

    const float dx = (float)g.dx, r = a.radius, sr = 2.0f * r;
    const float maxd = (float)(3.0 * g.dx);  // particlelevelset.cpp:295-297
    float best = (maxd + r) * 1.0001f;
    best *= best;  // squared distances from here up leave phi at maxd
    if (any) {
        const int bi = i / kBW, bj = j / kBW, bk = k / kBW;
        const F3 boff = idx_to_pos(bi, bj, bk, kBW * g.dx);
        const F3 c = f3(idx_to_center1(i - bi * kBW, g.dx), idx_to_center1(j - bj * kBW, g.dx),
                        idx_to_center1(k - bk * kBW, g.dx));
        const float sure2 = (a.sure * dx) * (a.sure * dx), possible = a.possible * dx;
        // Whether the reference folds the particle at p0 (block-local p) into
        // this cell: its assignment to the cell's block and its index range.
        auto reaches = [&](F3 p0, F3 p) -> bool {
            const float blockdx = (float)(kBW * g.dx);
            if (!point_in_block(p0, sr, blockdx, 1.0 / (double)blockdx, bi, bj, bk)) return false;
            const I3 lo = pos_to_index((double)(p.x - sr), (double)(p.y - sr), (double)(p.z - sr), g.invdx);
            const I3 hi = pos_to_index((double)(p.x + sr), (double)(p.y + sr), (double)(p.z + sr), g.invdx);
            const int li = i - bi * kBW, lj = j - bj * kBW, lk = k - bk * kBW;
            return li >= lo.i && li <= hi.i && lj >= lo.j && lj <= hi.j && lk >= lo.k && lk <= hi.k;
        };
        auto fold = [&](float4 p4) {
            const F3 p0 = f3(p4.x, p4.y, p4.z);
            const F3 p = p0 - boff;
            const F3 dv = c - p;
            const float d2 = dot3(dv, dv);
            if (!(d2 < best)) return;
            if (d2 < sure2 ||
                (fmaxf(fmaxf(fabsf(dv.x), fabsf(dv.y)), fabsf(dv.z)) < possible && reaches(p0, p)))
                best = d2;
        };
        // Particles of half-cells [2 i - ext, 2 i + 1 + ext] of row (oy, oz).
        auto run = [&](int oy, int oz, int ext, int &b, int &e) {
            const int sy = 2 * j + oy, sz = 2 * k + oz;
            b = e = 0;
            if (sy < 0 || sz < 0 || sy >= SJ || sz >= SK) return;
            const size_t row = (size_t)SI * ((size_t)sy + (size_t)SJ * (size_t)sz);
            b = a.sub_offset[row + (size_t)max(2 * i - ext, 0)];
            e = a.sub_offset[row + (size_t)min(2 * i + 2 + ext, SI)];
        };
        // Folds four rows: their first two particles each are loaded
        // together, before any is used.
        auto fold_rows = [&](const int (&b)[4], const int (&e)[4]) {
            float4 p[4][2];
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int u = 0; u < 2; u++)
                    if (b[q] + u < e[q]) p[q][u] = a.spos[b[q] + u];
#pragma unroll
            for (int q = 0; q < 4; q++) {
#pragma unroll
                for (int u = 0; u < 2; u++)
                    if (b[q] + u < e[q]) fold(p[q][u]);
                for (int t = b[q] + 2; t < e[q]; t += 4) {
                    float4 m[4];
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (t + u < e[q]) m[u] = a.spos[t + u];
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (t + u < e[q]) fold(m[u]);
                }
            }
        };
        int b[4], e[4];
        // The eight half-cells around the centre.
#pragma unroll
        for (int q = 0; q < 4; q++) run(q & 1, q >> 1, 0, b[q], e[q]);
        fold_rows(b, e);
        // Then the rows by distance, four at a time, each over the half-cells
        // that can still hold a nearer particle.
        auto ring = [&](int n) { return fmaxf(0.5f * (float)n - a.margin, 0.0f) * dx; };
        const float near = ring(1);
        if (best > near * near) {
            const float inv = 2.0f / dx;
            for (int q0 = 0; q0 < kCellRows; q0 += 4) {
                bool open = false;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const CellRow cr = c_cell_rows.r[q0 + q];
                    const float dy = ring(cr.ry), dz = ring(cr.rz);
                    const float left = best - (dy * dy + dz * dz);
                    b[q] = e[q] = 0;
                    if (!(left > 0.0f)) continue;
                    open = true;
                    run(cr.oy, cr.oz, min((int)(sqrtf(left) * inv + 2.0f * a.margin), 4), b[q], e[q]);
                }
                if (!open) break;  // so are all rows after these
                fold_rows(b, e);
            }
        }
    }
    float v = sqrtf(best) - r;
    v = v < maxd ? v : maxd;
    if (a.solid) v = postprocess_phi(g, a.solid, i, j, k, v);
    a.phi[(size_t)i + (size_t)g.I * ((size_t)j + (size_t)g.J * k)] = v;
}

// The post-processing pass on its own, over an existing field (one thread
// per cell).
__global__ void k_liquid_postprocess(GridGeom g, const float *__restrict__ solid, float *phi) {
    size_t n = (size_t)g.I * g.J * g.K;
    size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    int i = (int)(c % (size_t)g.I), j = (int)((c / (size_t)g.I) % (size_t)g.J), k = (int)(c / ((size_t)g.I * g.J));
    phi[c] = postprocess_phi(g, solid, i, j, k, phi[c]);
}

hipError_t launch_liquid_postprocess(const GridGeom &g, const float *solid_phi_nodal, float *phi,
                                     hipStream_t s) {
    size_t n = (size_t)g.I * g.J * g.K;
    if (n == 0) return hipSuccess;
    k_liquid_postprocess<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(g, solid_phi_nodal, phi);
    return hipGetLastError();
}

hipError_t launch_liquid_sdf(const GridGeom &g, const float4 *spos, const int *sub_offset, double radius,
                             const float *solid_phi_nodal, float *phi, hipStream_t s) {
    // A cell's particles lie within 2 r + dx / 2 of its centre along each
    // axis: under 2.5 cells, the half-cells that k_cell_sdf walks, while 2 r
    // is below two cells.  Larger (and non-positive) radii keep the pass by
    // particles, whose candidates are its block's and two cells around it.
    const double reach = 2.0 * radius / g.dx;
    if (reach > 0.0 && reach < 1.99) {
        CellSdfArgs a{};
        a.g = g;
        a.spos = spos;
        a.sub_offset = sub_offset;
        a.solid = solid_phi_nodal;
        a.phi = phi;
        a.radius = (float)radius;
        // On a grid of at most 4096 cells along each axis a coordinate is
        // below 2^12 dx, so one float rounding moves it by at most 2^-12 dx,
        // and a distance or a test rounds at most four times: 0.001 dx.  On
        // larger grids every half-cell in reach is walked and every particle
        // tested.
        const bool small_grid = g.I <= 4096 && g.J <= 4096 && g.K <= 4096;
        a.margin = small_grid ? 0.01f : 16.0f;
        a.sure = small_grid ? (float)(reach + 0.5 - 0.01) : 0.0f;
        a.possible = small_grid ? (float)(reach + 0.5 + 0.01) : 1e30f;
        a.nti = (g.I + kTileI - 1) / kTileI;
        a.ntj = (g.J + kTileJ - 1) / kTileJ;
        a.ntiles = (unsigned)a.nti * (unsigned)a.ntj * (unsigned)((g.K + kTileK - 1) / kTileK);
        a.nblocks = (a.ntiles + 7u) / 8u * 8u;
        k_cell_sdf<<<a.nblocks, kSdfThreads, 0, s>>>(a);
        return hipGetLastError();
    }
    int nbi = (g.I + kBW - 1) / kBW, nbj = (g.J + kBW - 1) / kBW, nbk = (g.K + kBW - 1) / kBW;
    k_liquid_sdf<<<nbi * nbj * nbk, kSdfThreads, 0, s>>>(g, spos, sub_offset, (float)radius, solid_phi_nodal,
                                                         phi);
    return hipGetLastError();
}

}  // namespace flipmi
