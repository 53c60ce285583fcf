// Device code shared by the pressure solvers (k_pressure.hip, k_multigrid.hip):
// the assembly of one row and the split of work lists over the XCDs.
#pragma once

#include "device_math.h"
#include "flipmi_kernels.h"

namespace flipmi {

constexpr double kMaxTheta = 25.0;  // pressuresolver.h:163

// A coupling entry of the matrix from the face weight it is formed from:
// -weight * dt / dx^2, the product the assembly takes (pressuresolver.cpp:
// 725, 753-798), so the FP64 entry comes out bit for bit.  A slot without
// the coupling holds -0.0f, which gives the +0.0 it stands for.
__device__ __forceinline__ double coupling(float w, double mf) { return -(double)w * mf; }

__device__ __forceinline__ bool interior(const GridGeom &g, int i, int j, int k) {
    return i >= 1 && j >= 1 && k >= 1 && i <= g.I - 2 && j <= g.J - 2 && k <= g.K - 2;
}

__device__ __forceinline__ bool is_row_cell(const GridGeom &g, const float *liquid, int i, int j,
                                            int k) {
    if (!interior(g, i, j, k)) return false;
    return liquid[(size_t)i + (size_t)g.I * ((size_t)j + (size_t)g.J * k)] < 0;
}

// One row of the system: right-hand side (pressuresolver.cpp:580-669) and
// matrix coefficients (pressuresolver.cpp:723-808).  Couplings to the
// +x/+y/+z rows are kept as the face weight they are formed from (entry =
// -weight * mf); -0.0f stands for "no coupling" (entry +0.0).  `coupled` is
// the sum of the face weights towards all six neighbouring rows.
struct AssembleInputs {
    const float *liquid, *wU, *wV, *wW, *wC, *u, *v, *w, *sU, *sV, *sW;
};
struct PressureRow {
    double rhs = 0, diag = 0, coupled = 0;
    float wx = -0.0f, wy = -0.0f, wz = -0.0f;
};
__device__ __forceinline__ PressureRow assemble_row(const GridGeom &g, double mf, const AssembleInputs &in, int i,
                                                    int j, int k) {
    const float *__restrict__ liquid = in.liquid;
    const float *__restrict__ wU = in.wU, *__restrict__ wV = in.wV, *__restrict__ wW = in.wW;
    const float *__restrict__ wC = in.wC;
    const float *__restrict__ u = in.u, *__restrict__ v = in.v, *__restrict__ w = in.w;
    const float *__restrict__ sU = in.sU, *__restrict__ sV = in.sV, *__restrict__ sW = in.sW;
    PressureRow row;
    size_t c = (size_t)i + (size_t)g.I * ((size_t)j + (size_t)g.J * k);
    Dims DU{g.I + 1, g.J, g.K}, DV{g.I, g.J + 1, g.K}, DW{g.I, g.J, g.K + 1};
    double volCenter = wC[c];
    double volRight = wU[DU.at(i + 1, j, k)], volLeft = wU[DU.at(i, j, k)];
    double volTop = wV[DV.at(i, j + 1, k)], volBottom = wV[DV.at(i, j, k)];
    double volFront = wW[DW.at(i, j, k + 1)], volBack = wW[DW.at(i, j, k)];
    double factor = 1.0 / g.dx;
    double div = 0.0;
    div += -factor * volRight * u[DU.at(i + 1, j, k)];
    div += factor * volLeft * u[DU.at(i, j, k)];
    div += -factor * volTop * v[DV.at(i, j + 1, k)];
    div += factor * volBottom * v[DV.at(i, j, k)];
    div += -factor * volFront * w[DW.at(i, j, k + 1)];
    div += factor * volBack * w[DW.at(i, j, k)];
    div += factor * (volRight - volCenter) * sU[DU.at(i + 1, j, k)];
    div += -factor * (volLeft - volCenter) * sU[DU.at(i, j, k)];
    div += factor * (volTop - volCenter) * sV[DV.at(i, j + 1, k)];
    div += -factor * (volBottom - volCenter) * sV[DV.at(i, j, k)];
    div += factor * (volFront - volCenter) * sW[DW.at(i, j, k + 1)];
    div += -factor * (volBack - volCenter) * sW[DW.at(i, j, k)];
    row.rhs = div;

    double eps = 1e-9;
    double pc = liquid[c];
    double diag = (volRight + volLeft + volTop + volBottom + volFront + volBack) * mf;
    auto side = [&](double vol, int a, int b, int d, float *off) {
        double pn = liquid[(size_t)a + (size_t)g.I * ((size_t)b + (size_t)g.J * d)];
        if (pn < 0.0) {
            // vol is a float weight widened: (float)vol is exact.
            if (!is_row_cell(g, liquid, a, b, d)) return;
            row.coupled += vol;
            if (off) *off = (float)vol;
        } else {
            double theta = pn / (pc + eps);
            theta = theta < -kMaxTheta ? -kMaxTheta : (theta > kMaxTheta ? kMaxTheta : theta);
            diag -= vol * mf * theta;
        }
    };
    side(volRight, i + 1, j, k, &row.wx);
    side(volLeft, i - 1, j, k, nullptr);
    side(volTop, i, j + 1, k, &row.wy);
    side(volBottom, i, j - 1, k, nullptr);
    side(volFront, i, j, k + 1, &row.wz);
    side(volBack, i, j, k - 1, nullptr);
    row.diag = diag > 0.0 ? diag : 0.0;
    return row;
}

// Blocks are dispatched to the eight XCDs round-robin (block b on XCD b %
// 8).  Entries of a work list for this block: the blocks of one XCD take one
// contiguous eighth of the list, so what neighbouring entries share sits in
// the same L2.  Any other placement only costs locality.  gridDim.x is a
// multiple of kXcds.
constexpr unsigned kXcds = 8;
struct ListRange {
    int begin, end, step;
};
__device__ __forceinline__ ListRange xcd_list(int n) {
    const int x = (int)(blockIdx.x % kXcds), l = (int)(blockIdx.x / kXcds);
    const int part = (n + (int)kXcds - 1) / (int)kXcds;
    const int b = x * part, e = b + part < n ? b + part : n;
    return ListRange{b + l, e, (int)(gridDim.x / kXcds)};
}
}  // namespace flipmi
