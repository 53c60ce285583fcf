// Memory-bound grid passes: fills, velocity extrapolation, saving the MAC
// grid with the body force, and the solid velocity constraint.
#include <algorithm>

#include "device_math.h"
#include "flipmi_kernels.h"
#include "inflow_device.h"

namespace flipmi {

template <class T>
__global__ void k_fill(T *p, size_t n, T v) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

template <class T>
static hipError_t fill(T *p, size_t n, T v, hipStream_t s) {
    if (n == 0) return hipSuccess;
    size_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    k_fill<T><<<(unsigned)blocks, 256, 0, s>>>(p, n, v);
    return hipGetLastError();
}

hipError_t launch_fill_u8(uint8_t *p, size_t n, uint8_t v, hipStream_t s) { return fill(p, n, v, s); }
hipError_t launch_fill_f32(float *p, size_t n, float v, hipStream_t s) { return fill(p, n, v, s); }
hipError_t launch_fill_f64(double *p, size_t n, double v, hipStream_t s) { return fill(p, n, v, s); }
hipError_t launch_fill_i32(int *p, size_t n, int v, hipStream_t s) { return fill(p, n, v, s); }

// Extrapolation status codes: 0 = valid on entry, L = filled in layer L,
// kBorder = face on the grid border (always finished, never a source),
// kUnknown = not reached yet.
constexpr uint8_t kBorder = 254;
constexpr uint8_t kUnknown = 255;

// Both kernels take four consecutive faces (one word of status bytes) a
// thread and one component a blockIdx.y.  On small grids launches count (a
// layer of one component took 4.2 us at 64^3 and there were 48 launches a time
// step; now 5.3 us for all three components and 16 launches), on large ones the
// instructions per face: most words hold no unreached face, or none next to
// the last layer, and are done after one to seven loads.  The three
// components' layer took 42.7 us with a thread per face on 320x160x160 and
// takes 19.3; sixteen faces a thread took 26.7 there, and 13.7 against 5.3 at
// 64^3 (too few waves for the loads' latency).
struct ExtrapolateFields {
    ExtrapolateField f[3];
};

// 0x80 in every byte of v that equals c.
__device__ __forceinline__ unsigned bytes_equal(unsigned v, unsigned c) {
    const unsigned x = v ^ (c * 0x01010101u);
    return ~(((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x | 0x7f7f7f7fu);
}
// The four bytes at p, at any alignment.
__device__ __forceinline__ unsigned load_bytes(const uint8_t *p) {
    unsigned v;
    __builtin_memcpy(&v, p, 4);
    return v;
}

__global__ __launch_bounds__(256) void k_extrap_init(ExtrapolateFields fs) {
    const ExtrapolateField &f = fs.f[blockIdx.y];
    const unsigned n = (unsigned)f.ni * (unsigned)f.nj * (unsigned)f.nk;
    const unsigned w = 4u * (blockIdx.x * 256u + threadIdx.x);
    if (w >= n) return;
    unsigned valid = 0;
    if (n - w >= 4) {
        valid = load_bytes(f.valid + w);
    } else {
        for (unsigned m = 0; m < n - w; m++) valid |= (unsigned)f.valid[w + m] << (8 * m);
    }
    int i, j, k;
    unflatten3(w, f.ni, f.nj, i, j, k);
    unsigned st = 0;
#pragma unroll
    for (int m = 0; m < 4; m++) {
        // Faces past the end count as border (k reaches nk).
        const bool border = i == 0 || j == 0 || k == 0 || i == f.ni - 1 || j == f.nj - 1 || k >= f.nk - 1;
        const unsigned b = border ? kBorder : ((valid >> (8 * m)) & 255u) ? 0u : kUnknown;
        st |= b << (8 * m);
        if (++i == f.ni) {
            i = 0;
            if (++j == f.nj) {
                j = 0;
                k++;
            }
        }
    }
    *reinterpret_cast<unsigned *>(f.status + w) = st;
}

// One layer of GridUtils::extrapolateGrid (gridutils.cpp:32-228): every
// unreached face next to a face finished in the previous layer takes the
// mean of its finished 6-neighbours, summed in the order +i,-i,+j,-j,+k,-k.
// Faces written in this pass are neither read as sources nor averaged, so
// the in-place update is race free.
__global__ __launch_bounds__(256) void k_extrap_layer(ExtrapolateFields fs, int layer) {
    const ExtrapolateField &f = fs.f[blockIdx.y];
    const unsigned n = (unsigned)f.ni * (unsigned)f.nj * (unsigned)f.nk;
    const unsigned w = 4u * (blockIdx.x * 256u + threadIdx.x);
    if (w >= n) return;
    uint8_t *const st = f.status + w;
    const unsigned own = *reinterpret_cast<const unsigned *>(st);
    const unsigned unknown = bytes_equal(own, kUnknown);
    if (!unknown) return;
    // An unknown face is never on the border, so its 6 neighbours exist; bytes
    // read for the other faces of the word may lie outside by less than
    // kExtrapolatePad and count for nothing.
    const size_t sj = (size_t)f.ni, sk = (size_t)f.ni * (size_t)f.nj;
    const unsigned before = *reinterpret_cast<const unsigned *>(st - 4), after = *reinterpret_cast<const unsigned *>(st + 4);
    const unsigned nb[6] = {(own >> 8) | (after << 24), (own << 8) | (before >> 24), load_bytes(st + sj),
                            load_bytes(st - sj), load_bytes(st + sk), load_bytes(st - sk)};
    const unsigned known = (unsigned)(layer - 1);
    unsigned touch = 0;
#pragma unroll
    for (int q = 0; q < 6; q++) touch |= bytes_equal(nb[q], known);
    touch &= unknown;
    if (!touch) return;
    float *const grid = f.grid + w;
    const ptrdiff_t off[6] = {1, -1, (ptrdiff_t)sj, -(ptrdiff_t)sj, (ptrdiff_t)sk, -(ptrdiff_t)sk};
    // Every value is loaded before the first is used; one that does not count
    // is replaced by the word's first, which exists.
    float v[4][6];
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const bool due = (touch >> (8 * m)) & 0x80u;
#pragma unroll
        for (int q = 0; q < 6; q++) {
            const unsigned s = (nb[q] >> (8 * m)) & 255u;
            v[m][q] = grid[due && (s <= known || s == kBorder) ? m + off[q] : 0];
        }
    }
    unsigned now = own;
#pragma unroll
    for (int m = 0; m < 4; m++) {
        if (!((touch >> (8 * m)) & 0x80u)) continue;
        float sum = 0.0f;
        int count = 0;
#pragma unroll
        for (int q = 0; q < 6; q++) {
            const unsigned s = (nb[q] >> (8 * m)) & 255u;
            if (s <= known || s == kBorder) {
                sum += v[m][q];
                count++;
            }
        }
        grid[m] = sum / (float)count;
        now = (now & ~(255u << (8 * m))) | ((unsigned)layer << (8 * m));
    }
    *reinterpret_cast<unsigned *>(st) = now;
}

hipError_t launch_extrapolate(const ExtrapolateField *fields, int count, int layers, hipStream_t s) {
    ExtrapolateFields fs{};
    size_t most = 0;
    for (int c = 0; c < count; c++) {
        fs.f[c] = fields[c];
        most = std::max(most, (size_t)fields[c].ni * fields[c].nj * fields[c].nk);
    }
    const dim3 nb((unsigned)((most + 1023) / 1024), (unsigned)count);
    k_extrap_init<<<nb, 256, 0, s>>>(fs);
    for (int l = 1; l <= layers; l++) k_extrap_layer<<<nb, 256, 0, s>>>(fs, l);
    return hipGetLastError();
}

// _saveVelocityField + _applyConstantBodyForces (fluidsimulation.cpp:
// 3287-3297, 3450-3489): saved = mac, then mac += (float)(g * dt) on every
// face (no inflow faces are constrained in these scenes).
__global__ void k_save_force(size_t n, float *mac, float *saved, float add, int do_add) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float v = mac[i];
    saved[i] = v;
    if (do_add) mac[i] = v + add;
}

hipError_t launch_save_and_body_force(size_t n, const float *mac, float *saved, float add,
                                      int do_add, hipStream_t s) {
    k_save_force<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, const_cast<float *>(mac), saved,
                                                             add, do_add);
    return hipGetLastError();
}

// The same with the inflow constraint: valid faces held by an inflow source
// take no body force (fluidsimulation.cpp:3372-3438, 3450-3489).  Face
// positions are Grid3d::FaceIndexToPositionU/V/W (grid3d.h:111-133).
__global__ void k_save_force_inflow(GridGeom g, int comp, size_t n, float *mac, float *saved,
                                    float add, int do_add, const uint8_t *__restrict__ valid,
                                    InflowViews views) {
    size_t f = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= n) return;
    float v = mac[f];
    saved[f] = v;
    if (!do_add) return;
    if (valid[f]) {
        const int ni = g.I + (comp == 0), nj = g.J + (comp == 1);
        int i, j, k;
        unflatten3(f, ni, nj, i, j, k);
        F3 p = f3(comp == 0 ? (float)((double)(float)i * g.dx) : (float)(((double)(float)i + 0.5) * g.dx),
                  comp == 1 ? (float)((double)(float)j * g.dx) : (float)(((double)(float)j + 0.5) * g.dx),
                  comp == 2 ? (float)((double)(float)k * g.dx) : (float)(((double)(float)k + 0.5) * g.dx));
        for (int s = 0; s < views.n; s++)
            if (views.v[s].constrain && inflow_holds_face(views.v[s], g, p)) return;
    }
    mac[f] = v + add;
}

hipError_t launch_save_and_body_force_inflow(const GridGeom &g, int comp, const float *mac,
                                             float *saved, float add, int do_add,
                                             const uint8_t *valid, const InflowViews &views,
                                             hipStream_t s) {
    size_t n = (size_t)(g.I + (comp == 0)) * (g.J + (comp == 1)) * (g.K + (comp == 2));
    k_save_force_inflow<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(g, comp, n, const_cast<float *>(mac),
                                                                    saved, add, do_add, valid, views);
    return hipGetLastError();
}

// FluidSimulation::_constrainVelocityFieldThread (fluidsimulation.cpp:3873-3935)
// with the domain boundary's friction f = 0 (fluidsimulation.h:1524).
__global__ void k_constrain(size_t n, float *mac, const float *__restrict__ weight,
                            const float *__restrict__ solid_vel) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float w = weight[i];
    if (w == 0) {
        mac[i] = solid_vel[i];
    } else if (w < 1.0f) {
        const float f = 0.0f;
        mac[i] = f * solid_vel[i] + (1.0f - f) * mac[i];
    }
}

hipError_t launch_constrain(size_t n, float *mac, const float *weight, const float *solid_vel,
                            hipStream_t s) {
    k_constrain<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, mac, weight, solid_vel);
    return hipGetLastError();
}

}  // namespace flipmi
