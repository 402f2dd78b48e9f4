// kernel_common.hpp -- device helpers shared by the face-per-thread and fused kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "block.hpp"
#include "gdtk_device.hpp"

namespace gdtk {

__device__ __forceinline__ FaceGeom load_face(const double* g, int64_t nface, int64_t f) {
    FaceGeom r;
    r.n.x = g[f];
    r.n.y = g[f + nface];
    r.n.z = g[f + 2 * nface];
    r.t1.x = g[f + 3 * nface];
    r.t1.y = g[f + 4 * nface];
    r.t1.z = g[f + 5 * nface];
    r.t2.x = g[f + 6 * nface];
    r.t2.y = g[f + 7 * nface];
    r.t2.z = g[f + 8 * nface];
    r.area = g[f + 9 * nface];
    return r;
}

__device__ __forceinline__ int64_t face_index(const BlockDev& b, int d, int fi, int fj, int fk) {
    return (int64_t)fi + (int64_t)b.nf[d][0] * ((int64_t)fj + (int64_t)b.nf[d][1] * (int64_t)fk);
}

__device__ __forceinline__ StencilCell load_sc(const double* fs, int64_t np, int64_t c) {
    StencilCell s;
    s.rho = fs[c + FS_RHO * np];
    s.u = fs[c + FS_U * np];
    s.vel.x = fs[c + FS_VX * np];
    s.vel.y = fs[c + FS_VY * np];
    s.vel.z = fs[c + FS_VZ * np];
    return s;
}

// The ghost cells that copy a cell, written with its new state v (plane order) by the thread that
// has it, as k_ghost_fill does: h is the first record's index (BlockDev::ghead), or -1.
template <int NFS>
__device__ __forceinline__ void push_ghosts(const GhostRec* __restrict__ rec, int h, const double (&v)[NFS]) {
    while (h >= 0) {
        const GhostRec r = rec[h];
        Vec3d w{v[FS_VX], v[FS_VY], v[FS_VZ]};
        if (r.wall) {
            // ghost_cell.d:33-43
            const FaceGeom fg = load_face(r.wall, r.nface, 0);
            Vec3d l = to_local(w, fg);
            l.x = -(l.x);
            w = to_global(l, fg);
        }
#pragma unroll
        for (int f = 0; f < NFS; ++f)
            r.dst[(int64_t)f * r.npd] = (f == FS_VX) ? w.x : (f == FS_VY) ? w.y : (f == FS_VZ) ? w.z : v[f];
        h = r.next;
    }
}

// The first ghost record of interior cell (i, j) of a 2-D block, at padded index c.  Ghost cells
// copy cells within NGHOST of a side, so no other cell has its entry read.
__device__ __forceinline__ int ghost_head(const BlockDev& b, int i, int j, unsigned c) {
    const bool near = i < NGHOST || i >= b.nic - NGHOST || j < NGHOST || j >= b.njc - NGHOST;
    return near ? b.ghead[c] : -1;
}

// Stage update and decode of one cell from its surface integrals si[] (fvcell.d:824-854,
// simcore_gasdynamic_step.d:1225-1321, fvcell.d:586-821, fluidblock.d:607-676).
template <int DIM, int STAGE>
__device__ __forceinline__ void update_decode_store(const BlockDev& b, const IdealGasDev& gas, unsigned c,
                                                    const double* si, double dt, double low_T, double max_vel,
                                                    double min_T, double max_T, const GhostRec* push = nullptr,
                                                    int head = -1) {
    using C = CQ<DIM>;
    const int64_t np = b.npad;
    const unsigned o = wave_origin(c);  // cells come in the lanes' order
    c -= o;
    const double vol_inv = quick_rcp(ld_plane(b.vol + o, c));
    double U[C::n];
#pragma unroll
    for (int jq = 0; jq < C::n; ++jq) {
        const double dUdt = vol_inv * si[jq] + 0.0;
        const double u0 = ld_plane(b.U0 + jq * np + o, c);
        if (STAGE == 1) {
            const double gamma_1 = 1.0;
            st_plane(b.dUdt0 + jq * np + o, c, dUdt);
            U[jq] = u0 + dt * gamma_1 * dUdt;
        } else {
            const double gamma_1 = 0.5, gamma_2 = 0.5;
            U[jq] = u0 + dt * (gamma_1 * ld_plane(b.dUdt0 + jq * np + o, c) + gamma_2 * dUdt);
        }
    }
    double rho, u, p, T, a;
    Vec3d vel;
    bool reenc;
    int bad = decode_ideal<DIM>(gas, U, low_T, rho, vel, u, p, T, a, reenc);
    double* fo = b.fs_out + o;
    if (bad) {
        atomicAdd(&b.counters[0], 1);
        if (push) {  // the ghosts copy what the cell keeps
            double v[FS_BASE_PLANES];
#pragma unroll
            for (int f = 0; f < FS_BASE_PLANES; ++f) v[f] = ld_plane(fo + f * np, c);
            push_ghosts<FS_BASE_PLANES>(push, head, v);
        }
        return;
    }
    if (STAGE == 2)
#pragma unroll
        for (int jq = 0; jq < C::n; ++jq) st_plane(b.Unew + jq * np + o, c, U[jq]);
    st_plane(fo + FS_RHO * np, c, rho);
    st_plane(fo + FS_VX * np, c, vel.x);
    st_plane(fo + FS_VY * np, c, vel.y);
    st_plane(fo + FS_VZ * np, c, vel.z);
    st_plane(fo + FS_U * np, c, u);
    st_plane(fo + FS_P * np, c, p);
    st_plane(fo + FS_T * np, c, T);
    st_plane(fo + FS_A * np, c, a);
    if (push) {
        const double v[FS_BASE_PLANES] = {rho, vel.x, vel.y, vel.z, u, p, T, a};
        push_ghosts<FS_BASE_PLANES>(push, head, v);
    }
    if (!check_data(rho, p, T, a, vel, max_vel, min_T, max_T)) atomicAdd(&b.counters[1], 1);
}

}  // namespace gdtk
