// flux_face.hpp -- the ideal-gas face-flux kernel of the face-per-thread path, shared by
// the translation units that instantiate it (flux_face_<dims>_<numerics>.hip, one per
// dimension and numerics so that they compile in parallel).
#pragma once
#include <hip/hip_runtime.h>

#include "block.hpp"
#include "gdtk_device.hpp"
#include "kernel_common.hpp"

namespace gdtk {

// One thread per face of index direction d: reconstruction + flux calculator, or the
// simple-outflow boundary flux effect on faces whose BC computes the flux itself.  The block
// and the direction are the same for the whole workgroup, so every plane is a scalar base and
// the lane's index a 32-bit offset from that of the wave's first lane.  Small launches are bound
// by their instructions and by the latency of their loads (4 waves a SIMD at 128 registers),
// large ones by the bytes too (256 x 128 x 128 cells along the axes: 152 B a face beyond L2 at
// 4.97 TB/s, a copy's rate, with the VALU 57 % busy): scalar bases, divisions through the refined
// hardware reciprocal and index divisions by multiplication took the launch over a 2-D tube of
// 200 x 100 cells from 7.0 to 5.2 us, over 97 x 75 x 63 curvilinear cells (EFM) from 64 to 59 us.
//
// AXIS: a direction whose faces all have the same axis-aligned frame.  The velocity components
// are loaded, and the momentum fluxes stored, in the frame's order, and the nine planes of
// frames are not read (72 of a face's 176 bytes) nor multiplied with (135 operations): 128^3 cells
// 273 -> 187 us, with the changes above.  Not for
// EFM, whose error function has its sign from a velocity that may be a signed zero, which the
// rotations' added zeros decide.
template <int DIM, int FC, bool LMR, bool AXIS>
__device__ __forceinline__ void face_flux_one(const BlockDev& b, const IdealGasDev& gas, int d, double eps,
                                              unsigned f) {
    using C = CQ<DIM>;
    unsigned fi, fj;
    const unsigned rest = b.fdiv[d][0].divmod(f, fi);
    const unsigned fk = b.fdiv[d][1].divmod(rest, fj);
    const int64_t np = b.npad;
    const int pos = (int)((d == 0) ? fi : (d == 1) ? fj : fk);
    const int nd = (d == 0) ? b.nic : (d == 1) ? b.njc : b.nkc;
    const unsigned stride = (d == 0) ? 1u : (d == 1) ? (unsigned)b.NI : (unsigned)(b.NI * b.NJ);
    // the cell on the face's right, and the stencil around the face
    const unsigned cabs = (fi + NGHOST) + (unsigned)b.NI * ((fj + NGHOST) + (unsigned)b.NJ * (fk + (DIM == 3 ? NGHOST : 0)));
    const unsigned oc = wave_origin(cabs - 2 * stride);
    const unsigned cL1 = cabs - 2 * stride - oc, cL0 = cL1 + stride, cR0 = cL0 + stride, cR1 = cR0 + stride;
    const double* fs = b.fs_in + oc;
    const int64_t nfc = b.nface[d];
    double F[C::n];
    const int side = (pos == 0) ? 2 * d : (pos == nd) ? 2 * d + 1 : -1;
    const unsigned of = wave_origin(f);
    f -= of;
    double* out = b.flux[d] + of;
    auto load_frame = [&] {
        const double* q = b.fgeom[d] + of;
        FaceGeom g;
        g.n = Vec3d{ld_plane(q, f), ld_plane(q + nfc, f), ld_plane(q + 2 * nfc, f)};
        g.t1 = Vec3d{ld_plane(q + 3 * nfc, f), ld_plane(q + 4 * nfc, f), ld_plane(q + 5 * nfc, f)};
        g.t2 = Vec3d{ld_plane(q + 6 * nfc, f), ld_plane(q + 7 * nfc, f), ld_plane(q + 8 * nfc, f)};
        g.area = 0.0;  // not used by the flux
        return g;
    };
    if (side >= 0 && b.bc_kind[side] == BC_OUTFLOW_SIMPLE_FLUX) {
        const int outsign = (side % 2 == 0) ? -1 : 1;
        const unsigned c = (side % 2 == 0) ? cR0 : cL0;
        const Vec3d v{ld_plane(fs + FS_VX * np, c), ld_plane(fs + FS_VY * np, c), ld_plane(fs + FS_VZ * np, c)};
        outflow_flux<DIM>(load_frame(), outsign, ld_plane(fs + FS_RHO * np, c), ld_plane(fs + FS_U * np, c),
                          ld_plane(fs + FS_P * np, c), v, F);
#pragma unroll
        for (int j = 0; j < C::n; ++j) st_plane(out + j * nfc, f, F[j]);
        return;
    }
    const double* len = b.len + d * np + oc;
    int ax[3] = {0, 1, 2};
    double sg[3] = {1.0, 1.0, 1.0};
    FaceGeom g{};
    if (AXIS) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            ax[q] = b.axis[d][q] & 3;
            sg[q] = (b.axis[d][q] & 4) ? -1.0 : 1.0;
        }
    } else {
        g = load_frame();
    }
    auto load = [&](unsigned c) {
        StencilCell s;
        s.rho = ld_plane(fs + FS_RHO * np, c);
        s.u = ld_plane(fs + FS_U * np, c);
        s.vel.x = sg[0] * ld_plane(fs + (FS_VX + ax[0]) * np, c);
        s.vel.y = sg[1] * ld_plane(fs + (FS_VX + ax[1]) * np, c);
        s.vel.z = sg[2] * ld_plane(fs + (FS_VX + ax[2]) * np, c);
        return s;
    };
    const StencilCell L1 = load(cL1), L0 = load(cL0), R0 = load(cR0), R1 = load(cR1);
    const FallbackFS fb{fs, np, (int64_t)cL0, (int64_t)cR0};
    // Adaptive calculator: EFM or Hanel where the face is shocked (strict rule), else AUSMDV.
    const bool shocked = flux_is_adaptive(FC) && ((b.shock[oc + cL0] | b.shock[oc + cR0]) != 0);
    face_flux_l2r2<DIM, FC, LMR, AXIS>(gas, g, L1, L0, R0, R1, ld_plane(fs + FS_A * np, cL0),
                                       ld_plane(fs + FS_A * np, cR0), fb, ld_plane(len, cL1), ld_plane(len, cL0),
                                       ld_plane(len, cR0), ld_plane(len, cR1), eps, F, shocked);
    st_plane(out + C::mass * nfc, f, F[C::mass]);
    st_plane(out + C::totEnergy * nfc, f, F[C::totEnergy]);
    const double m[3] = {F[C::xMom], F[C::yMom], (DIM == 3) ? F[C::zMom] : 0.0};
#pragma unroll
    for (int q = 0; q < 3; ++q)
        if (DIM == 3 || ax[q] < 2) st_plane(out + (C::xMom + ax[q]) * nfc, f, sg[q] * m[q]);
}

// Faces of every direction of every block in one launch.  Each block's faces of a direction
// start at a multiple of the workgroup size (FaceBatch), so every workgroup serves one
// direction of one block and reads that block's record with scalar loads.  LMR selects
// Eilmer 5's limiter smoothing and AUSMDV sound speed.
template <int DIM, int FC, bool LMR>
__global__ __launch_bounds__(256, 4) void k_face_flux_batch(const BlockDev* __restrict__ tab, FaceBatch fb,
                                                         int nblocks, double eps, IdealGasDev gas) {
    int64_t w0 = (int64_t)blockIdx.x * blockDim.x;
    const int d = __builtin_amdgcn_readfirstlane(face_batch_dir(fb, w0));
    const int64_t* __restrict__ start = fb.start[d];
    int lo = 0, hi = nblocks - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (start[mid] <= w0) lo = mid;
        else hi = mid - 1;
    }
    const int q = __builtin_amdgcn_readfirstlane(lo);
    const BlockDev& b = tab[q];
    const int64_t f = w0 - start[q] + threadIdx.x;
    if (f >= b.nface[d]) return;
    if (FC != 1 && FC != 2 && b.axis[d][0] >= 0) face_flux_one<DIM, FC, LMR, true>(b, gas, d, eps, (unsigned)f);
    else face_flux_one<DIM, FC, LMR, false>(b, gas, d, eps, (unsigned)f);
}

// Launchers of k_face_flux_batch<DIM, FC, LMR> for each dimension and numerics (defined in
// flux_face_<dims>_<numerics>.hip); flux_calc selects FC.
hipError_t launch_face_flux_3d_e4(const BlockDev* tab, const FaceBatch& fb, int nblocks, int flux_calc, double eps,
                                  const IdealGasDev& gas, int64_t total, hipStream_t s);
hipError_t launch_face_flux_2d_e4(const BlockDev* tab, const FaceBatch& fb, int nblocks, int flux_calc, double eps,
                                  const IdealGasDev& gas, int64_t total, hipStream_t s);
hipError_t launch_face_flux_3d_lmr(const BlockDev* tab, const FaceBatch& fb, int nblocks, int flux_calc, double eps,
                                   const IdealGasDev& gas, int64_t total, hipStream_t s);
hipError_t launch_face_flux_2d_lmr(const BlockDev* tab, const FaceBatch& fb, int nblocks, int flux_calc, double eps,
                                   const IdealGasDev& gas, int64_t total, hipStream_t s);

// Instantiates and launches k_face_flux_batch<DIM, FC, LMR> for the flux calculator code.
template <int DIM, bool LMR>
hipError_t launch_face_flux_fc(const BlockDev* tab, const FaceBatch& fb, int nblocks, int flux_calc, double eps,
                               const IdealGasDev& gas, int64_t total, hipStream_t s) {
    dim3 grid((unsigned)((total + 255) / 256)), blk(256);
#define GDTK_FACE(F) hipLaunchKernelGGL((k_face_flux_batch<DIM, F, LMR>), grid, blk, 0, s, tab, fb, nblocks, eps, gas)
    if (flux_calc == 4) GDTK_FACE(4);
    else if (flux_calc == 3) GDTK_FACE(3);
    else if (flux_calc == 2) GDTK_FACE(2);
    else if (flux_calc == 1) GDTK_FACE(1);
    else GDTK_FACE(0);
#undef GDTK_FACE
    return hipGetLastError();
}

}  // namespace gdtk
