// gfx950 kernels of the reference-structured path -- one kernel per loop of
// FDTD_PLRCSolver::stepScheme (src/fdtd_plrc.t:127-168): CPML currents, current totals, E
// update, ghost wrap, and the same for the magnetic side -- of the plain / Kerr-only / ADE
// solvers, and of the diagnostics and field output.  The fused kernels are in mpx_fused.hip,
// the pass kernels in mpx_pass.hip, the sweep in mpx_sweep.hip, the source sheets in
// mpx_sheet.hip.  Threads run along z (the contiguous dimension), 64 per wavefront, so every
// field load of a wavefront is one coalesced 256/512-byte segment.
#include <hip/hip_runtime.h>

#include "mpx_device.h"
#include "mpx_launch.h"

namespace mpx {

// ------------------------------------------------------------------------------------
// reference-structured path
// ------------------------------------------------------------------------------------

// CPMLBorderECurrent::stepScheme, src/cpml_border.cpp:398-425
__global__ __launch_bounds__(256) void k_ref_cpml_E(StepArgs<double> a, int fi, FaceCells at)
{
    const CpmlFace &f = a.face[fi];
    int k = at.lo[2] + blockIdx.x * 64 + threadIdx.x;
    int j = at.lo[1] + blockIdx.y * 4 + threadIdx.y;
    int i = at.lo[0] + blockIdx.z;
    if (k > at.hi[2] || j > at.hi[1]) return;
    int ind[3] = {i, j, k};
    int m[3] = {i, j, k};
    m[f.dim] -= 1;
    int q = ind[f.dim] - f.lo[f.dim];
    const GridDims &g = a.g;
    size_t c = g.at(i, j, k), cm = g.at(m[0], m[1], m[2]);
    const double *B0 = a.B[f.f0], *B1 = a.B[f.f1];
    double *p0 = (double *)f.psi0, *p1 = (double *)f.psi1;
    size_t l = f.at(i, j, k);
    p0[l] = f.b[q] * p0[l] - f.c[q] * (B1[c] - B1[cm]) / f.dxn;
    p1[l] = f.b[q] * p1[l] + f.c[q] * (B0[c] - B0[cm]) / f.dxn;
}

// CPMLBorderHCurrent::stepScheme, src/cpml_border.cpp:499-527
__global__ __launch_bounds__(256) void k_ref_cpml_H(StepArgs<double> a, int fi, FaceCells at)
{
    const CpmlFace &f = a.face[fi];
    int k = at.lo[2] + blockIdx.x * 64 + threadIdx.x;
    int j = at.lo[1] + blockIdx.y * 4 + threadIdx.y;
    int i = at.lo[0] + blockIdx.z;
    if (k > at.hi[2] || j > at.hi[1]) return;
    int ind[3] = {i, j, k};
    int p[3] = {i, j, k};
    p[f.dim] += 1;
    int q = ind[f.dim] - f.lo[f.dim];
    const GridDims &g = a.g;
    size_t c = g.at(i, j, k), cp = g.at(p[0], p[1], p[2]);
    const double *E0 = a.E[f.f0], *E1 = a.E[f.f1];
    double *p0 = (double *)f.psi0, *p1 = (double *)f.psi1;
    size_t l = f.at(i, j, k);
    p0[l] = f.b[q] * p0[l] + f.c[q] * (E1[cp] - E1[c]) / f.dxn;
    p1[l] = f.b[q] * p1[l] - f.c[q] * (E0[cp] - E0[c]) / f.dxn;
}

void launch_ref_cpml(const StepArgs<double> &a, int fi, bool isH, hipStream_t s)
{
    const CpmlFace &f = a.face[fi];
    dim3 blk(64, 4);
    const FaceCells c = face_cells(f, a.g.n, isH);
    dim3 grd((c.hi[2] - c.lo[2] + 64) / 64, (c.hi[1] - c.lo[1] + 4) / 4, c.hi[0] - c.lo[0] + 1);
    if (isH)
        hipLaunchKernelGGL(k_ref_cpml_H, grd, blk, 0, s, a, fi, c);
    else
        hipLaunchKernelGGL(k_ref_cpml_E, grd, blk, 0, s, a, fi, c);
}

// FDTD_PLRCSolver::sumCurrents / sumMagCurrents, src/fdtd_plrc.t:342-409: totals := 0, then
// += every current's layer in list order, cell by cell.
__global__ __launch_bounds__(256) void k_ref_sum(GridDims g, SumList L, double *T0, double *T1, double *T2)
{
    int k = blockIdx.x * 64 + threadIdx.x;
    int j = blockIdx.y * 4 + threadIdx.y;
    int i = blockIdx.z;
    if (k > g.n[2] + 1 || j > g.n[1] + 1) return;
    double t[3] = {0.0, 0.0, 0.0};
    for (int v = 0; v < L.n; ++v) {
        const SumView &w = L.v[v];
        if (i < w.lo[0] || i > w.hi[0] || j < w.lo[1] || j > w.hi[1] || k < w.lo[2] || k > w.hi[2]) continue;
        size_t l = w.padded ? g.at(i, j, k)
                            : ((size_t)(i - w.lo[0]) * w.n1 + (size_t)(j - w.lo[1])) * w.n2 + (size_t)(k - w.lo[2]);
#pragma unroll
        for (int c = 0; c < 3; ++c)
            if (w.comp[c]) t[c] += w.comp[c][l];
    }
    size_t c = g.at(i, j, k);
    T0[c] = t[0];
    T1[c] = t[1];
    T2[c] = t[2];
}

void launch_ref_sum(const GridDims &g, const SumList &L, double *const T[3], hipStream_t s)
{
    dim3 blk(64, 4);
    dim3 grd((g.n[2] + 2 + 63) / 64, (g.n[1] + 2 + 3) / 4, g.n[0] + 2);
    hipLaunchKernelGGL(k_ref_sum, grd, blk, 0, s, g, L, T[0], T[1], T[2]);
}

// Storage::applyBoundary + SinglePeriodicBoundary::exchange{X,Y,Z}, src/storage.cpp:194-204,
// src/periodic_bound.cpp:10-71: f(0) = f(N), f(N+1) = f(1) over the full planes.
template <typename T>
__global__ __launch_bounds__(256) void k_wrap(GridDims g, T *f0, T *f1, T *f2, int dim)
{
    T *f = blockIdx.z == 0 ? f0 : (blockIdx.z == 1 ? f1 : f2);
    if (!f) return;  // a group of one array (the residual words of float32 + residual storage)
    int a = blockIdx.x * 64 + threadIdx.x;  // fastest remaining dimension
    int b = blockIdx.y * 4 + threadIdx.y;
    int N = g.n[dim];
    if (dim == 0) {
        if (a > g.n[2] + 1 || b > g.n[1] + 1) return;
        f[g.at(0, b, a)] = f[g.at(N, b, a)];
        f[g.at(N + 1, b, a)] = f[g.at(1, b, a)];
    } else if (dim == 1) {
        if (a > g.n[2] + 1 || b > g.n[0] + 1) return;
        f[g.at(b, 0, a)] = f[g.at(b, N, a)];
        f[g.at(b, N + 1, a)] = f[g.at(b, 1, a)];
    } else {
        if (a > g.n[1] + 1 || b > g.n[0] + 1) return;
        f[g.at(b, a, 0)] = f[g.at(b, a, N)];
        f[g.at(b, a, N + 1)] = f[g.at(b, a, 1)];
    }
}

template <typename T>
void launch_wrap(const GridDims &g, T *const f[3], int dim, hipStream_t s)
{
    int na = dim == 2 ? g.n[1] + 2 : g.n[2] + 2;
    int nb = dim == 0 ? g.n[1] + 2 : g.n[0] + 2;
    dim3 blk(64, 4);
    dim3 grd((na + 63) / 64, (nb + 3) / 4, 3);
    hipLaunchKernelGGL(k_wrap<T>, grd, blk, 0, s, g, f[0], f[1], f[2], dim);
}
template void launch_wrap<double>(const GridDims &, double *const[3], int, hipStream_t);
template void launch_wrap<float>(const GridDims &, float *const[3], int, hipStream_t);
template void launch_wrap<unsigned>(const GridDims &, unsigned *const[3], int, hipStream_t);

// FDTD_PLRCSolver::stepD loop, src/fdtd_plrc.t:221-233, reading the current totals
template <int NP, bool NONLIN>
__global__ __launch_bounds__(256) void k_ref_stepD(StepArgs<double> a)
{
    int k = blockIdx.x * 64 + threadIdx.x + 1;
    int j = blockIdx.y * 4 + threadIdx.y + 1;
    int i = blockIdx.z + 1;
    const GridDims &g = a.g;
    if (k > g.n[2] || j > g.n[1]) return;
    size_t c = g.at(i, j, k);
    const double *Bx = a.B[0], *By = a.B[1], *Bz = a.B[2];
    double bx = Bx[c], by = By[c], bz = Bz[c];
    double dBz_y = bz - Bz[g.at(i, j - 1, k)];
    double dBy_z = by - By[g.at(i, j, k - 1)];
    double dBx_z = bx - Bx[g.at(i, j, k - 1)];
    double dBz_x = bz - Bz[g.at(i - 1, j, k)];
    double dBy_x = by - By[g.at(i - 1, j, k)];
    double dBx_y = bx - Bx[g.at(i, j - 1, k)];
    double jx = 0, jy = 0, jz = 0;
    if (a.haveJ) {
        jx = a.Jt[0][c];
        jy = a.Jt[1][c];
        jz = a.Jt[2][c];
    }
    double ex = a.E[0][c], ey = a.E[1][c], ez = a.E[2][c];
    double denom, numer;
    cell_eps<NONLIN>(a, c, a.plasma ? 0.5 * a.sigma[c] * a.dt : 0.0, denom, numer);
    unsigned fl = 0;
    plrc_e_update<NP, NONLIN, false>(ex, ey, ez, dBz_y, dBy_z, dBx_z, dBz_x, dBy_x, dBx_y, a.kdE[0][i], a.kdE[1][j],
                                     a.kdE[2][k], jx, jy, jz, a.psi, c, a.pc, a.dt, denom, numer, a.chi, a.ncap, &fl);
    report(a.status, fl | finite_flag(ex, ey, ez));
    a.E[0][c] = ex;
    a.E[1][c] = ey;
    a.E[2][c] = ez;
}

// FDTD_PLRCSolver::stepB + plrcStepB, src/fdtd_plrc.t:312-339, src/fdtd_plrc.cpp:429-459;
// Jt holds the magnetic current totals here.
__global__ __launch_bounds__(256) void k_ref_stepB(StepArgs<double> a)
{
    int k = blockIdx.x * 64 + threadIdx.x;
    int j = blockIdx.y * 4 + threadIdx.y;
    int i = blockIdx.z;
    const GridDims &g = a.g;
    if (k > g.n[2] || j > g.n[1]) return;
    size_t c = g.at(i, j, k);
    const double *Ex = a.E[0], *Ey = a.E[1], *Ez = a.E[2];
    double jx = 0, jy = 0, jz = 0;
    if (a.haveJ) {
        jx = a.Jt[0][c];
        jy = a.Jt[1][c];
        jz = a.Jt[2][c];
    }
    double kdx = a.kdH[0][i], kdy = a.kdH[1][j], kdz = a.kdH[2][k];
    double ex = Ex[c], ey = Ey[c], ez = Ez[c];
    a.B[0][c] = a.B[0][c] + a.dt * ((Ey[g.at(i, j, k + 1)] - ey) / kdz - (Ez[g.at(i, j + 1, k)] - ez) / kdy + jx);
    a.B[1][c] = a.B[1][c] + a.dt * ((Ez[g.at(i + 1, j, k)] - ez) / kdx - (Ex[g.at(i, j, k + 1)] - ex) / kdz + jy);
    a.B[2][c] = a.B[2][c] + a.dt * ((Ex[g.at(i, j + 1, k)] - ex) / kdy - (Ey[g.at(i + 1, j, k)] - ey) / kdx + jz);
}

void launch_ref_stepD(const StepArgs<double> &a, int np, bool nonlin, hipStream_t s)
{
    const GridDims &g = a.g;
    dim3 blk(64, 4);
    dim3 grd((g.n[2] + 63) / 64, (g.n[1] + 3) / 4, g.n[0]);
#define MPX_REF_D(NPV, NL) hipLaunchKernelGGL((k_ref_stepD<NPV, NL>), grd, blk, 0, s, a)
    if (nonlin) {
        switch (np) {
        case 0: MPX_REF_D(0, true); break;
        case 1: MPX_REF_D(1, true); break;
        case 2: MPX_REF_D(2, true); break;
        default: MPX_REF_D(3, true); break;
        }
    } else {
        switch (np) {
        case 0: MPX_REF_D(0, false); break;
        case 1: MPX_REF_D(1, false); break;
        case 2: MPX_REF_D(2, false); break;
        default: MPX_REF_D(3, false); break;
        }
    }
#undef MPX_REF_D
}

// PlasmaDensity over the whole storage box 0..N+1 (Sigma was cleared: it becomes w I^(K-1))
__global__ __launch_bounds__(256) void k_ref_plasma_density(StepArgs<double> a)
{
    int k = blockIdx.x * 64 + threadIdx.x;
    int j = blockIdx.y * 4 + threadIdx.y;
    int i = blockIdx.z;
    const GridDims &g = a.g;
    if (k > g.n[2] + 1 || j > g.n[1] + 1) return;
    size_t c = g.at(i, j, k);
    double r = a.rho[c];
    const double ikm = plasma_density_cell(a.E[0][c], a.E[1][c], a.E[2][c], r, a.pn, a.pm, a.pk - 1);
    a.rho[c] = r;
    a.sigma[c] = 0.0 + a.pw * ikm;
}

// PlasmaCurrent over low..high-1 = 0..N of the storage box
__global__ __launch_bounds__(256) void k_ref_plasma_current(StepArgs<double> a)
{
    int k = blockIdx.x * 64 + threadIdx.x;
    int j = blockIdx.y * 4 + threadIdx.y;
    int i = blockIdx.z;
    const GridDims &g = a.g;
    if (k > g.n[2] || j > g.n[1]) return;
    size_t c = g.at(i, j, k);
    const double rt = a.rho[c] + a.rho_bg;
    for (int q = 0; q < 3; ++q) a.jp[q][c] = plasma_current_comp(a.jp[q][c], a.E[q][c], rt, a.gdtn, a.gdtd, a.emdt);
}

void launch_ref_plasma_density(const StepArgs<double> &a, hipStream_t s)
{
    const GridDims &g = a.g;
    hipLaunchKernelGGL(k_ref_plasma_density, dim3((g.n[2] + 2 + 63) / 64, (g.n[1] + 2 + 3) / 4, g.n[0] + 2),
                       dim3(64, 4), 0, s, a);
}

void launch_ref_plasma_current(const StepArgs<double> &a, hipStream_t s)
{
    const GridDims &g = a.g;
    hipLaunchKernelGGL(k_ref_plasma_current, dim3((g.n[2] + 1 + 63) / 64, (g.n[1] + 1 + 3) / 4, g.n[0] + 1),
                       dim3(64, 4), 0, s, a);
}

void launch_ref_stepB(const StepArgs<double> &a, hipStream_t s)
{
    const GridDims &g = a.g;
    dim3 blk(64, 4);
    dim3 grd((g.n[2] + 1 + 63) / 64, (g.n[1] + 1 + 3) / 4, g.n[0] + 1);
    hipLaunchKernelGGL(k_ref_stepB, grd, blk, 0, s, a);
}

// FDTD_PLRCSolver::initAccumulator, src/fdtd_plrc.t:273-308 (stepSchemeInit only)
template <int NP>
__global__ __launch_bounds__(256) void k_init_accumulator(StepArgs<double> a)
{
    int k = blockIdx.x * 64 + threadIdx.x + 1;
    int j = blockIdx.y * 4 + threadIdx.y + 1;
    int i = blockIdx.z + 1;
    const GridDims &g = a.g;
    if (k > g.n[2] || j > g.n[1]) return;
    size_t c = g.at(i, j, k);
    double e[3] = {a.E[0][c], a.E[1][c], a.E[2][c]};
#pragma unroll
    for (int n = 0; n < NP; ++n)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            double2 p = a.psi[n][d][psi_at(c)];
            const double2 X = a.pc.dxi0[n], C = a.pc.crec[n];
            a.psi[n][d][psi_at(c)] = make_double2(X.x * e[d] + (C.x * p.x - C.y * p.y), X.y * e[d] + (C.x * p.y + C.y * p.x));
        }
}

void launch_init_accumulator(const StepArgs<double> &a, int np, hipStream_t s)
{
    const GridDims &g = a.g;
    dim3 blk(64, 4);
    dim3 grd((g.n[2] + 63) / 64, (g.n[1] + 3) / 4, g.n[0]);
    switch (np) {
    case 0: break;
    case 1: hipLaunchKernelGGL(k_init_accumulator<1>, grd, blk, 0, s, a); break;
    case 2: hipLaunchKernelGGL(k_init_accumulator<2>, grd, blk, 0, s, a); break;
    default: hipLaunchKernelGGL(k_init_accumulator<3>, grd, blk, 0, s, a); break;
    }
}

// ------------------------------------------------------------------------------------
// fdtd-plain, fdtd-nl, fdtd-disp (no currents)
// ------------------------------------------------------------------------------------
//
// Memory bound: 12 words a cell and step, fdtd-disp 27 more for its polarisations.  The
// reference updates E over [1, N+1]^3 and B over [0, N]^3 and exchanges the ghosts after each
// (src/fdtd_plain.cpp:54-118, src/storage.cpp:194-204); the exchange took six launches of 5 us
// a step with four-cell rows, 30 of the 160 us of a 120x112x100 step.  Here the B kernel takes
// E beyond N from the periodic image by index and leaves the images of E and of the new B in
// the ghosts with the stores of the cells that own them; along a non-periodic z the update
// covers the reference's range instead.  The ADE solver writes P of the new step over P of the
// step before last and the host exchanges the two names, 9 words a cell less than moving P to
// Pp.  Blocks take their tiles in XCD-contiguous slabs (xcd_tile), so the neighbour planes of
// B and E are read from one L2.
// Measured, fdtd-disp 120x112x100, us a step: stepD 102, stepB 29, exchange 30 before; 98, 24 and none now
// (4.1 TB/s in stepD: 18 polarisation streams a lane, each its own pages).

// E loops of FDTD_Plain / FDTD_Nonlinear / FDTD_Dispersion over [1, N+1]^3
// (src/fdtd_plain.cpp:54-75, src/fdtd_nl.cpp:55-98, src/fdtd_disp.cpp:113-204); KIND 0, 1, 2.
// E of a periodic dimension's ghost is left to the B kernel; the threads of those ghosts (all
// kinds but plain) do what else the reference does there.
template <int KIND>
__global__ __launch_bounds__(256) void k_simple_stepD(SimpleArgs a, int nbx, int nby, int nbz)
{
    constexpr int LO = KIND == 2 ? 0 : 1;  // the polarisations at coordinate 0 change buffers
    int bx, by, bz;
    xcd_tile(nbx, nby, nbz, bx, by, bz);
    const int k = bx * 64 + threadIdx.x + LO, i = bz + LO;
    const int j = __builtin_amdgcn_readfirstlane(by * 4 + (int)threadIdx.y + LO);  // one row a wave
    const GridDims &g = a.g;
    if (k > g.n[2] + 1 || j > g.n[1] + 1) return;
    const bool low = i == 0 || j == 0 || k == 0;
    const bool ghost = low || i > g.n[0] || j > g.n[1] || (a.zper && k > g.n[2]);
    const size_t row = g.at(i, j, 0);
    const unsigned o = 8u * k;
    const double dx = a.dx, dy = a.dy, dz = a.dz, dt = a.dt;
    double ex = 0, ey = 0, ez = 0, cx = 0, cy = 0, cz = 0;
    // every polarisation is read before the first is stored, so that the reads leave together
    double p1[3][3], p0[3][3];
    if (KIND == 2) {
#pragma unroll
        for (int n = 0; n < 3; ++n)
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                p1[n][d] = ldp_once(a.P[n][d] + row, o);
                p0[n][d] = ldp_once(a.Pp[n][d] + row, o);
            }
    }
    if (!low) {
        ex = ldp(a.E[0] + row, o);
        ey = ldp(a.E[1] + row, o);
        ez = ldp(a.E[2] + row, o);
        const double *Bx = a.B[0] + row, *By = a.B[1] + row, *Bz = a.B[2] + row;
        const double bx0 = ldp(Bx, o), by0 = ldp(By, o), bz0 = ldp(Bz, o);
        const size_t si = (size_t)g.sx, sj = g.pz;
        cx = (bz0 - ldp(Bz - sj, o)) / dy - (by0 - ldp(By, o - 8u)) / dz;
        cy = (bx0 - ldp(Bx, o - 8u)) / dz - (bz0 - ldp(Bz - si, o)) / dx;
        cz = (by0 - ldp(By - si, o)) / dx - (bx0 - ldp(Bx - sj, o)) / dy;
    }
    if (KIND == 0) {
        ex = ex + dt * cx;
        ey = ey + dt * cy;
        ez = ez + dt * cz;
    } else if (KIND == 1) {
        double E2 = ex * ex + ey * ey + ez * ez;
        double Dx = (a.eps + a.chi * E2) * ex + dt * cx;
        double Dy = (a.eps + a.chi * E2) * ey + dt * cy;
        double Dz = (a.eps + a.chi * E2) * ez + dt * cz;
        double E = sqrt(E2);
        double D = sqrt(Dx * Dx + Dy * Dy + Dz * Dz);
        double Eold;
        int it = 0;
        do {
            Eold = E;
            E2 = E * E;
            E = (2 * a.chi * E2 * E + D) / (3 * a.chi * E2 + a.eps);
        } while (fabs(E - Eold) > 1e-9 && ++it < a.ncap);
        ex = E * Dx / D;
        ey = E * Dy / D;
        ez = E * Dz / D;
        // a zero D gives NaN, as in the reference (src/fdtd_nl.cpp:86-89): reported, not avoided
        report(a.status, (it >= a.ncap ? 1u : 0u) | finite_flag(ex, ey, ez));
    } else {
        const double e[3] = {ex, ey, ez};
        double P[3] = {0, 0, 0}, Pp[3] = {0, 0, 0};
        const double dt2 = dt * dt;
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            const double aa = dt2 * a.om2[n];
            const double b = aa * a.eps2[n];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const double p = p1[n][d], pp = p0[n][d];
                const double pn = (2 - aa) * p - pp + b * e[d];
                stp_once(a.Pp[n][d] + row, o, low ? p : pn);
                if (low) stp(a.P[n][d] + row, o, pp);
                P[d] += pn;
                Pp[d] += p;
            }
        }
        ex = ex + Pp[0] - P[0] + dt * cx;
        ey = ey + Pp[1] - P[1] + dt * cy;
        ez = ez + Pp[2] - P[2] + dt * cz;
    }
    if (ghost) return;
    stp(a.E[0] + row, o, ex);
    stp(a.E[1] + row, o, ey);
    stp(a.E[2] + row, o, ez);
}

// The cells that hold the value of coordinate c of a periodic dimension: itself and its ghost
// images (N + 1 for cell 1, 0 for cell N)
struct Images {
    int c[3], n;
};
__device__ __forceinline__ Images images_of(int c, int N, bool periodic)
{
    Images m;
    m.c[0] = m.c[1] = m.c[2] = c;
    m.n = 1;
    if (periodic) {
        if (c == 1) m.c[m.n++] = N + 1;
        if (c == N) m.c[m.n++] = 0;
    }
    return m;
}

// stepB shared by the three solvers, including the /dx of both Bz terms
// (src/fdtd_plain.cpp:97-118), and the ghosts of B and (EXCH) of E.  Without EXCH
// (FDTD_Plain::stepSchemeInit, src/fdtd_plain.cpp:26-29) E beyond N is read as stored and left.
template <bool EXCH>
__global__ __launch_bounds__(256) void k_simple_stepB(SimpleArgs a, int nbx, int nby, int nbz)
{
    int bx, by, bz;
    xcd_tile(nbx, nby, nbz, bx, by, bz);
    const GridDims &g = a.g;
    const int k = bx * 64 + threadIdx.x + (a.zper ? 1 : 0), i = bz + 1;
    const int j = __builtin_amdgcn_readfirstlane(by * 4 + (int)threadIdx.y + 1);
    if (k > g.n[2] || j > g.n[1]) return;
    const size_t row = g.at(i, j, 0);
    const unsigned o = 8u * k;
    const size_t ri = EXCH && i == g.n[0] ? g.at(1, j, 0) : row + (size_t)g.sx;
    const size_t rj = EXCH && j == g.n[1] ? g.at(i, 1, 0) : row + g.pz;
    const unsigned ok = EXCH && a.zper && k == g.n[2] ? 8u : o + 8u;
    double dx = a.dx, dy = a.dy, dz = a.dz, dt = a.dt;
    const double e[3] = {ldp(a.E[0] + row, o), ldp(a.E[1] + row, o), ldp(a.E[2] + row, o)};
    const double ex = e[0], ey = e[1], ez = e[2];
    double b[3] = {ldp(a.B[0] + row, o), ldp(a.B[1] + row, o), ldp(a.B[2] + row, o)};
    b[0] = b[0] + dt * ((ldp(a.E[1] + row, ok) - ey) / dz - (ldp(a.E[2] + rj, o) - ez) / dy);
    b[1] = b[1] + dt * ((ldp(a.E[2] + ri, o) - ez) / dx - (ldp(a.E[0] + row, ok) - ex) / dz);
    b[2] = b[2] + dt * ((ldp(a.E[0] + rj, o) - ex) / dx - (ldp(a.E[1] + ri, o) - ey) / dx);
    for (int d = 0; d < 3; ++d) stp(a.B[d] + row, o, b[d]);
    if (i > 1 && i < g.n[0] && j > 1 && j < g.n[1]) {  // at most z images: every wave meets a row end
        if (a.zper && (k == 1 || k == g.n[2])) {
            const unsigned q = k == 1 ? 8u * (g.n[2] + 1) : 0u;
            for (int d = 0; d < 3; ++d) {
                stp(a.B[d] + row, q, b[d]);
                if (EXCH) stp(a.E[d] + row, q, e[d]);
            }
            if (g.n[2] == 1)  // cell 1 is cell N too
                for (int d = 0; d < 3; ++d) {
                    stp(a.B[d] + row, 0u, b[d]);
                    if (EXCH) stp(a.E[d] + row, 0u, e[d]);
                }
        }
        return;
    }
    const Images x = images_of(i, g.n[0], true), y = images_of(j, g.n[1], true), z = images_of(k, g.n[2], a.zper);
    for (int u = 0; u < x.n; ++u)
        for (int v = 0; v < y.n; ++v)
            for (int w = 0; w < z.n; ++w) {
                if (u + v + w == 0) continue;
                const size_t q = g.at(x.c[u], y.c[v], z.c[w]);
                for (int d = 0; d < 3; ++d) {
                    a.B[d][q] = b[d];
                    if (EXCH) a.E[d][q] = e[d];
                }
                if (!a.zper && k == g.n[2])  // the plane above, outside B's range
                    for (int d = 0; d < 3; ++d) {
                        a.B[d][q + 1] = a.B[d][row + k + 1];
                        if (EXCH) a.E[d][q + 1] = a.E[d][row + k + 1];
                    }
            }
}

void launch_simple_stepD(const SimpleArgs &a, hipStream_t s)
{
    const GridDims &g = a.g;
    const int more = a.kind == 2 ? 2 : (a.kind == 1 ? 1 : 0);  // the ghosts whose threads have work
    const int nk = g.n[2] + (a.zper || more ? more : 1), nj = g.n[1] + more;
    const int nbx = (nk + 63) / 64, nby = (nj + 3) / 4, nbz = g.n[0] + more;
    dim3 blk(64, 4), grd(nbx, nby, nbz);
    switch (a.kind) {
    case 0: hipLaunchKernelGGL(k_simple_stepD<0>, grd, blk, 0, s, a, nbx, nby, nbz); break;
    case 1: hipLaunchKernelGGL(k_simple_stepD<1>, grd, blk, 0, s, a, nbx, nby, nbz); break;
    default: hipLaunchKernelGGL(k_simple_stepD<2>, grd, blk, 0, s, a, nbx, nby, nbz); break;
    }
}

void launch_simple_stepB(const SimpleArgs &a, bool exchange, hipStream_t s)
{
    const GridDims &g = a.g;
    const int nbx = (g.n[2] + (a.zper ? 0 : 1) + 63) / 64, nby = (g.n[1] + 3) / 4, nbz = g.n[0];
    dim3 blk(64, 4), grd(nbx, nby, nbz);
    if (exchange)
        hipLaunchKernelGGL(k_simple_stepB<true>, grd, blk, 0, s, a, nbx, nby, nbz);
    else
        hipLaunchKernelGGL(k_simple_stepB<false>, grd, blk, 0, s, a, nbx, nby, nbz);
}

// ------------------------------------------------------------------------------------
// diagnostics: probes and energy
// ------------------------------------------------------------------------------------

template <typename T>
__global__ void k_probe(ProbeArgs<T> a, double *row)
{
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.n) return;
    const int q = a.comp[p];
    const size_t c = a.idx[p];
    const unsigned *lo = a.lo[q / 3];
    row[p] = lo ? res_decode((float)a.f[q][c], lo[c], q % 3) : (double)a.f[q][c];
}

template <typename T>
void launch_probe(const ProbeArgs<T> &a, double *row, hipStream_t s)
{
    hipLaunchKernelGGL(k_probe<T>, dim3((a.n + 63) / 64), dim3(64), 0, s, a, row);
}
template void launch_probe<double>(const ProbeArgs<double> &, double *, hipStream_t);
template void launch_probe<float>(const ProbeArgs<float> &, double *, hipStream_t);

// FieldEnergyDiag::calculate, src/fielddiag.cpp:255-286: per-block partial sums, then one
// block adds the partials in a fixed order.
template <typename T>
__device__ __forceinline__ void cell3(const T *f0, const T *f1, const T *f2, const unsigned *lo, size_t c, double v[3])
{
    if (lo) {
        const unsigned w = lo[c];
        v[0] = res_decode((float)f0[c], w, 0);
        v[1] = res_decode((float)f1[c], w, 1);
        v[2] = res_decode((float)f2[c], w, 2);
    } else {
        v[0] = f0[c];
        v[1] = f1[c];
        v[2] = f2[c];
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_energy_partial(GridDims g, const T *e0, const T *e1, const T *e2,
                                                        const T *b0, const T *b1, const T *b2, const unsigned *elo,
                                                        const unsigned *blo, double *part)
{
    __shared__ double red[256];
    int k = blockIdx.x * 64 + threadIdx.x + 1;
    int j = blockIdx.y * 4 + threadIdx.y + 1;
    int i = blockIdx.z + 1;
    double v = 0;
    if (k <= g.n[2] && j <= g.n[1]) {
        size_t c = g.at(i, j, k);
        double e[3], b[3];
        cell3(e0, e1, e2, elo, c, e);
        cell3(b0, b1, b2, blo, c, b);
        v = e[0] * e[0] + e[1] * e[1] + e[2] * e[2] + b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
    }
    int t = threadIdx.y * 64 + threadIdx.x;
    red[t] = v;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) red[t] += red[t + w];
        __syncthreads();
    }
    if (t == 0) part[blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = red[0];
}

__global__ __launch_bounds__(256) void k_sum_partials(const double *part, size_t n, double *out, double scale)
{
    __shared__ double red[256];
    double v = 0;
    for (size_t q = threadIdx.x; q < n; q += 256) v += part[q];
    red[threadIdx.x] = v;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0] * scale;
}

size_t energy_partials(const GridDims &g)
{
    return (size_t)((g.n[2] + 63) / 64) * ((g.n[1] + 3) / 4) * g.n[0];
}

template <typename T>
void launch_energy(const GridDims &g, T *const e[3], T *const b[3], double *part, double *out, hipStream_t s,
                   const unsigned *elo, const unsigned *blo, double scale)
{
    dim3 blk(64, 4);
    dim3 grd((g.n[2] + 63) / 64, (g.n[1] + 3) / 4, g.n[0]);
    hipLaunchKernelGGL(k_energy_partial<T>, grd, blk, 0, s, g, e[0], e[1], e[2], b[0], b[1], b[2], elo, blo, part);
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, s, part, energy_partials(g), out, scale);
}
void launch_sum_partials(const double *part, size_t n, double *out, double scale, hipStream_t s)
{
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, s, part, n, out, scale);
}
template void launch_energy<double>(const GridDims &, double *const[3], double *const[3], double *, double *,
                                    hipStream_t, const unsigned *, const unsigned *, double);
template void launch_energy<float>(const GridDims &, float *const[3], float *const[3], double *, double *,
                                   hipStream_t, const unsigned *, const unsigned *, double);

}  // namespace mpx

namespace mpx {

// Plain streaming copy, one 16-byte vector per thread over a grid that covers the buffer
// (the fastest copy shape measured on gfx950): the calibration kernel for HBM byte counters
// and the practical bandwidth ceiling of the device.
__global__ __launch_bounds__(256) void k_hbm_copy(const double2 *__restrict__ src, double2 *__restrict__ dst, size_t n)
{
    size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) dst[q] = src[q];
}

void launch_hbm_copy(const void *src, void *dst, size_t bytes, hipStream_t s)
{
    size_t n = bytes / 16;
    hipLaunchKernelGGL(k_hbm_copy, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (const double2 *)src,
                       (double2 *)dst, n);
}

// Coordinate c of dimension d as the grid holds it: where bit d of wrapmask is set, a ghost (0 or
// N + 1) reads its periodic image (N or 1), which is what the ghost holds once the wrap has run.
// Reading the image costs the pack kernels nothing; running the wrap first took six launches a
// group of E or B (twelve with residual words), 36 of them and 0.15 of 0.49 ms for the six fields
// of a 24^3 grid.
__device__ __forceinline__ int image(const GridDims &g, int wrapmask, int d, int c)
{
    if ((wrapmask >> d) & 1) c = c == 0 ? g.n[d] : (c == g.n[d] + 1 ? 1 : c);
    return c;
}

// A grid over the storage box 0..N+1 in the order of the reference's Grid (x fastest), as
// float64: dst[(k (ny+2) + j) (nx+2) + i] = src(i, j, k), the form FieldDiag hands to its HDF5
// stream.  A block transposes a 32 (z) x 32 (x) tile of one y row through LDS, so that both
// the reads (z contiguous) and the writes (x contiguous) are coalesced.
template <typename T>
__global__ __launch_bounds__(256) void k_pack_xfast(GridDims g, const T *__restrict__ src, const unsigned *lo, int q,
                                                    int wrapmask, double *__restrict__ dst)
{
    __shared__ double tile[32][33];
    const int nx2 = g.n[0] + 2, ny2 = g.n[1] + 2, nz2 = g.n[2] + 2;
    const int k0 = blockIdx.x * 32, i0 = blockIdx.y * 32, j = blockIdx.z;
    const int js = image(g, wrapmask, 1, j);
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int i = i0 + r, k = k0 + threadIdx.x;
        if (i < nx2 && k < nz2) {
            const size_t c = g.at(image(g, wrapmask, 0, i), js, image(g, wrapmask, 2, k));
            tile[r][threadIdx.x] = lo ? res_decode((float)src[c], lo[c], q) : (double)src[c];
        }
    }
    __syncthreads();
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int k = k0 + r, i = i0 + threadIdx.x;
        if (i < nx2 && k < nz2) dst[((size_t)k * ny2 + j) * nx2 + i] = tile[threadIdx.x][r];
    }
}

template <typename T>
void launch_pack_xfast(const GridDims &g, const T *src, double *dst, hipStream_t s, int wrapmask, const unsigned *lo,
                       int q)
{
    dim3 grd((g.n[2] + 2 + 31) / 32, (g.n[0] + 2 + 31) / 32, g.n[1] + 2);
    hipLaunchKernelGGL(k_pack_xfast<T>, grd, dim3(32, 8), 0, s, g, src, lo, q, wrapmask, dst);
}
template void launch_pack_xfast<float>(const GridDims &, const float *, double *, hipStream_t, int, const unsigned *,
                                       int);
template void launch_pack_xfast<double>(const GridDims &, const double *, double *, hipStream_t, int, const unsigned *,
                                        int);

// Planes i0 .. of the storage box in z-fastest order as float64, the form of mpx_get_field /
// mpx_set_field: box[((i - i0) (ny+2) + j) (nz+2) + k] <-> the grid's cell (i, j, k).  PSI: the grid is component 0 of a
// pole's accumulator block shifted to its component (psi_at), and q is the part (0 re, 1 im).
// Unpacking into float32 + residual storage replaces slot q of the cell's residual word.  The
// conversion and the padding were a loop over the cells on one host core (0.25 ms of the 0.33 ms
// of a 50 x 42 x 58 read, 3 s of a 514^3 one); here they run at the copy rate and the host
// buffer takes one copy.
template <typename T, bool PSI>
__global__ __launch_bounds__(256) void k_pack_box(GridDims g, const T *__restrict__ src, const unsigned *lo, int q,
                                                  int wrapmask, int i0, double *__restrict__ box)
{
    const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y, i = i0 + blockIdx.z;
    if (k > g.n[2] + 1 || j > g.n[1] + 1) return;
    const size_t c = g.at(image(g, wrapmask, 0, i), image(g, wrapmask, 1, j), image(g, wrapmask, 2, k));
    double v;
    if (PSI)
        v = (double)src[2 * psi_at(c) + q];
    else
        v = lo ? res_decode((float)src[c], lo[c], q) : (double)src[c];
    box[((size_t)blockIdx.z * (g.n[1] + 2) + j) * (g.n[2] + 2) + k] = v;
}

template <typename T, bool PSI>
__global__ __launch_bounds__(256) void k_unpack_box(GridDims g, const double *__restrict__ box, T *__restrict__ dst,
                                                    unsigned *lo, int q, int i0)
{
    const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y, i = i0 + blockIdx.z;
    if (k > g.n[2] + 1 || j > g.n[1] + 1) return;
    const size_t c = g.at(i, j, k);
    const double v = box[((size_t)blockIdx.z * (g.n[1] + 2) + j) * (g.n[2] + 2) + k];
    if (PSI)
        dst[2 * psi_at(c) + q] = (T)v;
    else if (lo) {
        unsigned w = 0;
        dst[c] = (T)res_encode(v, w, q);
        lo[c] = (lo[c] & ~(0x3ffu << (10 * q))) | w;
    } else
        dst[c] = (T)v;
}

static dim3 box_grid(const GridDims &g, int ni) { return dim3((g.n[2] + 2 + 63) / 64, (g.n[1] + 2 + 3) / 4, ni); }

template <typename T>
void launch_pack_box(const GridDims &g, const T *src, double *box, int i0, int ni, hipStream_t s, bool psi, int wrapmask,
                     const unsigned *lo, int q)
{
    if (psi)
        hipLaunchKernelGGL((k_pack_box<T, true>), box_grid(g, ni), dim3(64, 4), 0, s, g, src, lo, q, wrapmask, i0, box);
    else
        hipLaunchKernelGGL((k_pack_box<T, false>), box_grid(g, ni), dim3(64, 4), 0, s, g, src, lo, q, wrapmask, i0, box);
}
template <typename T>
void launch_unpack_box(const GridDims &g, const double *box, T *dst, int i0, int ni, hipStream_t s, bool psi, unsigned *lo, int q)
{
    if (psi)
        hipLaunchKernelGGL((k_unpack_box<T, true>), box_grid(g, ni), dim3(64, 4), 0, s, g, box, dst, lo, q, i0);
    else
        hipLaunchKernelGGL((k_unpack_box<T, false>), box_grid(g, ni), dim3(64, 4), 0, s, g, box, dst, lo, q, i0);
}
template void launch_pack_box<float>(const GridDims &, const float *, double *, int, int, hipStream_t, bool, int,
                                     const unsigned *, int);
template void launch_pack_box<double>(const GridDims &, const double *, double *, int, int, hipStream_t, bool, int,
                                      const unsigned *, int);
template void launch_unpack_box<float>(const GridDims &, const double *, float *, int, int, hipStream_t, bool, unsigned *,
                                       int);
template void launch_unpack_box<double>(const GridDims &, const double *, double *, int, int, hipStream_t, bool, unsigned *,
                                        int);

// One record of a sampler: the value at storage cell c (dim < 0) or the len = N[dim] + 2 values
// of the storage line through c along dim, as float64.  A coordinate of a dimension in
// wrapmask that names a ghost reads its periodic image (0 -> N, N + 1 -> 1), which is what the
// ghost holds once the wrap has run; the caller checks 0 <= c[d] <= N[d] + 1.
template <typename T>
__global__ __launch_bounds__(256) void k_sample_gather(GridDims g, const T *__restrict__ src, const unsigned *lo, int qc,
                                                      int dim, int c0, int c1, int c2, int len, int wrapmask,
                                                      double *__restrict__ dst)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= len) return;
    int c[3] = {c0, c1, c2};
    if (dim >= 0) c[dim] = q;
    const size_t at = g.at(image(g, wrapmask, 0, c[0]), image(g, wrapmask, 1, c[1]), image(g, wrapmask, 2, c[2]));
    dst[q] = lo ? res_decode((float)src[at], lo[at], qc) : (double)src[at];
}

template <typename T>
void launch_sample_gather(const GridDims &g, const T *src, int dim, const int *c, int len, int wrapmask, double *dst,
                         hipStream_t s, const unsigned *lo, int q)
{
    hipLaunchKernelGGL(k_sample_gather<T>, dim3((len + 255) / 256), dim3(256), 0, s, g, src, lo, q, dim, c[0], c[1],
                       c[2], len, wrapmask, dst);
}
template void launch_sample_gather<float>(const GridDims &, const float *, int, const int *, int, int, double *,
                                         hipStream_t, const unsigned *, int);
template void launch_sample_gather<double>(const GridDims &, const double *, int, const int *, int, int, double *,
                                          hipStream_t, const unsigned *, int);

}  // namespace mpx
