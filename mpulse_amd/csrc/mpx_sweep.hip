// gfx950 kernels of the sweep path: E and B of a step in one kernel, periodic boundaries.  The
// file is compiled once per word type (MPX_FORM 0: float64, 1: float32), so that the variants
// compile in parallel.
#include <hip/hip_runtime.h>

#include "mpx_device.h"
#include "mpx_launch.h"

#ifndef MPX_FORM
#error "MPX_FORM selects the storage form this object holds"
#endif

namespace mpx {

// ------------------------------------------------------------------------------------
// single-pass sweep path (periodic boundaries): E and B of a step in one kernel
// ------------------------------------------------------------------------------------
//
// Block = 64 lanes along z x BY thread rows along y; each thread row handles RPT tile rows,
// so a tile is 64 x TYR cells (TYR = BY * RPT).  Lane 63 and tile row TYR-1 are a one-cell
// halo: E is computed there (identically to the owning block) but never stored, so the
// B update of the owned 63 x (TYR-1) cells finds E_new at k+1 and j+1 inside the block.
// The block walks the x planes i0..i1 of its segment: at plane p it computes E_new(p), puts
// it in a triple-buffered LDS tile, synchronises once, and updates B at plane p-1 from
// E_new(p-1) and E_new(p).  Every array the step reads is an "old" buffer and every array it
// writes a "new" buffer (CPML H auxiliaries excepted: only owners touch them), so halo
// readers never see another block's results.
//
// sweep_tile is one tile's walk; k_sweep maps the blocks of one grid onto tiles, k_sweep_batch
// walks the tiles of many independent grids from one persistent launch.
template <typename T, int NP, bool NONLIN, bool CPML, int BY, int RPT>
__device__ __forceinline__ void sweep_tile(const SweepArgs<T> &a, int tz, int ty, int tx,
                                           T (&lds)[3][3][BY * RPT][64])
{
    constexpr int TYR = BY * RPT;
    const GridDims &g = a.g;
    const int Nx = g.n[0], Ny = g.n[1], Nz = g.n[2];
    const int sx = (int)g.sx, pz = g.pz;
    const int lane = threadIdx.x;
    const int k = 1 + 63 * tz + lane;
    const bool kact = k <= Nz + 1;
    // physical z index (periodic image of the halo lane); idle lanes get 1 so that every
    // index they form stays inside the arrays, although they load nothing from the grids
    const int kk = (!kact || k == Nz + 1) ? 1 : k;
    const int okm = (kk == 1) ? (Nz - 1) : -1;
    const int i0 = 1 + a.seg * tx;
    const int i1 = min(i0 + a.seg - 1, Nx);
    int jj[RPT], ojm[RPT], rowi[RPT];
    bool eact[RPT], own[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        rowi[r] = threadIdx.y + BY * r;
        int j = 1 + (TYR - 1) * ty + rowi[r];
        eact[r] = kact && j <= Ny + 1;
        own[r] = eact[r] && lane < 63 && k <= Nz && rowi[r] < TYR - 1 && j <= Ny;
        jj[r] = (j == Ny + 1) ? 1 : j;
        ojm[r] = (jj[r] == 1) ? (Ny - 1) * pz : -pz;
        if (!eact[r]) jj[r] = 1;  // keeps idle threads' addresses in range; they load nothing
    }
    const T *Bxo = a.Bo[0], *Byo = a.Bo[1], *Bzo = a.Bo[2];
    // B_old at plane i0-1 (the x neighbour of the first E plane)
    const int im0 = (i0 == 1) ? Nx : i0 - 1;
    double bprev[RPT][3], eprev[RPT][3];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        eprev[r][0] = eprev[r][1] = eprev[r][2] = 0.0;
        bprev[r][0] = bprev[r][1] = bprev[r][2] = 0.0;
        if (eact[r]) {
            int c = im0 * sx + jj[r] * pz + kk + g.z0;
            bprev[r][0] = Bxo[c];
            bprev[r][1] = Byo[c];
            bprev[r][2] = Bzo[c];
        }
    }
    const double kdz_e = a.ikdE[2][kk], kdz_h = a.ikdH[2][kk];  // reciprocals
    // the grid inputs of a plane (B and its y / z neighbours, E, the pole accumulators) are
    // loaded one plane ahead, so that their latency overlaps the work and the barrier of the
    // plane before
    T nb[RPT][7], ne[RPT][3];
    PsiRegs<NP> npsi[RPT];
    auto load_plane = [&](int p) {
        const int pp = (p == Nx + 1) ? 1 : p;
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
            if (!eact[r]) continue;
            const int c = pp * sx + jj[r] * pz + kk + g.z0;
            nb[r][0] = Bxo[c];
            nb[r][1] = Byo[c];
            nb[r][2] = Bzo[c];
            nb[r][3] = Bzo[c + ojm[r]];
            nb[r][4] = Bxo[c + ojm[r]];
            nb[r][5] = Byo[c + okm];
            nb[r][6] = Bxo[c + okm];
            ne[r][0] = a.Eo[0][c];
            ne[r][1] = a.Eo[1][c];
            ne[r][2] = a.Eo[2][c];
#pragma unroll
            for (int n = 0; n < NP; ++n)
#pragma unroll
                for (int q = 0; q < 3; ++q) npsi[r].v[n][q] = load_once(&a.psio[n][q][psi_at(c)]);
        }
    };
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
#pragma unroll
        for (int q = 0; q < 7; ++q) nb[r][q] = (T)0;
        ne[r][0] = ne[r][1] = ne[r][2] = (T)0;
#pragma unroll
        for (int n = 0; n < NP; ++n)
#pragma unroll
            for (int q = 0; q < 3; ++q) npsi[r].v[n][q] = make_double2(0.0, 0.0);
    }
    load_plane(i0);
    for (int p = i0; p <= i1 + 1; ++p) {
        const int pp = (p == Nx + 1) ? 1 : p;
        const int buf = p % 3;
        T cb[RPT][7], ce[RPT][3];
        PsiRegs<NP> cpsi[RPT];
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
#pragma unroll
            for (int q = 0; q < 7; ++q) cb[r][q] = nb[r][q];
            ce[r][0] = ne[r][0];
            ce[r][1] = ne[r][1];
            ce[r][2] = ne[r][2];
            cpsi[r] = npsi[r];
        }
        if (p <= i1) load_plane(p + 1);
        double ecur[RPT][3], bcur[RPT][3];
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
            ecur[r][0] = ecur[r][1] = ecur[r][2] = 0.0;
            bcur[r][0] = bcur[r][1] = bcur[r][2] = 0.0;
            if (!eact[r]) continue;
            const int j = jj[r];
            const int c = pp * sx + j * pz + kk + g.z0;
            const double bx = cb[r][0], by = cb[r][1], bz = cb[r][2];
            const double dBz_y = bz - (double)cb[r][3];
            const double dBx_y = bx - (double)cb[r][4];
            const double dBy_z = by - (double)cb[r][5];
            const double dBx_z = bx - (double)cb[r][6];
            const double dBz_x = bz - bprev[r][2];
            const double dBy_x = by - bprev[r][1];
            bcur[r][0] = bx;
            bcur[r][1] = by;
            bcur[r][2] = bz;
            const bool store = own[r] && p <= i1;
            double jx = 0.0, jy = 0.0, jz = 0.0;
            if (a.sheets_first) add_sheet_planes(a.sheet, a.nsheets, g.py, pp, j, kk, 0, jx, jy, jz);
            if (CPML) {
                // E auxiliaries, list order N,S (y), E,W (x), U,D (z), high face first
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const int dim = d == 0 ? 1 : (d == 1 ? 0 : 2);
                    const int coord = dim == 0 ? pp : (dim == 1 ? j : kk);
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        const int fi = a.efbd[dim][s];
                        if (fi < 0) continue;
                        const CpmlFace &f = a.eface[fi];
                        if (coord < f.lo[dim] || coord > f.hi[dim]) continue;
                        const int l = layer_index(f, pp, j, kk);
                        const int q = coord - f.lo[dim];
                        const T *o0 = (const T *)a.epsi_old[fi][0], *o1 = (const T *)a.epsi_old[fi][1];
                        double d1 = dim == 0 ? dBz_x : (dim == 1 ? dBx_y : dBy_z);
                        double d0 = dim == 0 ? dBy_x : (dim == 1 ? dBz_y : dBx_z);
                        T n0 = (T)(f.b[q] * (double)o0[l] - f.c[q] * d1 * f.idxn);
                        T n1 = (T)(f.b[q] * (double)o1[l] + f.c[q] * d0 * f.idxn);
                        if (store) {
                            ((T *)f.psi0)[l] = n0;
                            ((T *)f.psi1)[l] = n1;
                        }
                        if (dim == 0) {
                            jy += (double)n0;
                            jz += (double)n1;
                        } else if (dim == 1) {
                            jz += (double)n0;
                            jx += (double)n1;
                        } else {
                            jx += (double)n0;
                            jy += (double)n1;
                        }
                    }
                }
            }
            if (!a.sheets_first) add_sheet_planes(a.sheet, a.nsheets, g.py, pp, j, kk, 0, jx, jy, jz);
            double ex = (double)ce[r][0], ey = (double)ce[r][1], ez = (double)ce[r][2];
            unsigned fl = 0;
            plrc_e_update_pp<NP, NONLIN, true>(ex, ey, ez, dBz_y, dBy_z, dBx_z, dBz_x, dBy_x, dBx_y,
                                               a.ikdE[0][pp], a.ikdE[1][j], kdz_e, jx, jy, jz, cpsi[r], a.psin, c,
                                               store, a.pc, a.dt, a.idenom, a.numer, a.chi, a.ncap, &fl);
            if (store) fl |= finite_flag(ex, ey, ez);
            report(a.status, fl);
            const T tx_ = (T)ex, ty_ = (T)ey, tz_ = (T)ez;
            if (store) {
                a.En[0][c] = tx_;
                a.En[1][c] = ty_;
                a.En[2][c] = tz_;
            }
            lds[buf][0][rowi[r]][lane] = tx_;
            lds[buf][1][rowi[r]][lane] = ty_;
            lds[buf][2][rowi[r]][lane] = tz_;
            ecur[r][0] = (double)tx_;
            ecur[r][1] = (double)ty_;
            ecur[r][2] = (double)tz_;
        }
        __syncthreads();
        if (p > i0) {
            const int pb = p - 1;  // B plane, inside [i0, i1]
            const int pbuf = pb % 3;
#pragma unroll
            for (int r = 0; r < RPT; ++r) {
                if (!own[r]) continue;
                const int j = jj[r];
                const int c = pb * sx + j * pz + kk + g.z0;
                const int row = rowi[r];
                const double ex = eprev[r][0], ey = eprev[r][1], ez = eprev[r][2];
                const double dEy_z = (double)lds[pbuf][1][row][lane + 1] - ey;
                const double dEx_z = (double)lds[pbuf][0][row][lane + 1] - ex;
                const double dEz_y = (double)lds[pbuf][2][row + 1][lane] - ez;
                const double dEx_y = (double)lds[pbuf][0][row + 1][lane] - ex;
                const double dEz_x = ecur[r][2] - ez;
                const double dEy_x = ecur[r][1] - ey;
                double mx = 0.0, my = 0.0, mz = 0.0;
                if (a.sheets_first) add_sheet_planes(a.hsheet, a.nhsheets, g.py, pb, j, kk, 0, mx, my, mz);
                if (CPML) {
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        const int dim = d == 0 ? 1 : (d == 1 ? 0 : 2);
                        const int coord = dim == 0 ? pb : (dim == 1 ? j : kk);
#pragma unroll
                        for (int s = 0; s < 2; ++s) {
                            const int fi = a.hfbd[dim][s];
                            if (fi < 0) continue;
                            const CpmlFace &f = a.hface[fi];
                            if (coord < f.lo[dim] || coord > f.hi[dim]) continue;
                            const int l = layer_index(f, pb, j, kk);
                            const int q = coord - f.lo[dim];
                            T *p0 = (T *)f.psi0, *p1 = (T *)f.psi1;
                            double d1 = dim == 0 ? dEz_x : (dim == 1 ? dEx_y : dEy_z);
                            double d0 = dim == 0 ? dEy_x : (dim == 1 ? dEz_y : dEx_z);
                            T n0 = (T)(f.b[q] * (double)p0[l] + f.c[q] * d1 * f.idxn);
                            T n1 = (T)(f.b[q] * (double)p1[l] - f.c[q] * d0 * f.idxn);
                            p0[l] = n0;
                            p1[l] = n1;
                            if (dim == 0) {
                                my += (double)n0;
                                mz += (double)n1;
                            } else if (dim == 1) {
                                mz += (double)n0;
                                mx += (double)n1;
                            } else {
                                mx += (double)n0;
                                my += (double)n1;
                            }
                        }
                    }
                }
                if (!a.sheets_first) add_sheet_planes(a.hsheet, a.nhsheets, g.py, pb, j, kk, 0, mx, my, mz);
                const double kdx = a.ikdH[0][pb], kdy = a.ikdH[1][j];
                a.Bn[0][c] = (T)(bprev[r][0] + a.dt * ((dEy_z * kdz_h - dEz_y * kdy) + mx));
                a.Bn[1][c] = (T)(bprev[r][1] + a.dt * ((dEz_x * kdx - dEx_z * kdz_h) + my));
                a.Bn[2][c] = (T)(bprev[r][2] + a.dt * ((dEx_y * kdy - dEy_x * kdx) + mz));
            }
        }
#pragma unroll
        for (int r = 0; r < RPT; ++r)
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                eprev[r][q] = ecur[r][q];
                bprev[r][q] = bcur[r][q];
            }
    }
}

template <typename T, int NP, bool NONLIN, bool CPML, int BY, int RPT>
__global__ __launch_bounds__(64 * BY) void k_sweep(SweepArgs<T> a, int ntz, int nty, int nseg)
{
    __shared__ T lds[3][3][BY * RPT][64];
    int tz, ty, tx;
    xcd_tile(ntz, nty, nseg, tz, ty, tx);
    sweep_tile<T, NP, NONLIN, CPML, BY, RPT>(a, tz, ty, tx, lds);
}

// Persistent batched sweep over the tiles of all runs (see batch_tiles).
template <typename T, int NP, bool NONLIN, bool CPML, int BY, int RPT>
__global__ __launch_bounds__(64 * BY) void k_sweep_batch(const SweepArgs<T> *__restrict__ args,
                                                         const BatchRun *__restrict__ runs, int nruns, int total)
{
    __shared__ T lds[3][3][BY * RPT][64];
    batch_tiles(runs, nruns, total, [&](int r, int tz, int ty, int tx) {
        sweep_tile<T, NP, NONLIN, CPML, BY, RPT>(args[r], tz, ty, tx, lds);
        __syncthreads();  // the next tile rewrites the LDS planes
    });
}

template <typename T, int NP, bool NONLIN, bool CPML>
static void launch_sweep_np(const SweepArgs<T> &a, hipStream_t s)
{
    int ntz, nty, nseg;
    sweep_tiles(a.g, a.variant, a.seg, ntz, nty, nseg);
    if (a.variant == 1)  // 64 x 4 threads: 4-row tiles
        hipLaunchKernelGGL((k_sweep<T, NP, NONLIN, CPML, 4, 1>), dim3(ntz, nty, nseg), dim3(64, 4), 0, s, a, ntz, nty,
                           nseg);
    else if (a.variant == 2)  // 64 x 16 threads, 1 row each
        hipLaunchKernelGGL((k_sweep<T, NP, NONLIN, CPML, 16, 1>), dim3(ntz, nty, nseg), dim3(64, 16), 0, s, a, ntz,
                           nty, nseg);
    else  // 64 x 8 threads, 1 row each: 8-row tiles
        hipLaunchKernelGGL((k_sweep<T, NP, NONLIN, CPML, 8, 1>), dim3(ntz, nty, nseg), dim3(64, 8), 0, s, a, ntz, nty,
                           nseg);
}

#if MPX_FORM == 0
// tile grid of one run for the block shape `variant` and segment length `seg`
void sweep_tiles(const GridDims &g, int variant, int seg, int &ntz, int &nty, int &nseg)
{
    ntz = (g.n[2] + 62) / 63;
    nty = variant == 0 ? (g.n[1] + 6) / 7 : (variant == 1 ? (g.n[1] + 2) / 3 : (g.n[1] + 14) / 15);
    nseg = (g.n[0] + seg - 1) / seg;
}
#endif

template <typename T, int NP, bool NONLIN, bool CPML>
static void launch_sweep_batch_np(const SweepArgs<T> *args, const BatchRun *runs, int nruns, int total, int variant,
                                  int blocks, hipStream_t s)
{
    if (variant == 1)
        hipLaunchKernelGGL((k_sweep_batch<T, NP, NONLIN, CPML, 4, 1>), dim3(blocks), dim3(64, 4), 0, s, args, runs,
                           nruns, total);
    else if (variant == 2)
        hipLaunchKernelGGL((k_sweep_batch<T, NP, NONLIN, CPML, 16, 1>), dim3(blocks), dim3(64, 16), 0, s, args, runs,
                           nruns, total);
    else
        hipLaunchKernelGGL((k_sweep_batch<T, NP, NONLIN, CPML, 8, 1>), dim3(blocks), dim3(64, 8), 0, s, args, runs,
                           nruns, total);
}

template <typename T>
void launch_sweep_batch(const SweepArgs<T> *args, const BatchRun *runs, int nruns, int total, int variant,
                        int blocks, int np, bool nonlin, bool cpml, hipStream_t s)
{
#define MPX_SB(NPV, NL, CP) launch_sweep_batch_np<T, NPV, NL, CP>(args, runs, nruns, total, variant, blocks, s)
#define MPX_SB_NP(NL, CP)             \
    switch (np) {                     \
    case 0: MPX_SB(0, NL, CP); break; \
    case 1: MPX_SB(1, NL, CP); break; \
    case 2: MPX_SB(2, NL, CP); break; \
    default: MPX_SB(3, NL, CP); break; \
    }
    if (nonlin) {
        if (cpml) { MPX_SB_NP(true, true) } else { MPX_SB_NP(true, false) }
    } else {
        if (cpml) { MPX_SB_NP(false, true) } else { MPX_SB_NP(false, false) }
    }
#undef MPX_SB_NP
#undef MPX_SB
}
#if MPX_FORM == 0
template void launch_sweep_batch<double>(const SweepArgs<double> *, const BatchRun *, int, int, int, int, int, bool,
                                         bool, hipStream_t);
#else
template void launch_sweep_batch<float>(const SweepArgs<float> *, const BatchRun *, int, int, int, int, int, bool,
                                        bool, hipStream_t);
#endif

template <typename T>
void launch_sweep(const SweepArgs<T> &a, int np, bool nonlin, hipStream_t s)
{
    bool cp = a.nefaces > 0;
#define MPX_SW(NPV, NL, CP) launch_sweep_np<T, NPV, NL, CP>(a, s)
#define MPX_SW_NP(NL, CP)            \
    switch (np) {                    \
    case 0: MPX_SW(0, NL, CP); break; \
    case 1: MPX_SW(1, NL, CP); break; \
    case 2: MPX_SW(2, NL, CP); break; \
    default: MPX_SW(3, NL, CP); break; \
    }
    if (nonlin) {
        if (cp) { MPX_SW_NP(true, true) } else { MPX_SW_NP(true, false) }
    } else {
        if (cp) { MPX_SW_NP(false, true) } else { MPX_SW_NP(false, false) }
    }
#undef MPX_SW_NP
#undef MPX_SW
}
#if MPX_FORM == 0
template void launch_sweep<double>(const SweepArgs<double> &, int, bool, hipStream_t);
#else
template void launch_sweep<float>(const SweepArgs<float> &, int, bool, hipStream_t);
#endif

}  // namespace mpx
