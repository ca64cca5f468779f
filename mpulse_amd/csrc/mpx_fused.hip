// gfx950 kernels of the fused path: one E-side kernel (Yee curl + PLRC pole recursion + Kerr
// Newton solve + CPML E auxiliaries + source sheet) and one B-side kernel (curl + CPML H
// auxiliaries + source sheet), with the periodic ghost wrap done by index arithmetic
// (FDTD_PLRCSolver::stepScheme, src/fdtd_plrc.t:127-168).  Threads run along z (the contiguous
// dimension), 64 per wavefront, so every field load of a wavefront is one coalesced
// 256/512-byte segment.  The file is compiled once per word type (MPX_FORM 0: float64, 1:
// float32 with and without residual words), so that the variants compile in parallel.
#include <hip/hip_runtime.h>

#include "mpx_device.h"
#include "mpx_launch.h"

#ifndef MPX_FORM
#error "MPX_FORM selects the storage form this object holds"
#endif

namespace mpx {

// Fused E side of one step.  A thread owns one (j, k) column segment of L cells along x and
// walks it plane by plane, keeping B of the previous plane in registers for the x difference.
template <typename T, int NP, bool NONLIN, bool CPML, int L, bool LIN = false, bool RES = false>
__device__ __forceinline__ void fused_E_tile(const StepArgs<T> &a, int tbx, int tby, int tbz, int soff)
{
    using V = typename Word<T, RES>::V;
    const GridDims &g = a.g;
    const int one[3] = {1, 1, 1};
    int j, k;
    tile_jk<LIN>(g, one, tbx, tby, j, k);
    const int i0 = tbz * L + 1;
    if (k > g.n[2] || j > g.n[1] || i0 > g.n[0]) return;
    const int i1 = min(i0 + L - 1, g.n[0]);
    const int sx = (int)g.sx, pz = g.pz;
    const int ojm = (j == 1 && a.periodic[1]) ? (g.n[1] - 1) * pz : -pz;
    const int okm = (k == 1 && a.periodic[2]) ? (g.n[2] - 1) : -1;
    int c = i0 * sx + j * pz + k + g.z0;
    const T *Bx = a.B[0], *By = a.B[1], *Bz = a.B[2];
    const int cim = (i0 == 1 && a.periodic[0]) ? c + (g.n[0] - 1) * sx : c - sx;
    const unsigned wim = lo_ld<RES>(a.Blo, cim);
    double bz_im = (double)rd<T, RES>(Bz, wim, 2, cim), by_im = (double)rd<T, RES>(By, wim, 1, cim);
    bool iny[2] = {false, false}, inz[2] = {false, false};
    if (CPML) {
        in_faces(a.face_by_dim, a.face, 1, j, iny);
        in_faces(a.face_by_dim, a.face, 2, k, inz);
    }
    const double kdy = gld(a.ikdE[1] + j), kdz = gld(a.ikdE[2] + k);
#pragma unroll
    for (int u = 0; u < L; ++u, c += sx) {
        const int i = i0 + u;
        if (i > i1) break;
        // z neighbours: the first lane of a wave and the first cell of a row load them, every
        // other lane takes them from the previous lane (the loads are issued first, so that one
        // wait covers them and the cell's own loads)
        const bool zload = threadIdx.x == 0 || k == 1;
        V bym = (V)0, bxm = (V)0;
        if (zload) {
            const unsigned wm = lo_ld<RES>(a.Blo, c + okm);
            bym = rd<T, RES>(By, wm, 1, c + okm);
            bxm = rd<T, RES>(Bx, wm, 0, c + okm);
        }
        const unsigned wb = lo_ld<RES>(a.Blo, c);
        const V bxt = rd<T, RES>(Bx, wb, 0, c), byt = rd<T, RES>(By, wb, 1, c);
        const double bx = bxt, by = byt, bz = rd<T, RES>(Bz, wb, 2, c);
        // E and the pole accumulators are read before any store of the cell (the CPML
        // auxiliaries), so that all its reads leave together
        const unsigned we = lo_once<RES>(a.Elo, c);
        double ex = (double)rd_once<T, RES>(a.E[0], we, 0, c), ey = (double)rd_once<T, RES>(a.E[1], we, 1, c);
        double ez = (double)rd_once<T, RES>(a.E[2], we, 2, c);
        PsiRegs<NP> pr;
#pragma unroll
        for (int n = 0; n < NP; ++n)
#pragma unroll
            for (int q = 0; q < 3; ++q) pr.v[n][q] = load_once(&a.psi[n][q][psi_at(c)]);
        const unsigned wj = lo_ld<RES>(a.Blo, c + ojm);
        const double dBz_y = bz - (double)rd<T, RES>(Bz, wj, 2, c + ojm);
        const double dBx_y = bx - (double)rd<T, RES>(Bx, wj, 0, c + ojm);
        const V bys = lane_prev(byt), bxs = lane_prev(bxt);
        const double dBy_z = by - (double)(zload ? bym : bys);
        const double dBx_z = bx - (double)(zload ? bxm : bxs);
        const double dBz_x = bz - bz_im;
        const double dBy_x = by - by_im;
        bz_im = bz;
        by_im = by;
        // the plasma OptField and the plasma current run before the E update, on E of this step
        double sg = 0.0, jpv[3] = {0.0, 0.0, 0.0};
        if (a.plasma || a.pcur) {
            double r = gld(a.rho + c);
            if (a.plasma) {
                sg = a.pw * plasma_density_cell(ex, ey, ez, r, a.pn, a.pm, a.pk - 1);
                gst(a.rho + c, r);
                gst(a.sigma + c, sg);
            }
            if (a.pcur) {
                const double rt = r + a.rho_bg, ev[3] = {ex, ey, ez};
                for (int q = 0; q < 3; ++q) {
                    jpv[q] = plasma_current_comp(gld(a.jp[q] + c), ev[q], rt, a.gdtn, a.gdtd, a.emdt);
                    gst(a.jp[q] + c, jpv[q]);
                }
            }
        }
        // current totals in list order: the CPML and sheet groups, the plasma current at its place
        double jx = 0.0, jy = 0.0, jz = 0.0;
        auto add_cpml = [&]() {
            if (CPML) {
                // current totals in the reference's list order N,S (y), E,W (x), U,D (z); within a
                // dimension the high face comes first in that list
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    if (iny[s]) {
                        const CpmlFace &f = a.face[a.face_by_dim[1][s]];
                        double v0, v1;
                        cpml_face<T, false, RES>(f, j, layer_index(f, i, j, k), dBx_y, dBz_y, v0, v1);
                        jz += v0;
                        jx += v1;
                    }
                bool inx[2];
                in_faces(a.face_by_dim, a.face, 0, i, inx);
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    if (inx[s]) {
                        const CpmlFace &f = a.face[a.face_by_dim[0][s]];
                        double v0, v1;
                        cpml_face<T, false, RES>(f, i, layer_index(f, i, j, k), dBz_x, dBy_x, v0, v1);
                        jy += v0;
                        jz += v1;
                    }
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    if (inz[s]) {
                        const CpmlFace &f = a.face[a.face_by_dim[2][s]];
                        double v0, v1;
                        cpml_face<T, false, RES>(f, k, layer_index(f, i, j, k), dBy_z, dBx_z, v0, v1);
                        jx += v0;
                        jy += v1;
                    }
            }
        };
        auto add_plasma = [&](int pos) {
            if (a.pcur && a.pcur_pos == pos) {
                jx += jpv[0];
                jy += jpv[1];
                jz += jpv[2];
            }
        };
        add_plasma(0);
        if (a.sheets_first)
            add_sheets(a, i, j, k, soff, jx, jy, jz);
        else
            add_cpml();
        add_plasma(1);
        if (a.sheets_first)
            add_cpml();
        else
            add_sheets(a, i, j, k, soff, jx, jy, jz);
        add_plasma(2);
        double idenom = a.idenom, numer = a.numer;
        if (a.epsf || a.plasma) {
            double denom;
            cell_eps<NONLIN>(a, (size_t)c, 0.5 * sg * a.dt, denom, numer);
            idenom = 1.0 / denom;
        }
        unsigned fl = 0;
        plrc_e_update_pp<NP, NONLIN, true>(ex, ey, ez, dBz_y, dBy_z, dBx_z, dBz_x, dBy_x, dBx_y, gld(a.ikdE[0] + i), kdy,
                                           kdz, jx, jy, jz, pr, a.psi, (size_t)c, true, a.pc, a.dt, idenom, numer,
                                           a.chi, a.ncap, &fl);
        report(a.status, fl | finite_flag(ex, ey, ez));
        unsigned wn = 0;
        const T hx = put<T, RES>(ex, wn, 0), hy = put<T, RES>(ey, wn, 1), hz = put<T, RES>(ez, wn, 2);
        store_once(&a.En[0][c], hx);
        store_once(&a.En[1][c], hy);
        store_once(&a.En[2][c], hz);
        if (RES) store_once(&a.Elo[c], wn);
    }
}

// Fused B side of one step: a thread walks L planes along x keeping E of the next plane in
// registers as the centre of the following iteration.
template <typename T, bool CPML, int L, bool LIN = false, bool RES = false>
__device__ __forceinline__ void fused_B_tile(const StepArgs<T> &a, int tbx, int tby, int tbz, int soff)
{
    using V = typename Word<T, RES>::V;
    const GridDims &g = a.g;
    int j, k;
    tile_jk<LIN>(g, a.blo, tbx, tby, j, k);
    const int i0 = tbz * L + a.blo[0];
    if (k > g.n[2] || j > g.n[1] || i0 > g.n[0]) return;
    const int i1 = min(i0 + L - 1, g.n[0]);
    const int sx = (int)g.sx, pz = g.pz;
    const int ojp = (j == g.n[1] && a.periodic[1]) ? -(g.n[1] - 1) * pz : pz;
    const int okp = (k == g.n[2] && a.periodic[2]) ? -(g.n[2] - 1) : 1;
    int c = i0 * sx + j * pz + k + g.z0;
    const T *Ex = a.E[0], *Ey = a.E[1], *Ez = a.E[2];
    T *Bx = a.B[0], *By = a.B[1], *Bz = a.B[2];
    // z neighbours: the last lane of a wave and the last cell of a row load them, every other
    // lane takes them from the next lane
    const bool zload = threadIdx.x == 63 || k == g.n[2];
    V ezl[L][2];
    if (zload) {
#pragma unroll
        for (int u = 0; u < L; ++u) {
            const int cu = c + u * sx;
            ezl[u][0] = ezl[u][1] = (V)0;
            if (i0 + u <= i1) {
                const unsigned w = lo_ld<RES>(a.Elo, cu + okp);
                ezl[u][0] = rd<T, RES>(Ey, w, 1, cu + okp);
                ezl[u][1] = rd<T, RES>(Ex, w, 0, cu + okp);
            }
        }
    }
    const unsigned w0 = lo_ld<RES>(a.Elo, c);
    const V ex0 = rd<T, RES>(Ex, w0, 0, c), ey0 = rd<T, RES>(Ey, w0, 1, c), ez0 = rd<T, RES>(Ez, w0, 2, c);
    double ex = ex0, ey = ey0, ez = ez0;
    bool iny[2] = {false, false}, inz[2] = {false, false};
    if (CPML) {
        in_faces(a.face_by_dim, a.face, 1, j, iny);
        in_faces(a.face_by_dim, a.face, 2, k, inz);
    }
    const double kdy = gld(a.ikdH[1] + j), kdz = gld(a.ikdH[2] + k);
    // the E and B values of all L planes are read before the first store, so that they leave
    // together (per plane: E at x+1, E_y and E_x at z+1, E_z and E_x at y+1, B)
    V pe[L][7], pb[L][3];
#pragma unroll
    for (int u = 0; u < L; ++u) {
        const int i = i0 + u;
        if (i > i1) break;
        const int cu = c + u * sx;
        const int cip = (i == g.n[0] && a.periodic[0]) ? cu - (g.n[0] - 1) * sx : cu + sx;
        const unsigned wx = lo_ld<RES>(a.Elo, cip), wy = lo_ld<RES>(a.Elo, cu + ojp);
        const unsigned wbu = lo_once<RES>(a.Blo, cu);
        pe[u][0] = rd<T, RES>(Ex, wx, 0, cip);
        pe[u][1] = rd<T, RES>(Ey, wx, 1, cip);
        pe[u][2] = rd<T, RES>(Ez, wx, 2, cip);
        pe[u][5] = rd<T, RES>(Ez, wy, 2, cu + ojp);
        pe[u][6] = rd<T, RES>(Ex, wy, 0, cu + ojp);
        pb[u][0] = rd_once<T, RES>(Bx, wbu, 0, cu);
        pb[u][1] = rd_once<T, RES>(By, wbu, 1, cu);
        pb[u][2] = rd_once<T, RES>(Bz, wbu, 2, cu);
    }
#pragma unroll
    for (int u = 0; u < L; ++u) {
        if (i0 + u > i1) break;
        // E at z+1: the next lane's centre value of the same plane
        const V sy = lane_next(u == 0 ? ey0 : pe[u - 1][1]), sx_ = lane_next(u == 0 ? ex0 : pe[u - 1][0]);
        pe[u][3] = zload ? ezl[u][0] : sy;
        pe[u][4] = zload ? ezl[u][1] : sx_;
    }
#pragma unroll
    for (int u = 0; u < L; ++u, c += sx) {
        const int i = i0 + u;
        if (i > i1) break;
        const double ex1 = pe[u][0], ey1 = pe[u][1], ez1 = pe[u][2];
        const double dEy_z = (double)pe[u][3] - ey;
        const double dEx_z = (double)pe[u][4] - ex;
        const double dEz_y = (double)pe[u][5] - ez;
        const double dEx_y = (double)pe[u][6] - ex;
        const double dEz_x = ez1 - ez;
        const double dEy_x = ey1 - ey;
        double mx = 0.0, my = 0.0, mz = 0.0;
        if (a.sheets_first) add_sheets(a, i, j, k, soff, mx, my, mz);
        if (CPML) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
                if (iny[s]) {
                    const CpmlFace &f = a.face[a.face_by_dim[1][s]];
                    double v0, v1;  // psi0 -> Mz from dEx_y, psi1 -> Mx from dEz_y
                    cpml_face<T, true, RES>(f, j, layer_index(f, i, j, k), dEx_y, dEz_y, v0, v1);
                    mz += v0;
                    mx += v1;
                }
            bool inx[2];
            in_faces(a.face_by_dim, a.face, 0, i, inx);
#pragma unroll
            for (int s = 0; s < 2; ++s)
                if (inx[s]) {
                    const CpmlFace &f = a.face[a.face_by_dim[0][s]];
                    double v0, v1;  // psi0 -> My from dEz_x, psi1 -> Mz from dEy_x
                    cpml_face<T, true, RES>(f, i, layer_index(f, i, j, k), dEz_x, dEy_x, v0, v1);
                    my += v0;
                    mz += v1;
                }
#pragma unroll
            for (int s = 0; s < 2; ++s)
                if (inz[s]) {
                    const CpmlFace &f = a.face[a.face_by_dim[2][s]];
                    double v0, v1;  // psi0 -> Mx from dEy_z, psi1 -> My from dEx_z
                    cpml_face<T, true, RES>(f, k, layer_index(f, i, j, k), dEy_z, dEx_z, v0, v1);
                    mx += v0;
                    my += v1;
                }
        }
        if (!a.sheets_first) add_sheets(a, i, j, k, soff, mx, my, mz);
        const double kdx = gld(a.ikdH[0] + i);
        unsigned wn = 0;
        const T hx = put<T, RES>((double)pb[u][0] + a.dt * ((dEy_z * kdz - dEz_y * kdy) + mx), wn, 0);
        const T hy = put<T, RES>((double)pb[u][1] + a.dt * ((dEz_x * kdx - dEx_z * kdz) + my), wn, 1);
        const T hz = put<T, RES>((double)pb[u][2] + a.dt * ((dEx_y * kdy - dEy_x * kdx) + mz), wn, 2);
        store_once(&Bx[c], hx);
        store_once(&By[c], hy);
        store_once(&Bz[c], hz);
        if (RES) store_once(&a.Blo[c], wn);
        ex = ex1;
        ey = ey1;
        ez = ez1;
    }
}

// The argument block is read from device memory (the solver keeps a copy there): the face
// tables are indexed at run time, which a by-value kernel argument would have to copy into
// per-lane scratch.
// Waves per SIMD the E kernel is compiled for: 6 (at most 80 registers) for the float32 Kerr
// kernel with one pole and one plane per thread, measured 0.3 % faster than the 5 its registers
// allow; no constraint otherwise (other variants would spill).
template <typename T, int NP, bool NONLIN, int L, bool RES>
struct FusedEWaves {
    static constexpr int v = (sizeof(T) == 4 && !RES && NP <= 1 && NONLIN && L == 1) ? 6 : 1;
};

template <typename T, int NP, bool NONLIN, bool CPML, int L, bool RES = false>
__global__ __attribute__((amdgpu_waves_per_eu(FusedEWaves<T, NP, NONLIN, L, RES>::v))) __launch_bounds__(256) void k_fused_E(
    const StepArgs<T> *__restrict__ pa, int nbx, int nby, int nbz, int soff)
{
    int tbx, tby, tbz;
    fused_tile_of(pa->order, pa->band, pa->rev, nbx, nby, nbz, tbx, tby, tbz);
    fused_E_tile<T, NP, NONLIN, CPML, L, false, RES>(*pa, tbx, tby, tbz, soff);
}

template <typename T, bool CPML, int L, bool RES = false>
__global__ __launch_bounds__(256) void k_fused_B(const StepArgs<T> *__restrict__ pa, int nbx, int nby, int nbz,
                                                 int soff)
{
    int tbx, tby, tbz;
    fused_tile_of(pa->order, pa->band, pa->rev, nbx, nby, nbz, tbx, tby, tbz);
    fused_B_tile<T, CPML, L, false, RES>(*pa, tbx, tby, tbz, soff);
}

// the fused kernels over the tiles of many independent runs, one persistent launch
template <typename T, int NP, bool NONLIN, bool CPML, int L>
__global__ __launch_bounds__(256) void k_fused_E_batch(const StepArgs<T> *__restrict__ args,
                                                       const BatchRun *__restrict__ runs, int nruns, int total)
{
    batch_tiles(runs, nruns, total, [&](int r, int tz, int ty, int tx) {
        fused_E_tile<T, NP, NONLIN, CPML, L, true>(args[r], tz, ty, tx, 0);
    });
}

template <typename T, bool CPML, int L>
__global__ __launch_bounds__(256) void k_fused_B_batch(const StepArgs<T> *__restrict__ args,
                                                       const BatchRun *__restrict__ runs, int nruns, int total)
{
    batch_tiles(runs, nruns, total,
                [&](int r, int tz, int ty, int tx) { fused_B_tile<T, CPML, L, true>(args[r], tz, ty, tx, 0); });
}

#if MPX_FORM == 0
// tile grid of the batched fused kernels of one run: 256 consecutive y-z cells per tile
// (tile_jk with LIN), L x planes per thread
void fused_tiles(const GridDims &g, const int blo[3], bool hside, int L, int &ntz, int &nty, int &nseg)
{
    const int one[3] = {1, 1, 1};
    const int *lo = hside ? blo : one;
    long long yz = (long long)(g.n[1] - lo[1] + 1) * (g.n[2] - lo[2] + 1);
    ntz = (int)((yz + 255) / 256);
    nty = 1;
    nseg = (g.n[0] - lo[0] + 1 + L - 1) / L;
}
#endif

template <typename T, int L>
static void launch_fused_E_batch_L(const StepArgs<T> *args, const BatchRun *runs, int nruns, int total, int blocks,
                                   int np, bool nonlin, bool cpml, hipStream_t s)
{
#define MPX_FEB(NPV, NL, CP)                                                                                    \
    hipLaunchKernelGGL((k_fused_E_batch<T, NPV, NL, CP, L>), dim3(blocks), dim3(64, 4), 0, s, args, runs, nruns, \
                       total)
#define MPX_FEB_NP(NL, CP)             \
    switch (np) {                      \
    case 0: MPX_FEB(0, NL, CP); break; \
    case 1: MPX_FEB(1, NL, CP); break; \
    case 2: MPX_FEB(2, NL, CP); break; \
    default: MPX_FEB(3, NL, CP); break; \
    }
    if (nonlin) {
        if (cpml) { MPX_FEB_NP(true, true) } else { MPX_FEB_NP(true, false) }
    } else {
        if (cpml) { MPX_FEB_NP(false, true) } else { MPX_FEB_NP(false, false) }
    }
#undef MPX_FEB_NP
#undef MPX_FEB
}

template <typename T>
void launch_fused_E_batch(const StepArgs<T> *args, const BatchRun *runs, int nruns, int total, int blocks, int L,
                          int np, bool nonlin, bool cpml, hipStream_t s)
{
    (void)L;  // the batch walks one plane per thread on the E side
    launch_fused_E_batch_L<T, 1>(args, runs, nruns, total, blocks, np, nonlin, cpml, s);
}

template <typename T, int L>
static void launch_fused_B_batch_L(const StepArgs<T> *args, const BatchRun *runs, int nruns, int total, int blocks,
                                   bool cpml, hipStream_t s)
{
    if (cpml)
        hipLaunchKernelGGL((k_fused_B_batch<T, true, L>), dim3(blocks), dim3(64, 4), 0, s, args, runs, nruns, total);
    else
        hipLaunchKernelGGL((k_fused_B_batch<T, false, L>), dim3(blocks), dim3(64, 4), 0, s, args, runs, nruns, total);
}

template <typename T>
void launch_fused_B_batch(const StepArgs<T> *args, const BatchRun *runs, int nruns, int total, int blocks, int L,
                          bool cpml, hipStream_t s)
{
    switch (L) {
    case 2: launch_fused_B_batch_L<T, 2>(args, runs, nruns, total, blocks, cpml, s); break;
    case 4: launch_fused_B_batch_L<T, 4>(args, runs, nruns, total, blocks, cpml, s); break;
    default: launch_fused_B_batch_L<T, 1>(args, runs, nruns, total, blocks, cpml, s); break;
    }
}
#if MPX_FORM == 0
template void launch_fused_E_batch<double>(const StepArgs<double> *, const BatchRun *, int, int, int, int, int, bool,
                                           bool, hipStream_t);
template void launch_fused_B_batch<double>(const StepArgs<double> *, const BatchRun *, int, int, int, int, bool,
                                           hipStream_t);
#else
template void launch_fused_E_batch<float>(const StepArgs<float> *, const BatchRun *, int, int, int, int, int, bool,
                                          bool, hipStream_t);
template void launch_fused_B_batch<float>(const StepArgs<float> *, const BatchRun *, int, int, int, int, bool,
                                          hipStream_t);
#endif

template <typename T, int L, bool RES = false>
static void launch_fused_E_L(const StepArgs<T> &a, const StepArgs<T> *dev, int np, bool nonlin, int soff,
                             hipStream_t s)
{
    const GridDims &g = a.g;
    int nbx = (g.n[2] + 63) / 64, nby = (g.n[1] + 3) / 4, nbz = (g.n[0] + L - 1) / L;
    dim3 blk(64, 4);
    dim3 grd(nbx, nby, nbz);
    bool cp = a.nfaces > 0;
#define MPX_FE(NPV, NL, CP) hipLaunchKernelGGL((k_fused_E<T, NPV, NL, CP, L, RES>), grd, blk, 0, s, dev, nbx, nby, nbz, soff)
#define MPX_FE_NP(NL, CP)            \
    switch (np) {                    \
    case 0: MPX_FE(0, NL, CP); break; \
    case 1: MPX_FE(1, NL, CP); break; \
    case 2: MPX_FE(2, NL, CP); break; \
    default: MPX_FE(3, NL, CP); break; \
    }
    if (nonlin) {
        if (cp) { MPX_FE_NP(true, true) } else { MPX_FE_NP(true, false) }
    } else {
        if (cp) { MPX_FE_NP(false, true) } else { MPX_FE_NP(false, false) }
    }
#undef MPX_FE_NP
#undef MPX_FE
}

template <typename T>
void launch_fused_E(const StepArgs<T> &a, const StepArgs<T> *dev, int np, bool nonlin, int soff, hipStream_t s)
{
    if constexpr (sizeof(T) == 4) {
        // float32 + residual storage: one plane per thread (the march of the float32 default)
        if (a.Elo) {
            launch_fused_E_L<T, 1, true>(a, dev, np, nonlin, soff, s);
            return;
        }
    }
    switch (a.march) {
    case 2: launch_fused_E_L<T, 2>(a, dev, np, nonlin, soff, s); break;
    case 4: launch_fused_E_L<T, 4>(a, dev, np, nonlin, soff, s); break;
    default: launch_fused_E_L<T, 1>(a, dev, np, nonlin, soff, s); break;
    }
}

template <typename T, int L, bool RES = false>
static void launch_fused_B_L(const StepArgs<T> &a, const StepArgs<T> *dev, int soff, hipStream_t s)
{
    const GridDims &g = a.g;
    int nk = g.n[2] - a.blo[2] + 1, nj = g.n[1] - a.blo[1] + 1, ni = g.n[0] - a.blo[0] + 1;
    int nbx = (nk + 63) / 64, nby = (nj + 3) / 4, nbz = (ni + L - 1) / L;
    dim3 blk(64, 4);
    dim3 grd(nbx, nby, nbz);
    if (a.nfaces > 0)
        hipLaunchKernelGGL((k_fused_B<T, true, L, RES>), grd, blk, 0, s, dev, nbx, nby, nbz, soff);
    else
        hipLaunchKernelGGL((k_fused_B<T, false, L, RES>), grd, blk, 0, s, dev, nbx, nby, nbz, soff);
}

template <typename T>
void launch_fused_B(const StepArgs<T> &a, const StepArgs<T> *dev, int soff, hipStream_t s)
{
    if constexpr (sizeof(T) == 4) {
        // float32 + residual storage: one or two planes per thread
        if (a.Blo) {
            if (a.march == 1)
                launch_fused_B_L<T, 1, true>(a, dev, soff, s);
            else
                launch_fused_B_L<T, 2, true>(a, dev, soff, s);
            return;
        }
    }
    switch (a.march) {
    case 2: launch_fused_B_L<T, 2>(a, dev, soff, s); break;
    case 4: launch_fused_B_L<T, 4>(a, dev, soff, s); break;
    default: launch_fused_B_L<T, 1>(a, dev, soff, s); break;
    }
}

#if MPX_FORM == 0
template void launch_fused_E<double>(const StepArgs<double> &, const StepArgs<double> *, int, bool, int, hipStream_t);
template void launch_fused_B<double>(const StepArgs<double> &, const StepArgs<double> *, int, hipStream_t);
#else
template void launch_fused_E<float>(const StepArgs<float> &, const StepArgs<float> *, int, bool, int, hipStream_t);
template void launch_fused_B<float>(const StepArgs<float> &, const StepArgs<float> *, int, hipStream_t);
#endif

}  // namespace mpx
