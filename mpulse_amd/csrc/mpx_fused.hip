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

// A cell's place.  Blocks of 64 z cells x 4 rows: a wave holds cells of one row, so the row's
// offset is wave-uniform and a lane adds k alone -- one 32-bit offset register for every grid
// and neighbour row, where an index of its own took a 64-bit address for each.  LIN blocks (256
// consecutive y-z cells) cross rows and keep a lane's own index.
template <bool LIN>
struct At;
template <>
struct At<false> {
    size_t row;  // storage offset of k = 0
    unsigned k;
    __device__ __forceinline__ At shift(int d) const { return {row + (long long)d, k}; }  // d: wave-uniform
    __device__ __forceinline__ At along(int d) const { return {row, k + d}; }
    template <typename T>
    __device__ __forceinline__ T ld(const T *p) const
    {
        return ldp(p + row, k * (unsigned)sizeof(T));
    }
    template <typename T>
    __device__ __forceinline__ T once(const T *p) const
    {
        return ldp_once(p + row, k * (unsigned)sizeof(T));
    }
    template <typename T>
    __device__ __forceinline__ void st(T *p, T v) const
    {
        stp(p + row, k * (unsigned)sizeof(T), v);
    }
    template <typename T>
    __device__ __forceinline__ void st_once(T *p, T v) const
    {
        stp_once(p + row, k * (unsigned)sizeof(T), v);
    }
    // the accumulators (psi_at): the row's chunk is uniform, a lane counts on from it
    __device__ __forceinline__ size_t psi_row() const { return psi_base(row); }
    __device__ __forceinline__ unsigned psi_lane() const { return psi_ahead(row, k); }
};
template <>
struct At<true> {
    int c;
    __device__ __forceinline__ At shift(int d) const { return {c + d}; }
    __device__ __forceinline__ At along(int d) const { return {c + d}; }
    template <typename T>
    __device__ __forceinline__ T ld(const T *p) const
    {
        return gld(p + c);
    }
    template <typename T>
    __device__ __forceinline__ T once(const T *p) const
    {
        return load_once(p + c);
    }
    template <typename T>
    __device__ __forceinline__ void st(T *p, T v) const
    {
        gst(p + c, v);
    }
    template <typename T>
    __device__ __forceinline__ void st_once(T *p, T v) const
    {
        store_once(p + c, v);
    }
    // the accumulators count on from the wave's first cell, its lowest: psi_at itself as a 32-bit lane
    // offset wrapped at 4 GiB, storage cell 89478464 (a cube of 431^3)
    __device__ __forceinline__ unsigned first() const { return (unsigned)__builtin_amdgcn_readfirstlane(c); }
    __device__ __forceinline__ size_t psi_row() const { return psi_base(first()); }
    __device__ __forceinline__ unsigned psi_lane() const { return psi_ahead(first(), (unsigned)c - first()); }
};

// Two or three components of a cell and its residual word, as stored
template <typename T, bool RES>
struct Words {
    T x, y, z;
    unsigned w;
};
template <bool RES, typename A, typename T>
__device__ __forceinline__ Words<T, RES> read3(const A &at, const T *const f[3], const unsigned *lo)
{
    Words<T, RES> r;
    r.x = at.ld(f[0]);
    r.y = at.ld(f[1]);
    r.z = at.ld(f[2]);
    r.w = RES ? at.ld(lo) : 0u;
    return r;
}
template <bool RES, typename A, typename T>
__device__ __forceinline__ Words<T, RES> read3_once(const A &at, const T *const f[3], const unsigned *lo)
{
    Words<T, RES> r;
    r.x = at.once(f[0]);
    r.y = at.once(f[1]);
    r.z = at.once(f[2]);
    r.w = RES ? at.once(lo) : 0u;
    return r;
}
// components p and q only
template <typename T, bool RES>
struct Pair {
    T p, q;
    unsigned w;
};
template <bool RES, typename A, typename T>
__device__ __forceinline__ Pair<T, RES> read2(const A &at, const T *fp, const T *fq, const unsigned *lo)
{
    Pair<T, RES> r;
    r.p = at.ld(fp);
    r.q = at.ld(fq);
    r.w = RES ? at.ld(lo) : 0u;
    return r;
}

// accumulators of the active poles at a cell: component q of pole n sits 64 elements after
// component q - 1
template <int NP, bool LIN>
struct PsiCell {
    double2 *b[NP > 0 ? NP : 1];
    struct Comp {
        double2 *p;
        __device__ double2 &operator[](size_t) const { return *p; }
    };
    struct Pole {
        double2 *p;
        __device__ Comp operator[](int q) const { return Comp{p + 64 * q}; }
    };
    __device__ Pole operator[](int n) const { return Pole{b[n]}; }
};

// Fused E side of one step.  A thread owns one (j, k) column segment of L cells along x and
// walks it plane by plane, keeping B of the previous plane in registers for the x difference.
//
// Bound by memory latency at the occupancy its registers allow: a wave's life is one round of
// loads, the update and its stores, so whatever waits for memory before that round is issued
// adds a latency to every wave.  Every word of a cell -- its own, the three lower neighbours',
// the accumulators', the CPML auxiliaries' -- is therefore requested unconditionally before the
// first is used.  The z - 1 neighbour is in the previous lane (DPP) except for the first lane of
// a wave and the first cell of a row.  With residuals that word too is loaded by all lanes (at
// their own cell's address where it is not needed), since under a branch its decoding waited for it
// at once; a plain word has nothing to wait for there, and the lanes that need it load it (all / those,
// float64: 64^3 with one pole and plasma 12.6 / 11.6, 131x158x177 120 / 117).
// Measured against the form before (face by face CPML, per-lane 64-bit addresses, tile divisions in
// the kernel), us for E + B with a 16-cell CPML, one pole and the pulse under way: 512^3 float32 +
// residual 3616 + 1709 -> 3533 + 1447, float32 3191 + 1058 -> 3179 + 1066, float64 4235 + 2160 -> 4197 +
// 2187; 256^3 float32 + residual 509 + 271 -> 470 + 232, float32 418 + 180 -> 402 + 182; 64^3 float64, 4-cell
// layers, 13.5 + 12.3 -> 12.8 + 9.8.
template <typename T, int NP, bool NONLIN, bool CPML, int L, bool LIN = false, bool RES = false>
__device__ __forceinline__ void fused_E_tile(const StepArgs<T> &a, int tbx, int tby, int tbz, int soff)
{
    const GridDims &g = a.g;
    const int one[3] = {1, 1, 1};
    int j, k;
    tile_jk<LIN>(g, one, tbx, tby, j, k);
    if (!LIN) j = __builtin_amdgcn_readfirstlane(j);
    const int i0 = tbz * L + 1;
    if (k > g.n[2] || j > g.n[1] || i0 > g.n[0]) return;
    const int i1 = min(i0 + L - 1, g.n[0]);
    const int sx = (int)g.sx, pz = g.pz;
    const int ojm = (j == 1 && a.periodic[1]) ? (g.n[1] - 1) * pz : -pz;
    const int okm = (k == 1 && a.periodic[2]) ? (g.n[2] - 1) : -1;
    const int oim = (i0 == 1 && a.periodic[0]) ? (g.n[0] - 1) * sx : -sx;
    At<LIN> c;
    if constexpr (LIN) c = {i0 * sx + j * pz + k + g.z0};
    else c = {g.at(i0, j, 0), (unsigned)k};
    const T *const *B = a.B;
    const bool zload = threadIdx.x == 0 || k == 1;
    const Pair<T, RES> bim = read2<RES>(c.shift(oim), B[1], B[2], a.Blo);
    double by_im = 0.0, bz_im = 0.0;
    const double kdy = LIN ? gld(a.ikdE[1] + j) : kload(a.ikdE[1] + j), kdz = gld(a.ikdE[2] + k);
#pragma unroll
    for (int u = 0; u < L; ++u) {
        const int i = i0 + u;
        if (i > i1) break;
        const Words<T, RES> b = read3<RES>(c, B, a.Blo);
        Pair<T, RES> bk;
        if constexpr (RES) bk = read2<RES>(c.along(zload ? okm : 0), B[0], B[1], a.Blo);
        else if (zload) bk = read2<RES>(c.along(okm), B[0], B[1], a.Blo);
        const Pair<T, RES> bj = read2<RES>(c.shift(ojm), B[0], B[2], a.Blo);
        const Words<T, RES> e = read3_once<RES>(c, (const T *const *)a.E, a.Elo);
        const size_t prow = c.psi_row();
        const unsigned plane = c.psi_lane();
        PsiRegs<NP> pr;
        PsiCell<NP, LIN> ps;
#pragma unroll
        for (int n = 0; n < NP; ++n) {
            ps.b[n] = a.psi[n][0] + prow + plane;
#pragma unroll
            for (int q = 0; q < 3; ++q) pr.v[n][q] = ldp_once(a.psi[n][0] + prow + 64 * q, plane * 16u);
        }
        CellCpml<T, RES> cx;
        if (CPML) cpml_request<T, RES>(a.cd, i, j, k, true, cx);
        double epsc = 0.0;
        if (a.epsf) epsc = c.ld(a.epsf);
        const double bx = got<T, RES>(b.x, b.w, 0), by = got<T, RES>(b.y, b.w, 1), bz = got<T, RES>(b.z, b.w, 2);
        if (u == 0) {
            by_im = got<T, RES>(bim.p, bim.w, 1);
            bz_im = got<T, RES>(bim.q, bim.w, 2);
        }
        double ex = got<T, RES>(e.x, e.w, 0), ey = got<T, RES>(e.y, e.w, 1), ez = got<T, RES>(e.z, e.w, 2);
        const double dBz_y = bz - got<T, RES>(bj.q, bj.w, 2);
        const double dBx_y = bx - got<T, RES>(bj.p, bj.w, 0);
        double bxs, bys;
        if constexpr (RES) {
            bxs = lane_prev(bx);
            bys = lane_prev(by);
        } else {
            bxs = (double)lane_prev(b.x);
            bys = (double)lane_prev(b.y);
        }
        const double dBx_z = bx - (zload ? got<T, RES>(bk.p, bk.w, 0) : bxs);
        const double dBy_z = by - (zload ? got<T, RES>(bk.q, bk.w, 1) : bys);
        const double dBz_x = bz - bz_im;
        const double dBy_x = by - by_im;
        bz_im = bz;
        by_im = by;
        // the plasma OptField and the plasma current run before the E update, on E of this step
        double sg = 0.0, jpv[3] = {0.0, 0.0, 0.0};
        if (a.plasma || a.pcur) {
            double r = c.ld(a.rho);
            double jp[3] = {0.0, 0.0, 0.0};
            if (a.pcur)
                for (int q = 0; q < 3; ++q) jp[q] = c.ld(a.jp[q]);
            if (a.plasma) {
                sg = a.pw * plasma_density_cell(ex, ey, ez, r, a.pn, a.pm, a.pk - 1);
                c.st(a.rho, r);
                c.st(a.sigma, sg);
            }
            if (a.pcur) {
                const double rt = r + a.rho_bg, ev[3] = {ex, ey, ez};
                for (int q = 0; q < 3; ++q) {
                    jpv[q] = plasma_current_comp(jp[q], ev[q], rt, a.gdtn, a.gdtd, a.emdt);
                    c.st(a.jp[q], jpv[q]);
                }
            }
        }
        // current totals in list order: the CPML and sheet groups, the plasma current at its place
        double J[3] = {0.0, 0.0, 0.0};
        auto add_cpml = [&]() {
            if (CPML) {
                const double df[3][2] = {{dBy_x, dBz_x}, {dBz_y, dBx_y}, {dBx_z, dBy_z}};
                cpml_add<T, false, RES>(a.cd, i, j, k, cx, df, true, J);
            }
        };
        auto add_plasma = [&](int pos) {
            if (a.pcur && a.pcur_pos == pos) {
                J[0] += jpv[0];
                J[1] += jpv[1];
                J[2] += jpv[2];
            }
        };
        add_plasma(0);
        if (a.sheets_first)
            add_sheets(a, i, j, k, soff, J[0], J[1], J[2]);
        else
            add_cpml();
        add_plasma(1);
        if (a.sheets_first)
            add_cpml();
        else
            add_sheets(a, i, j, k, soff, J[0], J[1], J[2]);
        add_plasma(2);
        double idenom = a.idenom, numer = a.numer;
        if (a.epsf || a.plasma) {  // cell_eps with the permittivity read above and Sigma dt / 2
            const double ec = a.epsf ? epsc : a.eps, sgh = 0.5 * sg * a.dt;
            const double denom = NONLIN ? ec + a.sumChi0 - a.sumXi0 + sgh : ec + (a.sumChi0 - a.sumXi0) + sgh;
            numer = ec - a.sumXi0 - sgh;
            idenom = 1.0 / denom;
        }
        unsigned fl = 0;
        plrc_e_update_pp<NP, NONLIN, true>(ex, ey, ez, dBz_y, dBy_z, dBx_z, dBz_x, dBy_x, dBx_y, kload(a.ikdE[0] + i), kdy,
                                           kdz, J[0], J[1], J[2], pr, ps, (size_t)0, true, a.pc, a.dt, idenom, numer,
                                           a.chi, a.ncap, &fl);
        report(a.status, fl | finite_flag(ex, ey, ez));
        unsigned wn = 0;
        const T hx = put<T, RES>(ex, wn, 0), hy = put<T, RES>(ey, wn, 1), hz = put<T, RES>(ez, wn, 2);
        c.st_once(a.En[0], hx);
        c.st_once(a.En[1], hy);
        c.st_once(a.En[2], hz);
        if (RES) c.st_once(a.Elo, wn);
        c = c.shift(sx);
    }
}

// Fused B side of one step: a thread walks L planes along x keeping E of the next plane as the
// centre of the following iteration.  Bound and built as the E side: every word of the L planes
// is requested before the first is used, the z + 1 neighbour by all lanes with residuals, else by
// those that need it (float64 two planes 256^3 all / those 280 / 276, without layers 222 / 214).  Plain
// float32 loads a layer's auxiliaries where they are used: ahead of their use they cost it registers
// (78 against 66 for two planes) that its waves are worth more.  Two planes with the auxiliaries ahead
// and all lanes loading / as it is, us: layers of 8 cells 128^3 25.5 / 23.9, 200^3 93.1 / 82.3, 256^3
// 161 / 142, 320^3 258 / 234; without layers 200^3 68.7 / 63.6.
template <typename T, bool CPML, int L, bool LIN = false, bool RES = false>
__device__ __forceinline__ void fused_B_tile(const StepArgs<T> &a, int tbx, int tby, int tbz, int soff)
{
    constexpr bool F32 = sizeof(T) == 4 && !RES;
    const GridDims &g = a.g;
    int j, k;
    tile_jk<LIN>(g, a.blo, tbx, tby, j, k);
    if (!LIN) j = __builtin_amdgcn_readfirstlane(j);
    const int i0 = tbz * L + a.blo[0];
    if (k > g.n[2] || j > g.n[1] || i0 > g.n[0]) return;
    const int i1 = min(i0 + L - 1, g.n[0]);
    const int sx = (int)g.sx, pz = g.pz;
    const int ojp = (j == g.n[1] && a.periodic[1]) ? -(g.n[1] - 1) * pz : pz;
    const int okp = (k == g.n[2] && a.periodic[2]) ? -(g.n[2] - 1) : 1;
    At<LIN> c;
    if constexpr (LIN) c = {i0 * sx + j * pz + k + g.z0};
    else c = {g.at(i0, j, 0), (unsigned)k};
    const T *const *E = a.E;
    const bool zload = threadIdx.x == 63 || k == g.n[2];
    // per plane: E of the next plane, E_x and E_z of the next row, E_x and E_y of the next cell, B
    const Words<T, RES> ec = read3<RES>(c, E, a.Elo);
    Words<T, RES> en[L], b0[L];
    Pair<T, RES> ej[L], ek[L];
#pragma unroll
    for (int u = 0; u < L; ++u) {
        const int i = i0 + u;
        if (i > i1) break;
        const At<LIN> cu = c.shift(u * sx);
        en[u] = read3<RES>(cu.shift((i == g.n[0] && a.periodic[0]) ? -(g.n[0] - 1) * sx : sx), E, a.Elo);
        ej[u] = read2<RES>(cu.shift(ojp), E[0], E[2], a.Elo);
        if constexpr (RES) ek[u] = read2<RES>(cu.along(zload ? okp : 0), E[0], E[1], a.Elo);
        else if (zload) ek[u] = read2<RES>(cu.along(okp), E[0], E[1], a.Elo);
        b0[u] = read3_once<RES>(cu, (const T *const *)a.B, a.Blo);
    }
    CellCpml<T, RES> cx;
    if (CPML && !F32) cpml_request<T, RES>(a.cd, i0, j, k, true, cx);
    const double kdy = LIN ? gld(a.ikdH[1] + j) : kload(a.ikdH[1] + j), kdz = gld(a.ikdH[2] + k);
    T rx = ec.x, ry = ec.y;  // E_x, E_y of the centre as stored (float32 and float64)
    double ex = got<T, RES>(ec.x, ec.w, 0), ey = got<T, RES>(ec.y, ec.w, 1), ez = got<T, RES>(ec.z, ec.w, 2);
#pragma unroll
    for (int u = 0; u < L; ++u) {
        const int i = i0 + u;
        if (i > i1) break;
        const double ex1 = got<T, RES>(en[u].x, en[u].w, 0), ey1 = got<T, RES>(en[u].y, en[u].w, 1),
                     ez1 = got<T, RES>(en[u].z, en[u].w, 2);
        double exs, eys;
        if constexpr (RES) {
            exs = lane_next(ex);
            eys = lane_next(ey);
        } else {
            exs = (double)lane_next(rx);
            eys = (double)lane_next(ry);
        }
        const double dEx_z = (zload ? got<T, RES>(ek[u].p, ek[u].w, 0) : exs) - ex;
        const double dEy_z = (zload ? got<T, RES>(ek[u].q, ek[u].w, 1) : eys) - ey;
        const double dEx_y = got<T, RES>(ej[u].p, ej[u].w, 0) - ex;
        const double dEz_y = got<T, RES>(ej[u].q, ej[u].w, 2) - ez;
        const double dEz_x = ez1 - ez;
        const double dEy_x = ey1 - ey;
        double M[3] = {0.0, 0.0, 0.0};
        if (a.sheets_first) add_sheets(a, i, j, k, soff, M[0], M[1], M[2]);
        if (CPML) {
            const double df[3][2] = {{dEy_x, dEz_x}, {dEz_y, dEx_y}, {dEx_z, dEy_z}};
            if constexpr (F32) {
                cpml_each<T, true, RES>(a.cd, i, j, k, df, M);
            } else {
                const CellCpml<T, RES> now = cx;
                if (u + 1 < L && i < i1) cpml_request<T, RES>(a.cd, i + 1, j, k, true, cx);  // the next plane's
                cpml_add<T, true, RES>(a.cd, i, j, k, now, df, true, M);
            }
        }
        if (!a.sheets_first) add_sheets(a, i, j, k, soff, M[0], M[1], M[2]);
        const double kdx = kload(a.ikdH[0] + i);
        unsigned wn = 0;
        const T hx = put<T, RES>(got<T, RES>(b0[u].x, b0[u].w, 0) + a.dt * ((dEy_z * kdz - dEz_y * kdy) + M[0]), wn, 0);
        const T hy = put<T, RES>(got<T, RES>(b0[u].y, b0[u].w, 1) + a.dt * ((dEz_x * kdx - dEx_z * kdz) + M[1]), wn, 1);
        const T hz = put<T, RES>(got<T, RES>(b0[u].z, b0[u].w, 2) + a.dt * ((dEx_y * kdy - dEy_x * kdx) + M[2]), wn, 2);
        const At<LIN> cu = c.shift(u * sx);
        cu.st_once(a.B[0], hx);
        cu.st_once(a.B[1], hy);
        cu.st_once(a.B[2], hz);
        if (RES) cu.st_once(a.Blo, wn);
        ex = ex1;
        ey = ey1;
        ez = ez1;
        rx = en[u].x;
        ry = en[u].y;
    }
}

// The argument block is read from device memory, where the solver keeps a copy: one upload when it
// changes instead of 2 KB of kernel arguments a launch.  Nothing here indexes it at run time, so a
// compact by-value block is possible and would spare the head of a wave one dependent scalar load;
// it has not been measured.
// Waves per SIMD the E kernel is compiled for: 6 (at most 80 registers) for the float32 Kerr
// kernel with one pole and one plane per thread, measured 0.3 % faster than the 5 its registers
// allow; no constraint otherwise (other variants would spill).
template <typename T, int NP, bool NONLIN, int L, bool RES>
struct FusedEWaves {
    static constexpr int v = (sizeof(T) == 4 && !RES && NP <= 1 && NONLIN && L == 1) ? 6 : 1;
};

template <typename T, int NP, bool NONLIN, bool CPML, int L, bool RES = false>
__global__ __attribute__((amdgpu_waves_per_eu(FusedEWaves<T, NP, NONLIN, L, RES>::v))) __launch_bounds__(256) void k_fused_E(
    const StepArgs<T> *__restrict__ pa, TileMap map, int soff)
{
    int tbx, tby, tbz;
    if (!map_tile(map, tbx, tby, tbz)) return;
    fused_E_tile<T, NP, NONLIN, CPML, L, false, RES>(*pa, tbx, tby, tbz, soff);
}

template <typename T, bool CPML, int L, bool RES = false>
__global__ __launch_bounds__(256) void k_fused_B(const StepArgs<T> *__restrict__ pa, TileMap map, int soff)
{
    int tbx, tby, tbz;
    if (!map_tile(map, tbx, tby, tbz)) return;
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

// The block order of a launch.  bytes: what a cell without layers reads and writes; a layer adds the
// reads and writes of two auxiliaries (and their residual word).  Shares of equal work from 2048 tiles
// on (eight blocks a CU), where the XCDs run long enough to end at different times; equal / balanced, us
// a step with layers of 6 to 16 cells: 96x88x120 84.4 / 82.2, 131x158x177 211.5 / 207.6 (float32 +
// residual 179.4 / 175.0), 256^3 925 / 899 (748 / 726; float32 615 / 607), 512^3 4998 / 4980.
template <typename T>
static TileMap fused_map(const StepArgs<T> &a, int nbx, int nby, int nbz, int L, int j0, int i0, double bytes)
{
    TileMap m = tile_map(nbx, nby, nbz, a.order, a.band, a.rev);
    if (a.order == 2 && a.nfaces > 0 && m.total >= 2048)
        balance_shares(m, nbx, nby, nbz, L, j0, i0, a.cd, (4.0 * sizeof(T) + (a.Elo ? 8 : 0)) / bytes);
    return m;
}

template <typename T, int L, bool RES = false>
static void launch_fused_E_L(const StepArgs<T> &a, const StepArgs<T> *dev, int np, bool nonlin, int soff,
                             hipStream_t s)
{
    const GridDims &g = a.g;
    int nbx = (g.n[2] + 63) / 64, nby = (g.n[1] + 3) / 4, nbz = (g.n[0] + L - 1) / L;
    const TileMap map = fused_map<T>(a, nbx, nby, nbz, L, 1, 1, (3 * 3 * sizeof(T) + (RES ? 3 * 4 : 0)) + 96.0 * np);
    dim3 blk(64, 4), grd(tile_blocks(map));
    bool cp = a.nfaces > 0;
#define MPX_FE(NPV, NL, CP) hipLaunchKernelGGL((k_fused_E<T, NPV, NL, CP, L, RES>), grd, blk, 0, s, dev, map, soff)
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
    const TileMap map = fused_map<T>(a, nbx, nby, nbz, L, a.blo[1], a.blo[0], 3 * 3 * sizeof(T) + (RES ? 3 * 4 : 0));
    dim3 blk(64, 4), grd(tile_blocks(map));
    if (a.nfaces > 0)
        hipLaunchKernelGGL((k_fused_B<T, true, L, RES>), grd, blk, 0, s, dev, map, soff);
    else
        hipLaunchKernelGGL((k_fused_B<T, false, L, RES>), grd, blk, 0, s, dev, map, soff);
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
