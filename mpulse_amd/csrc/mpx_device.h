// Device helpers shared by the gfx950 kernel files: global-address loads and stores,
// nontemporal streams, DPP lane shuffles, the PLRC + Kerr E update core, the CPML face
// update, the float32 + residual storage form, tile maps.
#pragma once
#include <hip/hip_runtime.h>

#include "mpx_types.h"

namespace mpx {

// ------------------------------------------------------------------------------------
// PLRC + Kerr E update core, shared by both paths:
// FDTD_PLRCNonlinCore::plrcStepD src/fdtd_plrc.cpp:304-427,
// FDTD_PLRCLinCore::plrcStepD    src/fdtd_plrc.cpp:94-261.
// d* are the B differences in the reference's order, kd* the kappa*delta factors.
// ------------------------------------------------------------------------------------
// Every grid, table and layer pointer of the solver points into hipMalloc'd memory.  Kernels
// that read their argument block from device memory see those pointers as generic ones, and
// generic (flat) accesses also count against the scalar-load counter, so each wait for an
// argument load would wait for the outstanding grid loads too.  gld / gst access through the
// global address space instead.
#define MPX_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ T gld(const T *p)
{
    return *(const MPX_GLOBAL T *)p;
}
template <typename T>
__device__ __forceinline__ void gst(T *p, T v)
{
    *(MPX_GLOBAL T *)p = v;
}

// Words a launch touches exactly once (the pole accumulators, a cell's own E in the E kernel
// and B in the B kernel) move with nontemporal loads and stores: they then do not evict from L2
// the neighbour planes that other threads of the launch re-read.
typedef double double2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double2 load_once(const double2 *p)
{
    const double2v v = __builtin_nontemporal_load((const MPX_GLOBAL double2v *)p);
    return make_double2(v.x, v.y);
}
__device__ __forceinline__ void store_once(double2 *p, double2 v)
{
    double2v w;
    w.x = v.x;
    w.y = v.y;
    __builtin_nontemporal_store(w, (MPX_GLOBAL double2v *)p);
}
template <typename T>
__device__ __forceinline__ T load_once(const T *p)
{
    return __builtin_nontemporal_load((const MPX_GLOBAL T *)p);
}
template <typename T>
__device__ __forceinline__ void store_once(T *p, T v)
{
    __builtin_nontemporal_store(v, (MPX_GLOBAL T *)p);
}

// Word at byte offset bo (per lane, 32 bits) from the wave-uniform address `base` of a row or of
// a plane (of (ny + 2) pz words < 2^32 bytes): a scalar base and one offset register for all the
// grids a lane reads at its cell, instead of a 64-bit address each
template <typename T>
__device__ __forceinline__ T ldp(const T *base, unsigned bo)
{
    return gld((const T *)((const char *)base + bo));
}
template <typename T>
__device__ __forceinline__ void stp_once(T *base, unsigned bo, T v)
{
    store_once((T *)((char *)base + bo), v);
}
template <typename T>
__device__ __forceinline__ T ldp_once(const T *base, unsigned bo)
{
    return load_once((const T *)((const char *)base + bo));
}
template <typename T>
__device__ __forceinline__ void stp(T *base, unsigned bo, T v)
{
    gst((T *)((char *)base + bo), v);
}

// A read-only table entry at a wave-uniform address, through the constant address space: a
// scalar load into SGPRs, counted apart from the vector loads in flight
__device__ __forceinline__ double kload(const double *p)
{
    return *(const __attribute__((address_space(4))) double *)p;
}

// The value a neighbouring lane of the wavefront holds, by DPP: lane_prev gives lane l the
// value of lane l - 1 (wave_shr:1), lane_next that of lane l + 1 (wave_shl:1).  Lanes of a
// fused-kernel wave hold consecutive z cells of one row, so the z neighbour of a cell is in
// the next lane except at the ends of the wave and of the row, where it is loaded.
__device__ __forceinline__ float lane_prev(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_next(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, false));
}
__device__ __forceinline__ double lane_prev(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x138, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x138, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double lane_next(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x130, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x130, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Storage forms of a field word: T (float64 or float32) on its own, or (RES, T = float) the
// float32 word plus a slot of the cell's residual word (res_encode / res_decode).  V is the
// type a loaded value is carried in: T itself, or the decoded float64 value.
template <typename T, bool RES>
struct Word {
    using V = T;
};
template <>
struct Word<float, true> {
    using V = double;
};
// the residual word of cell c (0 without residual storage: nothing is loaded)
template <bool RES>
__device__ __forceinline__ unsigned lo_ld(const unsigned *lo, size_t c)
{
    if constexpr (RES) return gld(lo + c);
    else return 0u;
}
template <bool RES>
__device__ __forceinline__ unsigned lo_once(const unsigned *lo, size_t c)
{
    if constexpr (RES) return load_once(lo + c);
    else return 0u;
}
// component q of cell c, read from its word array p and the residual word w
template <typename T, bool RES>
__device__ __forceinline__ typename Word<T, RES>::V rd(const T *p, unsigned w, int q, size_t c)
{
    if constexpr (RES) return res_decode(gld(p + c), w, q);
    else return gld(p + c);
}
template <typename T, bool RES>
__device__ __forceinline__ typename Word<T, RES>::V rd_once(const T *p, unsigned w, int q, size_t c)
{
    if constexpr (RES) return res_decode(load_once(p + c), w, q);
    else return load_once(p + c);
}
// the word stored for x (its residual OR-ed into slot q of w), and the value that word holds
template <typename T, bool RES>
__device__ __forceinline__ T put(double x, unsigned &w, int q)
{
    if constexpr (RES) return res_encode(x, w, q);
    else return (T)x;
}
template <typename T, bool RES>
__device__ __forceinline__ double got(T h, unsigned w, int q)
{
    if constexpr (RES) return res_decode(h, w, q);
    else return (double)h;
}

// quotient x / k, or x * k when k already holds the reciprocal (RECIP)
template <bool RECIP>
__device__ __forceinline__ double qt(double x, double k)
{
    return RECIP ? x * k : x / k;
}

// RECIP: kdx, kdy, kdz and denom hold reciprocals (1/(kappa delta), 1/denom) and the divisions
// become products; otherwise the reference's quotients are formed.
template <int NP, bool NONLIN, bool RECIP, typename PIN, typename POUT>
__device__ __forceinline__ void plrc_e_update_pp(double &ex, double &ey, double &ez, double dBz_y, double dBy_z,
                                                 double dBx_z, double dBz_x, double dBy_x, double dBx_y,
                                                 double kdx, double kdy, double kdz, double jx, double jy,
                                                 double jz, const PIN &psi_in, const POUT &psi, size_t c,
                                                 bool store, const PoleConsts &pc, double dt, double denom,
                                                 double numer, double chi, int ncap = kNewtonCap,
                                                 unsigned *flag = nullptr)
{
    double Psix = 0, Psiy = 0, Psiz = 0;
    const size_t pq = psi_at(c);
#pragma unroll
    for (int n = 0; n < NP; ++n) {
        double2 px = psi_in[n][0][pq], py = psi_in[n][1][pq], pz = psi_in[n][2][pq];
        const double2 D = pc.dd[n], X = pc.dxi0[n], C = pc.crec[n];
        double pxr = D.x * ex + px.x, pxi = D.y * ex + px.y;
        double pyr = D.x * ey + py.x, pyi = D.y * ey + py.y;
        double pzr = D.x * ez + pz.x, pzi = D.y * ez + pz.y;
        Psix += pxr;
        Psiy += pyr;
        Psiz += pzr;
        if (store) {
            store_once(&psi[n][0][pq], make_double2(X.x * ex + (C.x * pxr - C.y * pxi), X.y * ex + (C.x * pxi + C.y * pxr)));
            store_once(&psi[n][1][pq], make_double2(X.x * ey + (C.x * pyr - C.y * pyi), X.y * ey + (C.x * pyi + C.y * pyr)));
            store_once(&psi[n][2][pq], make_double2(X.x * ez + (C.x * pzr - C.y * pzi), X.y * ez + (C.x * pzi + C.y * pzr)));
        }
    }
    if (NONLIN) {
        double E2 = ex * ex + ey * ey + ez * ez;
        double f = numer + chi * E2;
        double cx = qt<RECIP>(f * ex + dt * ((qt<RECIP>(dBz_y, kdy) - qt<RECIP>(dBy_z, kdz)) + jx) + Psix, denom);
        double cy = qt<RECIP>(f * ey + dt * ((qt<RECIP>(dBx_z, kdz) - qt<RECIP>(dBz_x, kdx)) + jy) + Psiy, denom);
        double cz = qt<RECIP>(f * ez + dt * ((qt<RECIP>(dBy_x, kdx) - qt<RECIP>(dBx_y, kdy)) + jz) + Psiz, denom);
        double E = sqrt(E2);
        double A = qt<RECIP>(chi, denom);
        double Cm = sqrt(cx * cx + cy * cy + cz * cz);
        // a non-finite input makes Cm NaN: the reference then stores E = 0 (its C > 0 test
        // fails) and the accumulators keep the NaN; reproduced, and reported
        if (flag && !isfinite(Cm)) *flag |= 2u;
        if (Cm > 0) {
            // the reference's stopping rule |E - Eold| <= 1e-9; the cap only guards a cell that
            // could never meet it (non-finite data, or fields far from O(1))
            double Eold;
            int it = 0;
            do {
                Eold = E;
                double Q = E * E;
                E = (2 * A * Q * E + Cm) / (3 * A * Q + 1);
            } while (fabs(E - Eold) > 1e-9 && ++it < ncap);
            if (flag && it >= ncap) *flag |= 1u;  // stopped by the cap, not by the rule
            if (RECIP) {
                const double sc = E / Cm;
                ex = sc * cx;
                ey = sc * cy;
                ez = sc * cz;
            } else {
                ex = E * cx / Cm;
                ey = E * cy / Cm;
                ez = E * cz / Cm;
            }
        } else {
            ex = 0.0;
            ey = 0.0;
            ez = 0.0;
        }
    } else {
        double exn = qt<RECIP>(numer * ex + (dt * ((qt<RECIP>(dBz_y, kdy) - qt<RECIP>(dBy_z, kdz)) + jx) + Psix), denom);
        double eyn = qt<RECIP>(numer * ey + (dt * ((qt<RECIP>(dBx_z, kdz) - qt<RECIP>(dBz_x, kdx)) + jy) + Psiy), denom);
        double ezn = qt<RECIP>(numer * ez + (dt * ((qt<RECIP>(dBy_x, kdx) - qt<RECIP>(dBx_y, kdy)) + jz) + Psiz), denom);
        ex = exn;
        ey = eyn;
        ez = ezn;
    }
}

// Denominator and numerator of the E update at cell c: the uniform ones, or those of a
// per-cell permittivity formed with the pole sums in the order the uniform ones are formed.
// sigma = Sigma dt / 2 of the plasma resistivity (src/fdtd_plrc.cpp:356-359).
template <bool NONLIN, typename A>
__device__ __forceinline__ void cell_eps(const A &a, size_t c, double sigma, double &denom, double &numer)
{
    if (a.epsf || a.plasma) {
        const double e = a.epsf ? gld(a.epsf + c) : a.eps;
        denom = NONLIN ? e + a.sumChi0 - a.sumXi0 + sigma : e + (a.sumChi0 - a.sumXi0) + sigma;
        numer = e - a.sumXi0 - sigma;
    } else {
        denom = a.denom;
        numer = a.numer;
    }
}

// PlasmaDensity::stepScheme at one cell (src/plasmadensity.cpp:40-53): rho <- (rho (1 + n I)
// + m I^K) / (1 - n I) with I = |E|^2; returns I^(K-1), which Sigma receives times w.
__device__ __forceinline__ double plasma_density_cell(double ex, double ey, double ez, double &rho, double n,
                                                      double m, int Km)
{
    const double I = ex * ex + ey * ey + ez * ez;
    double IKm = 1.0;
    for (int q = 0; q < Km; ++q) IKm *= I;  // ipow, src/util.h:67-73
    const double IK = I * IKm;
    rho = (rho * (1 + n * I) + m * IK) / (1 - n * I);
    return IKm;
}

// PlasmaCurrent::stepScheme at one cell (src/plasmacurrent.cpp:63-71)
__device__ __forceinline__ double plasma_current_comp(double j, double e, double rho_t, double gdtn, double gdtd,
                                                      double emdt)
{
    return (j * gdtn - emdt * e * rho_t) / gdtd;
}

template <int NP, bool NONLIN, bool RECIP>
__device__ __forceinline__ void plrc_e_update(double &ex, double &ey, double &ez, double dBz_y, double dBy_z,
                                              double dBx_z, double dBz_x, double dBy_x, double dBx_y,
                                              double kdx, double kdy, double kdz, double jx, double jy, double jz,
                                              double2 *const psi[3][3], size_t c, const PoleConsts &pc,
                                              double dt, double denom, double numer, double chi, int ncap,
                                              unsigned *flag)
{
    plrc_e_update_pp<NP, NONLIN, RECIP>(ex, ey, ez, dBz_y, dBy_z, dBx_z, dBz_x, dBy_x, dBx_y, kdx, kdy, kdz, jx, jy, jz, psi,
                                 psi, c, true, pc, dt, denom, numer, chi, ncap, flag);
}

// Device status of a solver (MPX_ERR_NUMERIC): bit 0 a Kerr Newton solve stopped at the
// iteration cap, bit 1 a non-finite value in an E update (its inputs or its result).  flag holds this lane's bits; one lane of the wave ORs
// the wave's bits into *status (a vector atomic), so a wave costs at most one atomic.
__device__ __forceinline__ unsigned finite_flag(double x, double y, double z)
{
    return (isfinite(x) && isfinite(y) && isfinite(z)) ? 0u : 2u;
}
__device__ __forceinline__ void report(unsigned *status, unsigned flag)
{
    const unsigned long long b1 = __ballot((flag & 1u) != 0), b2 = __ballot((flag & 2u) != 0);
    const unsigned long long any = b1 | b2;
    if (any && status && (int)__lane_id() == __ffsll((unsigned long long)any) - 1)
        atomicOr(status, (b1 ? 1u : 0u) | (b2 ? 2u : 0u));
}


// ------------------------------------------------------------------------------------
// fused path
// ------------------------------------------------------------------------------------

// accumulators of the active poles held in registers, indexable like the psi pointer table
// (psi[n][component][cell]) so that the shared E update reads them in place
template <int NP>
struct PsiRegs {
    double2 v[NP > 0 ? NP : 1][3];
    struct Comp {
        double2 x;
        __device__ double2 operator[](size_t) const { return x; }
    };
    struct Pole {
        const double2 *p;
        __device__ Comp operator[](int q) const { return Comp{p[q]}; }
    };
    __device__ Pole operator[](int n) const { return Pole{v[n]}; }
};


// ---- CPML by dimension (CpmlDim) ----
//
// The face map is x: (psi0 -> Jy from dBz, psi1 -> Jz from dBy), y: (psi0 -> Jz from dBx, psi1 -> Jx
// from dBz), z: (psi0 -> Jx from dBy, psi1 -> Jy from dBx) (src/cpml_border.cpp:357-386, 456-485).
//
// A cell's auxiliaries are requested with its field words and used after them, those of all
// three dimensions together: taken face by face, each with its descriptor, coefficients and
// auxiliaries loaded on the spot, a layer cell paid up to three memory latencies in a row, and
// a wave with any layer cell paid them whole.

// An opaque use of a loaded value: conversions of it stay behind this point instead of moving up
// to its load, where they would wait for memory.
template <typename T>
__device__ __forceinline__ void hold(T &v)
{
    asm volatile("" : "+v"(v));
}

// the side of the layer that holds coordinate x (0 high, 1 low), -1 outside
__device__ __forceinline__ int cpml_side(const CpmlDim &D, int x)
{
    return x >= D.lo[0] && x <= D.hi[0] ? 0 : (x >= D.lo[1] && x <= D.hi[1] ? 1 : -1);
}
// the two auxiliaries of a cell as stored
template <typename T, bool RES>
struct Aux {
    T o0, o1;
    unsigned w;
};
template <typename T, bool RES>
__device__ __forceinline__ Aux<T, RES> cpml_load(const CpmlDim &D, unsigned l)
{
    // ordinary loads: a face row covers only part of a cache line (z faces: 16 cells), and the
    // rest of the line is read by the neighbouring row
    return {gld((const T *)D.o0 + l), gld((const T *)D.o1 + l), lo_ld<RES>(D.orw, l)};
}
// The new auxiliaries (h0, h1, w: as stored) from the old (x), the coefficients and the cell's
// differences.  v0, v1: the stored values, which the current sums see.
// E side: CPMLBorderECurrent::stepScheme, src/cpml_border.cpp:398-425 (psi0 gets -c d1/dx);
// H side: CPMLBorderHCurrent::stepScheme, src/cpml_border.cpp:499-527 (psi0 gets +c d1/dx).
template <typename T, bool HSIDE, bool RES>
__device__ __forceinline__ void cpml_next(double idxn, double bq, double cq, const Aux<T, RES> &x, double d1, double d0,
                                          T &h0, T &h1, unsigned &w, double &v0, double &v1)
{
    T r0 = x.o0, r1 = x.o1;
    hold(r0);  // decoded here, not where they were requested
    hold(r1);
    const double a0 = got<T, RES>(r0, x.w, 0), a1 = got<T, RES>(r1, x.w, 1);
    double n0, n1;
    if (HSIDE) {
        n0 = bq * a0 + cq * d1 * idxn;
        n1 = bq * a1 - cq * d0 * idxn;
    } else {
        n0 = bq * a0 - cq * d1 * idxn;
        n1 = bq * a1 + cq * d0 * idxn;
    }
    w = 0;
    h0 = put<T, RES>(n0, w, 0);
    h1 = put<T, RES>(n1, w, 1);
    v0 = got<T, RES>(h0, w, 0);
    v1 = got<T, RES>(h1, w, 1);
}
// the same, the new auxiliaries stored at index l with `store`
template <typename T, bool HSIDE, bool RES>
__device__ __forceinline__ void cpml_update(const CpmlDim &D, double bq, double cq, unsigned l, const Aux<T, RES> &x, double d1,
                                            double d0, bool store, double &v0, double &v1)
{
    T h0, h1;
    unsigned w;
    cpml_next<T, HSIDE, RES>(D.idxn, bq, cq, x, d1, d0, h0, h1, w, v0, v1);
    if (store) {
        gst((T *)D.p0 + l, h0);
        gst((T *)D.p1 + l, h1);
        if (RES) gst(D.rw + l, w);
    }
}
// A cell's part in the layers of the three dimensions: its sides and what was loaded for them
template <typename T, bool RES>
struct CellCpml {
    int side[3];
    Aux<T, RES> x[3];
};
template <typename T, bool RES>
__device__ __forceinline__ void cpml_request(const CpmlDim D[3], int i, int j, int k, bool live, CellCpml<T, RES> &s)
{
    const int at[3] = {i, j, k};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        s.side[d] = live ? cpml_side(D[d], at[d]) : -1;
        // a wave with no cell in these layers skips them; in the others every lane loads, so that no
        // value is merged and waited for here (lanes outside take the block's first element)
        if (__ballot(s.side[d] >= 0))
            s.x[d] = cpml_load<T, RES>(D[d], s.side[d] >= 0 ? cpml_index(D[d], s.side[d], i, j, k) : 0u);
    }
}
// The current totals gain the auxiliaries of a cell of dimension d's layers (D, coordinate `at`); x: those
// of the layer on `side`.  d0, d1: the differences that feed psi0 and psi1; Jp, Jq: the currents these feed.
template <typename T, bool HSIDE, bool RES>
__device__ __forceinline__ void cpml_dim_add(const CpmlDim &D, int at, int side, int i, int j, int k, const Aux<T, RES> &x,
                                             double d1, double d0, bool store, double &Jp, double &Jq)
{
    double v0, v1;
    const double *line = D.bc + (2 * side * D.len + at);
    cpml_update<T, HSIDE, RES>(D, gld(line), gld(line + D.len), cpml_index(D, side, i, j, k), x, d1, d0, store, v0, v1);
    Jp += v0;
    Jq += v1;
    if (D.two && side == 0 && at >= D.lo[1] && at <= D.hi[1]) {
        const unsigned l = cpml_index(D, 1, i, j, k);
        line = D.bc + (2 * D.len + at);
        cpml_update<T, HSIDE, RES>(D, gld(line), gld(line + D.len), l, cpml_load<T, RES>(D, l), d1, d0, store, v0, v1);
        Jp += v0;
        Jq += v1;
    }
}
// The current totals gain the cell's auxiliaries in the reference's list order: faces N,S (y),
// E,W (x), U,D (z), the high face first.  df[d][0], df[d][1]: the differences along d of the field
// components d + 1 and d + 2, which feed psi1 and psi0; those feed the currents d + 2 and d + 1.
template <typename T, bool HSIDE, bool RES>
__device__ __forceinline__ void cpml_add(const CpmlDim D[3], int i, int j, int k, const CellCpml<T, RES> &s,
                                         const double df[3][2], bool store, double J[3])
{
    const int at[3] = {i, j, k};
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        constexpr int order[3] = {1, 0, 2};
        const int d = order[u];
        if (s.side[d] >= 0)
            cpml_dim_add<T, HSIDE, RES>(D[d], at[d], s.side[d], i, j, k, s.x[d], df[d][1], df[d][0], store, J[(d + 1) % 3],
                                        J[(d + 2) % 3]);
    }
}
// the same, each dimension's auxiliaries loaded where they are used
template <typename T, bool HSIDE, bool RES>
__device__ __forceinline__ void cpml_each(const CpmlDim D[3], int i, int j, int k, const double df[3][2], double J[3])
{
    const int at[3] = {i, j, k};
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        constexpr int order[3] = {1, 0, 2};
        const int d = order[u], side = cpml_side(D[d], at[d]);
        if (side >= 0)
            cpml_dim_add<T, HSIDE, RES>(D[d], at[d], side, i, j, k, cpml_load<T, RES>(D[d], cpml_index(D[d], side, i, j, k)),
                                        df[d][1], df[d][0], true, J[(d + 1) % 3], J[(d + 2) % 3]);
    }
}

// 32-bit layer index of cell (i, j, k) in a face box
__device__ __forceinline__ int layer_index(const CpmlFace &f, int i, int j, int k)
{
    return ((i - f.lo[0]) * f.n1 + (j - f.lo[1])) * f.n2 + (k - f.lo[2]);
}

// add the current-sheet layers that contain cell (i, j, k), in list order, from the slot at
// element offset soff of their planes
template <typename T>
__device__ __forceinline__ void add_sheets(const StepArgs<T> &a, int i, int j, int k, int soff, double &x, double &y,
                                           double &z)
{
    for (int s = 0; s < a.nsheets; ++s)
        if (k == a.sheet[s].kp) {
            int q = i * a.g.py + j + soff;
            x += gld(a.sheet[s].J[0] + q);
            y += gld(a.sheet[s].J[1] + q);
            z += gld(a.sheet[s].J[2] + q);
        }
}

// Map the linear block id to a tile so that each XCD (blocks are dealt round-robin over
// the 8 XCDs) walks a contiguous slab of x planes and keeps the x-neighbour planes in its L2.
__device__ __forceinline__ void xcd_tile(int nbx, int nby, int nbz, int &bx, int &by, int &bz)
{
    unsigned lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    unsigned total = (unsigned)nbx * nby * nbz;
    unsigned per = total / 8u;
    unsigned xcd = lin & 7u, idx = lin >> 3;
    unsigned t = (lin < per * 8u) ? xcd * per + idx : lin;
    bx = t % nbx;
    t /= nbx;
    by = t % nby;
    bz = t / nby;
}

// Banded order: the tile rows are cut into bands of R rows; inside a band the z tiles run
// fastest, then the rows of the band, then the x chunks, so the x-neighbour plane of a tile
// was read a band-plane (nbx * R tiles) earlier and is still in the XCD's L2.  Each XCD
// takes a contiguous share of the order as in xcd_tile.  With rev the order runs from its end,
// which the B-side kernel uses to begin on the tiles the E-side kernel finished last.
__device__ __forceinline__ void band_tile(int nbx, int nby, int nbz, int R, int rev, int &bx, int &by, int &bz)
{
    unsigned lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    unsigned total = (unsigned)nbx * nby * nbz;
    unsigned per = total / 8u;
    unsigned xcd = lin & 7u, idx = lin >> 3;
    unsigned t = (lin < per * 8u) ? xcd * per + idx : lin;
    if (rev) t = total - 1u - t;
    const unsigned full = (unsigned)nbx * R * nbz;  // tiles of a full band; only the last is shorter
    const unsigned b = t / full;
    unsigned rem = t - b * full;
    const unsigned rows = min((unsigned)R, (unsigned)nby - b * R);
    bx = rem % nbx;
    rem /= nbx;
    by = b * R + rem % rows;
    bz = rem / rows;
}

// Block -> tile of the fused kernels from a map made on the host (mpx_types.h): the orders above
// with multiplications in place of the divisions, which took some 150 instructions and several
// dependent argument loads at the head of every wave.
__device__ __forceinline__ unsigned fast_div(unsigned t, const FastDiv &f)
{
    return (unsigned)(((unsigned long long)t * f.m) >> f.sh);
}
__device__ __forceinline__ bool map_tile(const TileMap &M, int &bx, int &by, int &bz)
{
    const unsigned x = blockIdx.x & 7u;
    unsigned t = M.at[x] + (blockIdx.x >> 3);
    if (t >= M.at[x + 1]) return false;
    if (M.order == 2) {
        if (M.rev) t = M.total - 1u - t;
        const unsigned b = fast_div(t, M.full);
        unsigned rem = t - b * M.full.d;
        const bool last = (int)b == M.nbands - 1;
        const unsigned q = fast_div(rem, M.first);
        bx = rem - q * M.first.d;
        const unsigned rows = last ? M.rlast.d : M.rband.d;
        const unsigned z = last ? fast_div(q, M.rlast) : fast_div(q, M.rband);
        by = b * M.rband.d + (q - z * rows);
        bz = z;
    } else {
        const unsigned q = fast_div(t, M.first), z = fast_div(q, M.second);
        const int u = t - q * M.first.d, v = q - z * M.second.d;
        if (M.order == 1) {
            bz = u;
            bx = v;
            by = z;
        } else {
            bx = u;
            by = v;
            bz = z;
        }
    }
    return true;
}

// (j, k) of this thread in a tile of the fused kernels: 64 z cells x 4 y rows, or (LIN) 256 consecutive cells of
// the y-z plane taken row after row, which keeps every lane busy on grids whose z extent is
// not a multiple of 64.  lo = first index of the range in y and z.
template <bool LIN>
__device__ __forceinline__ void tile_jk(const GridDims &g, const int lo[3], int tbx, int tby, int &j, int &k)
{
    if (LIN) {
        const int nk = g.n[2] - lo[2] + 1;
        const int lin = tbx * 256 + threadIdx.y * 64 + threadIdx.x;
        const int q = lin / nk;
        j = q + lo[1];
        k = lin - q * nk + lo[2];
    } else {
        k = tbx * 64 + threadIdx.x + lo[2];
        j = tby * 4 + threadIdx.y + lo[1];
    }
}

// add the current-sheet layers of list `sh` that contain cell (i, j, k), in list order
__device__ __forceinline__ void add_sheet_planes(const Sheet *sh, int n, int py, int i, int j, int k, int soff,
                                                 double &x, double &y, double &z)
{
    for (int s = 0; s < n; ++s)
        if (k == sh[s].kp) {
            int q = i * py + j + soff;
            x += gld(sh[s].J[0] + q);
            y += gld(sh[s].J[1] + q);
            z += gld(sh[s].J[2] + q);
        }
}

// Walk this block's share of a batch's tile list: the tiles are numbered run by run (z tile
// fastest, then y, then x), the 8 XCDs take contiguous eighths of the list so that tiles
// sharing halo cells meet in one L2, and each block strides its XCD's eighth by
// gridDim.x / 8 (gridDim.x is a multiple of 8; the hardware deals blocks to the XCDs round
// robin).  Each XCD starts its eighth at a different point (XCD x at x/8 of it, wrapping
// round), so that the XCDs do not walk equal runs at equal offsets in lock step; that
// measured 2-5 % faster on batches of equal-size runs.  f(run, tz, ty, tx) processes one tile.
template <typename F>
__device__ __forceinline__ void batch_tiles(const BatchRun *__restrict__ runs, int nruns, int total, F &&f)
{
    const int per_xcd = gridDim.x >> 3;
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int chunk = (total + 7) >> 3;
    const int t0 = xcd * chunk, t1 = min(total, t0 + chunk);
    const int len = max(0, t1 - t0);
    const int rot = (int)(((long long)len * xcd) >> 3);
    int r = 0;
    for (int u = slot; u < len; u += per_xcd) {
        int v = u + rot;
        if (v >= len) v -= len;
        const int t = t0 + v;
        if (t < runs[r].first) r = 0;  // wrapped round to the start of the eighth
        while (r + 1 < nruns && t >= runs[r + 1].first) ++r;
        const int ntz = runs[r].ntz, nty = runs[r].nty;
        int local = t - runs[r].first;
        const int tz = local % ntz;
        local /= ntz;
        f(r, tz, local % nty, local / nty);
    }
}

}  // namespace mpx
