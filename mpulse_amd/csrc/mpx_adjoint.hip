// Discrete adjoint of one time step of the fused float64 PLRC update (the forward kernels are
// fused_E_tile / fused_B_tile in mpx_fused.hip; the reference update is
// FDTD_PLRCNonlinCore::plrcStepD, src/fdtd_plrc.cpp:304-427, with the pole recursion of
// src/fdtd_plrc.cpp:321-353, plrcStepB, src/fdtd_plrc.cpp:429-459, and the CPML auxiliaries
// of src/cpml_border.cpp:398-425, 499-527).  Periodic boundary in every dimension: E and B
// cells are 1..N, neighbours wrap.
//
// Forward step n (per cell; D_F[d][q] = difference along d of component q of field F):
//   E kernel: psiE' = b psiE -/+ c D_B / delta (face layers), J = sheets + psiE',
//             R = curl_kappa(D_B) + J, poles p: P_p = Dd_p E + Psi_p (complex, Dd = dchi0 -
//             dxi0), Psi_p' = dxi0_p E + Crec_p P_p,
//             C = ((numer + chi |E|^2) E + dt R + sum_p Re P_p) / denom with
//             denom = eps + sumChi0 - sumXi0 and numer = eps - sumXi0,
//             E' = (e / s) C with s = |C| and (chi / denom) e^3 + e = s (the linear solver:
//             chi = 0, E' = C);
//   B kernel: psiH' = b psiH +/- c D_E' / delta, B' = B + dt (curl_kappa(D_E') + M),
//             M = sheets + psiH'.
//
// The reverse of step n runs two kernels.  k_adj_e gathers the adjoint of E' from the adjoint
// of B', adds the objective, and takes the Newton solve, eps, chi and the pole recursion
// back; what it hands on is the adjoint of R, rb = dt Cb / denom (Cb the adjoint of C).
// k_adj_b adds the adjoints of the E kernel's B differences, from rb, to the adjoint of B.
//
// Memory bound: 30 words a cell and step (+12 a pole).  The adjoint of a difference is the
// adjoint of one component times a line factor, so both gathers form the differences of a cell
// and of its neighbour from that component instead of reading six stored differences: three
// kernels with the differences of both sides stored moved 50 words and took 376 us a step at
// 128x128x256, these two 271 (171 + 100).  A CPML auxiliary enters its difference as A c / delta with
// A = b A + (the adjoint of its current): A is what is stored, updated in place by the kernel
// that has just computed that adjoint and read, at a cell and its neighbour, by the next, so
// it needs no second copy.  dJ/dchi is summed per wave, not kept per cell.
//
// A complex accumulator's adjoint is held as (dL/dRe, dL/dIm); through w = K z it goes back as
// conj(K) lw, and a real input x of w = G x receives Re(conj(G) lw).
#include <hip/hip_runtime.h>

#include "mpx_device.h"
#include "mpx_launch.h"

namespace mpx {

namespace {

// periodic neighbour index along one dimension
__device__ __forceinline__ int wrapm(int v, int n) { return v == 1 ? n : v - 1; }
__device__ __forceinline__ int wrapp(int v, int n) { return v == n ? 1 : v + 1; }

// The adjoints of the two differences along d of a cell (x = coordinate along d): of component
// c1 = d + 2 from the adjoint l0 of the curl's component c0 = d + 1 (u1), and of component c0
// from l1 (u0), as the B kernel (sign +1) or the E kernel (sign -1) has them, its CPML faces
// included.
__device__ __forceinline__ void diff_pair(const AdjFace f[2], const double *ik, int i, int j, int k, int x, double sign,
                                          double l0, double l1, double &u0, double &u1)
{
    const double r = sign * gld(ik + x);
    u1 = l0 * r;
    u0 = -(l1 * r);
#pragma unroll
    for (int s = 0; s < 2; ++s)
        if (x >= f[s].lo && x <= f[s].hi) {
            const int l = i * f[s].s0 + j * f[s].s1 + k - f[s].off;
            const double cq = sign * (gld(f[s].c + (x - f[s].lo)) * f[s].idxn);
            u1 += gld(f[s].A0 + l) * cq;
            u0 -= gld(f[s].A1 + l) * cq;
        }
}

// A = b A + l of the faces along d that hold the cell
__device__ __forceinline__ void carry(const AdjFace f[2], int i, int j, int k, int x, double l0, double l1)
{
#pragma unroll
    for (int s = 0; s < 2; ++s)
        if (x >= f[s].lo && x <= f[s].hi) {
            const int l = i * f[s].s0 + j * f[s].s1 + k - f[s].off;
            const double b = gld(f[s].b + (x - f[s].lo));
            const double a0 = gld(f[s].A0 + l), a1 = gld(f[s].A1 + l);
            gst(f[s].A0 + l, b * a0 + l0);
            gst(f[s].A1 + l, b * a1 + l1);
        }
}

}  // namespace

// Adjoint of the E kernel at E cell (i, j, k).
template <int NP>
__global__ __launch_bounds__(256) void k_adj_e(AdjArgs a, AdjHistory h, int nbx, int nby, int nbz)
{
    int bx, by, bz;
    band_tile(nbx, nby, nbz, a.band, 0, bx, by, bz);
    const GridDims &g = a.g;
    const int k = bx * 64 + threadIdx.x + 1, j = by * 4 + threadIdx.y + 1, i = bz + 1;
    double chi_part = 0.0;
    if (k <= g.n[2] && j <= g.n[1]) {
        const int c = (int)g.at(i, j, k);
        const int im = wrapm(i, g.n[0]), jm = wrapm(j, g.n[1]), km = wrapm(k, g.n[2]);
        const int cx = c + (im - i) * (int)g.sx, cy = c + (jm - j) * g.pz, cz = c + (km - k);
        const double lb[3] = {gld(a.lB[0] + c), gld(a.lB[1] + c), gld(a.lB[2] + c)};
        const double bxy = gld(a.lB[1] + cx), bxz = gld(a.lB[2] + cx), byz = gld(a.lB[2] + cy);
        const double byx = gld(a.lB[0] + cy), bzx = gld(a.lB[0] + cz), bzy = gld(a.lB[1] + cz);
        double le[3] = {load_once(a.lE[0] + c), load_once(a.lE[1] + c), load_once(a.lE[2] + c)};
        const double e0[3] = {gld(h.E0[0] + c), gld(h.E0[1] + c), gld(h.E0[2] + c)};
        const double e1[3] = {gld(h.E1[0] + c), gld(h.E1[1] + c), gld(h.E1[2] + c)};
        const double eps = a.epsf ? gld(a.epsf + c) : a.eps;
        const double eb = load_once(a.epsb + c);
        double2 lp[NP > 0 ? NP : 1][3];
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int q = 0; q < 3; ++q) lp[p][q] = load_once(a.lpsi[p][q] + c);
        // adjoint of E' at c: its own plus, of the differences D_E'[d][q] = E'_q(c + e_d) - E'_q(c),
        // those of the cell and of the one before it
        const double dt = a.dt;
        double u0, u1, v0, v1;
        diff_pair(a.hf[0], a.ikdH[0], i, j, k, i, 1.0, dt * lb[1], dt * lb[2], u0, u1);
        diff_pair(a.hf[0], a.ikdH[0], im, j, k, im, 1.0, dt * bxy, dt * bxz, v0, v1);
        le[1] += v0 - u0;
        le[2] += v1 - u1;
        diff_pair(a.hf[1], a.ikdH[1], i, j, k, j, 1.0, dt * lb[2], dt * lb[0], u0, u1);
        diff_pair(a.hf[1], a.ikdH[1], i, jm, k, jm, 1.0, dt * byz, dt * byx, v0, v1);
        le[2] += v0 - u0;
        le[0] += v1 - u1;
        diff_pair(a.hf[2], a.ikdH[2], i, j, k, k, 1.0, dt * lb[0], dt * lb[1], u0, u1);
        diff_pair(a.hf[2], a.ikdH[2], i, j, km, km, 1.0, dt * bzx, dt * bzy, v0, v1);
        le[0] += v0 - u0;
        le[1] += v1 - u1;
        if (k == a.kobj)
            for (int q = 0; q < 3; ++q) le[q] += 2.0 * a.wobj * e1[q];
        double S = 0.0;  // sum_p Re Dd_p: the part of sum_p Re P_p proportional to E
#pragma unroll
        for (int p = 0; p < NP; ++p) S += a.pc.dd[p].x;
        const double idenom = 1.0 / (eps + a.sumChi0 - a.sumXi0);
        const double numer = eps - a.sumXi0;
        const double A = a.chi * idenom;
        // the Kerr solve E' = (e / s) C with s = A e^3 + e: C = E' / phi, phi = e / s = 1 / (1 + A e^2),
        // and with Q = e^2: dE'/dC along C is 1 / (3 A Q + 1), across it phi; d E' / d A along C is
        // -e^3 / (3 A Q + 1) (at e = 0 all of it is the identity)
        const double Q = e1[0] * e1[0] + e1[1] * e1[1] + e1[2] * e1[2];
        const double iphi = 1.0 + A * Q, phi = 1.0 / iphi, des = 1.0 / (3.0 * A * Q + 1.0);
        const double el = e1[0] * le[0] + e1[1] * le[1] + e1[2] * le[2];
        const double w = -2.0 * A * des * phi * el;  // (des - phi) el / Q
        double cb[3], cv[3];
        for (int q = 0; q < 3; ++q) {
            cb[q] = phi * le[q] + w * e1[q];
            cv[q] = e1[q] * iphi;
        }
        const double Ab = -Q * des * el;
        // C denom = (numer + S + chi |E|^2) E + dt R + sum_p Re Psi_p; denom and numer both
        // grow by d eps, so dC/deps = (E - C) / denom
        const double E2 = e0[0] * e0[0] + e0[1] * e0[1] + e0[2] * e0[2];
        const double Ecb = e0[0] * cb[0] + e0[1] * cb[1] + e0[2] * cb[2];
        const double f = numer + S + a.chi * E2;
        double lnew[3], rb[3];
        for (int q = 0; q < 3; ++q) {
            lnew[q] = (f * cb[q] + 2.0 * a.chi * e0[q] * Ecb) * idenom;
            rb[q] = dt * cb[q] * idenom;
        }
        // poles: Psi_p' = G_p E + Crec_p Psi_p with G_p = dxi0_p + Crec_p Dd_p, and C reads Re Psi_p
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const double2 K = a.pc.crec[p], X = a.pc.dxi0[p], Dd = a.pc.dd[p];
            const double Gr = X.x + (K.x * Dd.x - K.y * Dd.y), Gi = X.y + (K.x * Dd.y + K.y * Dd.x);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const double2 l = lp[p][q];
                lnew[q] += Gr * l.x + Gi * l.y;
                store_once(a.lpsi[p][q] + c, make_double2(K.x * l.x + K.y * l.y + cb[q] * idenom, K.x * l.y - K.y * l.x));
            }
        }
        double ecb = 0.0;
        for (int q = 0; q < 3; ++q) ecb += (e0[q] - cv[q]) * cb[q];
        store_once(a.epsb + c, eb - Ab * a.chi * idenom * idenom + ecb * idenom);
        chi_part = Ab * idenom + E2 * Ecb * idenom;
        for (int q = 0; q < 3; ++q) {
            store_once(a.lE[q] + c, lnew[q]);
            gst(a.rb[q] + c, rb[q]);
        }
        carry(a.ef[0], i, j, k, i, rb[1], rb[2]);
        carry(a.ef[1], i, j, k, j, rb[2], rb[0]);
        carry(a.ef[2], i, j, k, k, rb[0], rb[1]);
    }
    // dJ/dchi: this wave's cells, in a fixed order, into the wave's own slot
    for (int m = 32; m > 0; m >>= 1) chi_part += __shfl_xor(chi_part, m);
    if (threadIdx.x == 0) a.chiw[((bz * nby + by) * nbx + bx) * 4 + threadIdx.y] += chi_part;
}

// Adjoint of B at cell (i, j, k): the E kernel's differences D_B[d][q] = B_q(c) - B_q(c - e_d)
// give B_q(c) those of the cell and, negative, those of the cell after it.
__global__ __launch_bounds__(256) void k_adj_b(AdjArgs a, int nbx, int nby, int nbz)
{
    int bx, by, bz;
    band_tile(nbx, nby, nbz, a.band, 1, bx, by, bz);  // backwards: on the cells k_adj_e left last
    const GridDims &g = a.g;
    const int k = bx * 64 + threadIdx.x + 1, j = by * 4 + threadIdx.y + 1, i = bz + 1;
    if (k > g.n[2] || j > g.n[1]) return;
    const int c = (int)g.at(i, j, k);
    const int ip = wrapp(i, g.n[0]), jp = wrapp(j, g.n[1]), kp = wrapp(k, g.n[2]);
    const int cx = c + (ip - i) * (int)g.sx, cy = c + (jp - j) * g.pz, cz = c + (kp - k);
    const double r[3] = {gld(a.rb[0] + c), gld(a.rb[1] + c), gld(a.rb[2] + c)};
    const double rxy = gld(a.rb[1] + cx), rxz = gld(a.rb[2] + cx), ryz = gld(a.rb[2] + cy);
    const double ryx = gld(a.rb[0] + cy), rzx = gld(a.rb[0] + cz), rzy = gld(a.rb[1] + cz);
    double lb[3] = {gld(a.lB[0] + c), gld(a.lB[1] + c), gld(a.lB[2] + c)};
    double u0, u1, v0, v1;
    diff_pair(a.ef[0], a.ikdE[0], i, j, k, i, -1.0, r[1], r[2], u0, u1);
    diff_pair(a.ef[0], a.ikdE[0], ip, j, k, ip, -1.0, rxy, rxz, v0, v1);
    lb[1] += u0 - v0;
    lb[2] += u1 - v1;
    diff_pair(a.ef[1], a.ikdE[1], i, j, k, j, -1.0, r[2], r[0], u0, u1);
    diff_pair(a.ef[1], a.ikdE[1], i, jp, k, jp, -1.0, ryz, ryx, v0, v1);
    lb[2] += u0 - v0;
    lb[0] += u1 - v1;
    diff_pair(a.ef[2], a.ikdE[2], i, j, k, k, -1.0, r[0], r[1], u0, u1);
    diff_pair(a.ef[2], a.ikdE[2], i, j, kp, kp, -1.0, rzx, rzy, v0, v1);
    lb[0] += u0 - v0;
    lb[1] += u1 - v1;
    for (int q = 0; q < 3; ++q) gst(a.lB[q] + c, lb[q]);
    const double dt = a.dt;
    carry(a.hf[0], i, j, k, i, dt * lb[1], dt * lb[2]);
    carry(a.hf[1], i, j, k, j, dt * lb[2], dt * lb[0]);
    carry(a.hf[2], i, j, k, k, dt * lb[0], dt * lb[1]);
}

// sum_{i,j} |E(i, j, kobj)|^2 over the interior of the plane, one partial sum a block (summed
// over blocks and steps at the end, in a fixed order).  One block of 1024 threads for the whole
// plane spent 75 us a step on 16 rounds of one word from each of 16384 rows (128x128x256).
__global__ __launch_bounds__(256) void k_plane_objective(GridDims g, const double *Ex, const double *Ey,
                                                         const double *Ez, int kobj, double *part)
{
    __shared__ double red[256];
    double v = 0.0;
    const int n = g.n[0] * g.n[1];
    for (int t = blockIdx.x * 256 + threadIdx.x; t < n; t += gridDim.x * 256) {
        const int i = t / g.n[1] + 1, j = t % g.n[1] + 1;
        const size_t c = g.at(i, j, kobj);
        v += Ex[c] * Ex[c] + Ey[c] * Ey[c] + Ez[c] * Ez[c];
    }
    red[threadIdx.x] = v;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

static void adj_tiles(const GridDims &g, int &nbx, int &nby, int &nbz)
{
    nbx = (g.n[2] + 63) / 64;
    nby = (g.n[1] + 3) / 4;
    nbz = g.n[0];
}

size_t adjoint_waves(const GridDims &g)
{
    int nbx, nby, nbz;
    adj_tiles(g, nbx, nby, nbz);
    return (size_t)nbx * nby * nbz * 4;
}

void launch_adjoint_step(const AdjArgs &a, const AdjHistory &h, hipStream_t s)
{
    int nbx, nby, nbz;
    adj_tiles(a.g, nbx, nby, nbz);
    const dim3 grd(nbx, nby, nbz), blk(64, 4);
    switch (a.np) {
    case 0: hipLaunchKernelGGL(k_adj_e<0>, grd, blk, 0, s, a, h, nbx, nby, nbz); break;
    case 1: hipLaunchKernelGGL(k_adj_e<1>, grd, blk, 0, s, a, h, nbx, nby, nbz); break;
    case 2: hipLaunchKernelGGL(k_adj_e<2>, grd, blk, 0, s, a, h, nbx, nby, nbz); break;
    default: hipLaunchKernelGGL(k_adj_e<3>, grd, blk, 0, s, a, h, nbx, nby, nbz); break;
    }
    hipLaunchKernelGGL(k_adj_b, grd, blk, 0, s, a, nbx, nby, nbz);
}

// blocks of the objective: one per 256 cells of the plane, at most 256 (the rest in rounds)
int objective_blocks(const GridDims &g)
{
    const long long n = ((long long)g.n[0] * g.n[1] + 255) / 256;
    return (int)(n < 256 ? n : 256);
}

void launch_plane_objective(const GridDims &g, const double *const E[3], int kobj, double *part, hipStream_t s)
{
    hipLaunchKernelGGL(k_plane_objective, dim3(objective_blocks(g)), dim3(256), 0, s, g, E[0], E[1], E[2], kobj, part);
}

}  // namespace mpx
