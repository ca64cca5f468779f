// gfx950 kernels of the source sheets: IncidentSource{E,H}Current::stepScheme,
// src/incsource.t:40-73, 112-145.
//
// A sheet is two float64 component planes of (nx + 2) x (ny + 2) cells that depend on the step
// and on the transverse position only, never on the fields.
//
// What bounds it: the closed-form short pulse is one serial chain of float64 operations per
// cell (two Faddeeva functions, complex quotients, exponentials): 10 us for the 26^2 cells of
// a 24^3 grid as for 66^2 cells, and 0.035 ms per sheet at 514^2 (two waves per SIMD).  With
// one launch per sheet and step, one thread per cell and both B components in one thread the
// two sheets took 21 of the 46 us of a 64^3 step.  Hence:
//   * one launch holds both sides and every step that the call in progress still has to take,
//     up to the slots the solver keeps (sheet_slots), so a call pays the chain's latency once;
//   * the components of a step (B_x and B_y of the E sheet, E_x of the H sheet) are blocks of
//     their own (sheet_tasks) instead of one thread's sequence;
//   * the pulse depends on x^2 and y^2 (B_x: odd in both) and the cells lie mirrored about the
//     axis, so a quarter of the cells is evaluated and stored at its mirror images too, with
//     the very bits the mirror cell would compute.
// Measured with the rest unchanged: 64^3 float64, 100 steps a call and the fields read, 4.99 ->
// 2.98 ms; 24^3, one step a call, 597 -> 487 us; 256^3 float32 + residual 106.2 -> 103.9 ms
// per 100 steps, 512^3 560 -> 555 ms per 96.
#include <hip/hip_runtime.h>

#include "mpx_launch.h"
#include "mpx_memory.h"

namespace mpx {

__device__ inline void plane_getH(const PlaneParams &W, int i, int j, int l, int time, double out[3])
{
    // PlaneWaveSourceEFunc::getHField src/sources.cpp:107-125 / PlaneGaussSourceEFunc src/sources.cpp:266-284
    double realtime = W.dt * (time - 0.5);
    double posx = W.k[0] * i * W.dx + W.k[1] * (j + 0.5) * W.dy + W.k[2] * (l + 0.5) * W.dz + W.om * realtime;
    double posy = W.k[0] * (i + 0.5) * W.dx + W.k[1] * j * W.dy + W.k[2] * (l + 0.5) * W.dz + W.om * realtime;
    double posz = W.k[0] * (i + 0.5) * W.dx + W.k[1] * (j + 0.5) * W.dy + W.k[2] * l * W.dz + W.om * realtime;
    double pos[3] = {posx, posy, posz};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (!W.gauss) {
            double h = W.H[d] * sin(pos[d]) + W.H_bg[d];
            if (pos[d] < W.ramp) h *= pos[d] / W.ramp;
            out[d] = h;
        } else {
            double q = (pos[d] - W.offset) / W.width;
            out[d] = (W.H[d] * exp(-(q * q))) * sin(pos[d]);
        }
    }
}

__device__ inline void plane_getE(const PlaneParams &W, int i, int j, int l, int time, double out[3])
{
    // PlaneWaveSourceHFunc::getEField src/sources.cpp:150-173 / PlaneGaussSourceHFunc src/sources.cpp:308-331
    double realtime = W.dt * time;
    double posx = W.k[0] * (i + 0.5) * W.dx + W.k[1] * j * W.dy + W.k[2] * l * W.dz + W.om * realtime;
    double posy = W.k[0] * i * W.dx + W.k[1] * (j + 0.5) * W.dy + W.k[2] * l * W.dz + W.om * realtime;
    double posz = W.k[0] * i * W.dx + W.k[1] * j * W.dy + W.k[2] * (l + 0.5) * W.dz + W.om * realtime;
    double pos[3] = {posx, posy, posz};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (!W.gauss) {
            double e = W.E[d] * sin(pos[d]) + W.E_bg[d];
            if (pos[d] < W.ramp) e *= pos[d] / W.ramp;
            out[d] = e;
        } else {
            double q = (pos[d] - W.offset) / W.width;
            out[d] = (W.E[d] * exp(-(q * q))) * sin(pos[d]);
        }
    }
}

// Points of one transverse line of a short-pulse component that are evaluated: samples at
// integer positions (half false) mirror i <-> n + 1 - i, samples half a cell further out mirror
// i <-> n - i, the last one (i = n + 1) standing alone.
__host__ __device__ __forceinline__ int mirror_points(int n, bool half) { return half ? n / 2 + 2 : (n + 1) / 2 + 1; }
// cell of point p and its mirror image (the same cell where there is none)
__device__ __forceinline__ void mirror_cells(int n, bool half, int p, int &i, int &im)
{
    if (half) {
        i = p == n / 2 + 1 ? n + 1 : p;
        im = i == n + 1 ? i : n - i;
    } else {
        i = p;
        im = n + 1 - i;
    }
}
// whether component `task` of a short-pulse sheet samples x / y half a cell further out
// (task 0 of the E sheet: B_x at (i, j + 1/2); 1: B_y at (i + 1/2, j); H sheet: E_x at (i + 1/2, j))
__host__ __device__ __forceinline__ bool pulse_half_x(bool isH, int task) { return isH || task == 1; }
__host__ __device__ __forceinline__ bool pulse_half_y(bool isH, int task) { return !isH && task == 0; }

// separately evaluated components of a sheet, and the points of one
__host__ __device__ __forceinline__ int tasks_of(int kind, bool isH) { return kind == 1 && !isH ? 2 : 1; }
__host__ __device__ __forceinline__ int points_of(int kind, bool isH, int task, int nx2, int ny2)
{
    if (kind != 1) return nx2 * ny2;
    return mirror_points(nx2 - 2, pulse_half_x(isH, task)) * mirror_points(ny2 - 2, pulse_half_y(isH, task));
}

// point p of component `task` of one sheet at step `time`, into the slot at element offset so
// of its planes; KIND > 0 fixes the source kind at compile time (each kind then gets only the
// registers it needs), KIND = 0 reads it from the descriptor
template <int KIND>
__device__ __forceinline__ void sheet_point(const SheetEval &a, const FaddeevaTables &ft, bool isH, int task, int p,
                                            int time, size_t so)
{
    const int kind = KIND > 0 ? KIND : a.kind;
    int z = a.sheet.kp + a.off;
    double *J1 = a.sheet.J[a.t1] + so, *J2 = a.sheet.J[a.t2] + so;
    const PulseParams &P = a.pulse;
    if (kind == 1) {
        const int nx = a.nx2 - 2, ny = a.ny2 - 2;
        const bool hx = pulse_half_x(isH, task), hy = pulse_half_y(isH, task);
        const int nyp = mirror_points(ny, hy);
        const int pa = p / nyp, pb = p - pa * nyp;
        int i, im, j, jm;
        mirror_cells(nx, hx, pa, i, im);
        mirror_cells(ny, hy, pb, j, jm);
        double v;
        if (!isH) {
            // getHField, src/shortpulseinject.cpp:151-178
            double poszh = (z - 0.5 - P.centrez) * P.DZ - P.ZShift;
            double posTime = (time - 0.5) * P.DT - P.TShift;
            if (task == 0) {
                double posxo = (i - P.centrex) * P.DX;
                double posyh = (j + 0.5 - P.centrey) * P.DY;
                v = P.amp * pulse_bfunc(P, ft, posxo, posyh, poszh, posTime, true).re;
            } else {
                double posxh = (i + 0.5 - P.centrex) * P.DX;
                double posyo = (j - P.centrey) * P.DY;
                v = P.amp * pulse_bfunc(P, ft, posxh, posyo, poszh, posTime, false).re;
            }
        } else {
            // getEField, src/shortpulseinject.cpp:126-149
            double posxh = (i + 0.5 - P.centrex) * P.DX;
            double posyo = (j - P.centrey) * P.DY;
            double poszo = (z - P.centrez) * P.DZ - P.ZShift;
            double posTime = time * P.DT - P.TShift;
            v = P.amp * pulse_efunc(P, ft, posxh, posyo, poszo, posTime).re;
        }
        v = v / a.DX;
        // J[t1] takes the y component of the sampled field, J[t2] the x component; the H sheet
        // samples E_x only, its J[t1] is zero
        const bool odd = !isH && task == 0;
        double *J = (isH || task == 0) ? J2 : J1;
        const size_t ny2 = a.ny2;
        const size_t q00 = i * ny2 + j, q01 = i * ny2 + jm, q10 = im * ny2 + j, q11 = im * ny2 + jm;
        J[q00] = v;
        if (jm != j) J[q01] = odd ? -v : v;
        if (im != i) {
            J[q10] = odd ? -v : v;
            if (jm != j) J[q11] = v;
        }
        if (isH) J1[q00] = J1[q01] = J1[q10] = J1[q11] = 0.0;
        return;
    }
    const int i = p / a.ny2, j = p - i * a.ny2;
    double f[3] = {0, 0, 0};
    if (kind == 4) {
        // GaussInjectSourceFunc::getHField / getEField, src/gaussinject.cpp:203-224
        const GaussSheetParams &G = a.gauss;
        if (G.active) {
            const size_t q = ((size_t)(time - G.blockToff) * a.nx2 + i) * a.ny2 + j;
            if (!isH) {
                f[0] = G.sqeps * G.amp * G.F1[q];
            } else {
                f[0] = G.amp * G.F1[q];
                f[1] = G.amp * G.F2[q];
            }
        }
    } else if (kind == 3) {
        // amp Re[env(t - z/v) U exp(-i(om0 t - phase))], env(s) = exp(-s^2/T^2)
        const FocusedParams &F = a.focused;
        double t = isH ? time * F.DT - F.TShift : (time - 0.5) * F.DT - F.TShift;
        double zf = isH ? F.zE : F.zB;
        double s = t - zf / F.v;
        double env = F.amp * exp(-(s * s) / (F.T * F.T));
        double sn, cs;
        sincos(-(F.om0 * t - F.phase), &sn, &cs);
        if (isH) {
            double2 u = F.ex[p];
            f[0] = env * (u.x * cs - u.y * sn);
        } else {
            double2 u = F.bx[p], w = F.by[p];
            f[0] = env * (u.x * cs - u.y * sn);
            f[1] = env * (w.x * cs - w.y * sn);
        }
    } else {
        if (!isH)
            plane_getH(a.plane, i, j, z, time, f);
        else
            plane_getE(a.plane, i, j, z, time, f);
    }
    J1[p] = f[a.t2] / a.DX;
    J2[p] = f[a.t1] / a.DX;
}

// One source's E sheet for steps tE .. tE + nE - 1 and H sheet for steps tH .. tH + nH - 1:
// blockIdx.y counts the components (the ntE of the E sheet first), blockIdx.z the steps; step q
// of n goes to slot n - 1 - q, so the last one lands in slot 0, the layer that reads see.
template <int KIND>
__global__ __launch_bounds__(64) void k_sheet_steps(SheetEval e, SheetEval h, FaddeevaTables ft, int ntE, int nE, int tE,
                                                    int nH, int tH)
{
    const int p = blockIdx.x * 64 + threadIdx.x;
    const int q = blockIdx.z, t = blockIdx.y;
    if (t < ntE) {
        if (q >= nE || p >= points_of(KIND, false, t, e.nx2, e.ny2)) return;
        sheet_point<KIND>(e, ft, false, t, p, tE + q, (size_t)(nE - 1 - q) * e.nx2 * e.ny2);
    } else {
        if (q >= nH || p >= points_of(KIND, true, 0, h.nx2, h.ny2)) return;
        sheet_point<KIND>(h, ft, true, 0, p, tH + q, (size_t)(nH - 1 - q) * h.nx2 * h.ny2);
    }
}

// The sheets of many runs in one launch, one list entry per component.  Entry s owns blocks
// first[s] .. first[s+1]-1, one block per 64 points; the step is *time + tstep (the counter
// lives on the device so that a captured graph can be replayed at later steps), hshift less for
// the H currents.  Only the sheets of the sides in `sides` (bit 0: E currents, bit 1: H
// currents) are evaluated.
template <int KIND>
__global__ __launch_bounds__(64) void k_sheet_eval_batch(const SheetTask *__restrict__ list,
                                                         const int *__restrict__ first, int n, FaddeevaTables ft,
                                                         const int *__restrict__ time, int tstep, int hshift,
                                                         int sides)
{
    const int b = blockIdx.x;
    int lo = 0, hi = n - 1;  // last entry with first[s] <= b
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= b) lo = mid; else hi = mid - 1;
    }
    const SheetEval &a = list[lo].ev;
    const bool isH = a.isH != 0;
    if (!(sides >> (isH ? 1 : 0) & 1)) return;
    const int p = (b - first[lo]) * 64 + threadIdx.x;
    if (p >= list[lo].points) return;
    sheet_point<KIND>(a, ft, isH, list[lo].task, p, *time + tstep - (isH ? hshift : 0), 0);
}

__global__ void k_advance_time(int *time, int k)
{
    if (threadIdx.x == 0) *time += k;
}

int sheet_tasks(const SheetEval &a) { return tasks_of(a.kind, a.isH != 0); }
int sheet_points(const SheetEval &a, int task) { return points_of(a.kind, a.isH != 0, task, a.nx2, a.ny2); }

// Slots of a solver whose sheets hold `points` evaluated points per step: as many steps as give
// the chip 2^19 threads (512 per SIMD lane group of 64: beyond that a launch is throughput
// bound and longer windows only hold memory), at most 32 (the rest of a step then outweighs a
// 32nd of the chain's latency)
int sheet_slots(long long points)
{
    const long long n = points > 0 ? (1LL << 19) / points : 1;
    return (int)(n < 1 ? 1 : (n > 32 ? 32 : n));
}

void launch_sheet_eval_batch(const SheetTask *list, const int *first, int n, int blocks, bool pulses,
                             const FaddeevaTables &ft, const int *time, int tstep, hipStream_t s, int hshift, int sides)
{
    if (pulses)
        hipLaunchKernelGGL(k_sheet_eval_batch<1>, dim3(blocks), dim3(64), 0, s, list, first, n, ft, time, tstep, hshift,
                           sides);
    else
        hipLaunchKernelGGL(k_sheet_eval_batch<0>, dim3(blocks), dim3(64), 0, s, list, first, n, ft, time, tstep, hshift,
                           sides);
}

void launch_advance_time(int *time, int k, hipStream_t s)
{
    hipLaunchKernelGGL(k_advance_time, dim3(1), dim3(64), 0, s, time, k);
}

void launch_sheet_steps(const SheetEval *e, int tE, int nE, const SheetEval *h, int tH, int nH,
                        const FaddeevaTables &ft, hipStream_t s)
{
    if (!e) nE = 0;
    if (!h) nH = 0;
    const SheetEval &any = e ? *e : *h;
    const int ntE = nE ? sheet_tasks(*e) : 0, ntH = nH ? 1 : 0;
    int pts = nH ? sheet_points(*h, 0) : 0;
    for (int t = 0; t < ntE; ++t) pts = pts > sheet_points(*e, t) ? pts : sheet_points(*e, t);
    dim3 blk(64), grd((pts + 63) / 64, ntE + ntH, nE > nH ? nE : nH);
    const SheetEval &a = e ? *e : any, &b = h ? *h : any;
    switch (any.kind) {
    case 1: hipLaunchKernelGGL(k_sheet_steps<1>, grd, blk, 0, s, a, b, ft, ntE, nE, tE, nH, tH); break;
    case 3: hipLaunchKernelGGL(k_sheet_steps<3>, grd, blk, 0, s, a, b, ft, ntE, nE, tE, nH, tH); break;
    case 4: hipLaunchKernelGGL(k_sheet_steps<4>, grd, blk, 0, s, a, b, ft, ntE, nE, tE, nH, tH); break;
    default: hipLaunchKernelGGL(k_sheet_steps<2>, grd, blk, 0, s, a, b, ft, ntE, nE, tE, nH, tH); break;
    }
}

// Re Efunc(0,0,0,0) with Phase = TShift = ZShift = 0: the amplitude normalisation of
// ShortPulseInjectSourceFunc::setParam, src/shortpulseinject.cpp:101-112
__global__ void k_pulse_norm(PulseParams P, FaddeevaTables ft, double *out)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *out = pulse_efunc(P, ft, 0, 0, 0, 0).re;
}

double pulse_norm_device(const PulseParams &P, const FaddeevaTables &ft, hipStream_t s)
{
    double *d = nullptr, h = 0;
    if (dev_malloc(&d, sizeof(double)) != hipSuccess) return NAN;
    hipLaunchKernelGGL(k_pulse_norm, dim3(1), dim3(64), 0, s, P, ft, d);
    if (hipMemcpyAsync(&h, d, sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess) h = NAN;
    if (hipStreamSynchronize(s) != hipSuccess) h = NAN;
    (void)hipFree(d);
    return h;
}

}  // namespace mpx
