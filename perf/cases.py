"""The work whose speed matters to a user of this package, case by case.

A case is one pass of a program that keeps a solver on the GPU, advances it and reads the
fields it writes out: `step` (one call for many steps, or one step a call as a driver with
per-step diagnostics makes them), the energy diagnostic, and `fetch_async` into page-locked host
arrays, the route of the field output.  Every pass injects the window of the pulse around its
peak again (`set_time`), as a pulse train does, so that the fields stay of the order of the
source.  Units are those of mpulse_amd.configs: length lambda / 2 pi, eps0 = mu0 = c = 1.

`exact` is the same scheme in plain torch float64 on interior cells with periodic rolls (PLRC
recursion, Kerr solve, CPML, source sheets, plasma, the three simple solvers); gradients come
from autograd.
"""
import math
import random

import numpy as np
import torch

from mpulse_amd import abi

DX = 2 * math.pi / 20  # lambda / 20
DT = 0.5 * DX / math.sqrt(3)
T10FS = 10e-15 / (800e-9 / (2 * math.pi) / 299792458.0) / math.sqrt(2 * math.log(2))  # 10 fs intensity FWHM
FIELDS = ("Ex", "Ey", "Ez", "Bx", "By", "Bz")
POLES = {0: (), 1: ((1.1, 4.0, 0.005),),
         2: ((0.69, (0.8 / 0.068) ** 2, 0.0), (0.87, (0.8 / 9.9) ** 2, 0.0)),
         3: ((1.1, 4.0, 0.005), (0.3, 0.5, 0.002), (0.2, 9.0, 0.01))}  # (delta eps, Omega^2, damping)
SOLVERS = {"nonlin": abi.SOLVER_PLRC_NONLIN, "lin": abi.SOLVER_PLRC_LIN, "plain": abi.SOLVER_PLAIN,
           "nl": abi.SOLVER_NL, "disp": abi.SOLVER_DISP}
PRECISIONS = {"fp64": abi.PREC_FP64, "fp32_bulk": abi.PREC_FP32_BULK, "fp32_res": abi.PREC_FP32_RES}
PATHS = {"fused": abi.PATH_FUSED, "pass": abi.PATH_PASS, "sweep": abi.PATH_SWEEP}


def _pulse(name, grid, steps, **kw):
    c = {"name": name, "kind": "pulse", "nx": grid[0], "ny": grid[1], "nz": grid[2], "steps": steps, "a_call": steps,
         "warm": 100, "solver": "nonlin", "prec": "fp64", "path": "fused", "poles": 1, "cpml": 10, "cpml_1d": False,
         "xy": False, "source": "short", "plasma": False, "energies": 0, "fields": "EB"}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest: a driver that advances one step a call and watches the energy
        _pulse("tiny_step_a_call", (24, 24, 24), 8, a_call=1, cpml=4, energies=1),
        # the 64^3 parity workload, float64 on the default (fused) path
        _pulse("small_fused", (64, 64, 64), 100),
        # a setup file through the C++ driver, the way the reference's users run it
        {"name": "setup_file", "kind": "setup", "nx": 48, "ny": 40, "nz": 56, "steps": 150},
        # an ordinary float64 run on odd sizes with the energy diagnostic every 15 steps
        _pulse("medium_fused_odd", (131, 158, 177), 60, energies=4),
        # the single-precision-storage production form on a mid-size and on the 512^3 grid
        _pulse("mid_res_pass", (256, 256, 256), 100, prec="fp32_res", path="pass", cpml=16),
        _pulse("large_res_pass", (512, 512, 512), 96, prec="fp32_res", path="pass", cpml=16, warm=48, fields="E"),
        # the two-pole focused-pulse medium, float32 storage
        _pulse("focus_bulk_two_poles", (160, 160, 320), 80, prec="fp32_bulk", poles=2, cpml=16, source="focus"),
        # the uneven-size parameter sweep
        {"name": "batch_sweep", "kind": "batch", "runs": 10, "nmin": 48, "nmax": 160, "sizes": 1, "steps": 60,
         "prec": "fp64", "structure": 2},
        # the gradient with respect to a per-cell permittivity
        {"name": "adjoint", "kind": "adjoint", "nx": 128, "ny": 128, "nz": 256, "poles": 0, "steps": 100, "every": 50,
         "solver": "nonlin"},
        # ionisation and plasma current, float64 on the pass path
        _pulse("plasma_pass", (96, 88, 120), 60, path="pass", plasma=True),
        # a ramped plane wave in a long column: linear core, open z boundary
        _pulse("column_linear_open", (60, 75, 260), 60, solver="lin", xy=True, source="plane", cpml_1d=True),
        # the three-oscillator ADE solver from a given state
        {"name": "dispersive_state", "kind": "state", "solver": "disp", "nx": 120, "ny": 112, "nz": 100, "steps": 60},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pulse", "pulse", "pulse", "pulse", "batch", "adjoint", "state", "setup"])
    if kind == "pulse":
        grid = [_size(rng, 22, 330) for _ in range(3)]
        cells = grid[0] * grid[1] * grid[2]
        steps = max(4, min(100, int(4e8 / cells)))
        c = _pulse("", grid, steps, a_call=rng.choice([1, steps, steps]), warm=40, cpml=rng.choice([4, 6, 8]),
                   solver=rng.choice(["nonlin", "nonlin", "lin"]), prec=rng.choice(["fp64", "fp64", "fp32_res", "fp32_bulk"]),
                   path=rng.choice(["fused", "pass", "pass"]), poles=rng.choice([0, 1, 1, 2, 3]),
                   source=rng.choice(["short", "short", "plane"]), energies=rng.choice([0, 1]))
        c["xy"] = rng.random() < 0.2
        c["cpml_1d"] = rng.random() < 0.15
        c["plasma"] = rng.random() < 0.2
    elif kind == "batch":
        lo = _size(rng, 26, 60)
        c = {"kind": kind, "runs": rng.randint(3, 10), "nmin": lo, "nmax": lo + rng.randint(5, 90),
             "sizes": rng.randrange(1 << 20), "steps": rng.randint(10, 60), "prec": rng.choice(["fp64", "fp32_bulk"]),
             "structure": rng.choice([0, 2, 2])}
    elif kind == "adjoint":
        c = {"kind": kind, "nx": _size(rng, 24, 140), "ny": _size(rng, 24, 140), "nz": _size(rng, 40, 260),
             "poles": rng.choice([0, 0, 1]), "steps": rng.randint(30, 100), "every": rng.choice([10, 25, 50]),
             "solver": rng.choice(["nonlin", "nonlin", "lin"])}
    elif kind == "state":
        c = {"kind": kind, "solver": rng.choice(["plain", "nl", "disp"]), "nx": _size(rng, 16, 200),
             "ny": _size(rng, 16, 200), "nz": _size(rng, 16, 200), "steps": rng.randint(5, 80)}
    else:
        c = {"kind": kind, "nx": _size(rng, 24, 90), "ny": _size(rng, 24, 90), "nz": _size(rng, 28, 90),
             "steps": rng.randint(20, 200)}
    c.pop("name", None)
    return c


# ---- what a seed decides: the physical parameters of a case ----------------------------------


def _medium_eps(poles):
    return 1.0 + sum(de * om2 / (om2 - 1.0) for de, om2, _ in poles)


def _numbers(case, seed, d_cpml, grid):
    """The pulse, the medium and the start step of one run (plain numbers, shared with exact)."""
    r = random.Random(int(seed) * 1009 + 17)
    p = {"phase": r.random(), "amp": r.uniform(0.5, 5.0), "chi": 10.0 ** r.uniform(-5.0, -3.0),
         "length": T10FS * r.uniform(0.9, 1.1), "width": r.uniform(0.18, 0.25) * min(grid[0], grid[1], 96) * DX,
         "tilt": r.randint(0, 1), "om": r.uniform(0.9, 1.1), "jitter": r.randint(-20, 20)}
    p["tshift"] = 2 * p["length"]
    p["d_src"] = d_cpml + 2
    p["start"] = max(0, int(p["tshift"] / DT) - case.get("warm", 100) - case["steps"] // 2 + p["jitter"])
    p["sigma"] = 4 * math.log(1e6) / (2 * d_cpml * DX)
    return p


def _desc(case, p, grid, poles, d_cpml):
    d = abi.desc_defaults()
    d.nx, d.ny, d.nz = grid
    d.dx = d.dy = d.dz = DX
    d.dt = DT
    d.solver = SOLVERS[case["solver"]]
    d.precision = PRECISIONS[case.get("prec", "fp64")]
    d.path = PATHS[case.get("path", "fused")]
    d.boundary = abi.BOUNDARY_XY_PERIODIC if case.get("xy") else abi.BOUNDARY_PERIODIC
    d.eps, d.chi = 1.0, p["chi"]
    for q in range(3):
        d.l_eps[q], d.l_om2[q], d.l_delta[q] = poles[q] if q < len(poles) else (0.0, 1.0, 0.0)
    cp = abi.factory_defaults(abi.FACTORY_CPML_1D if case.get("cpml_1d") else abi.FACTORY_CPML)
    cp.d, cp.sigma_max = d_cpml, p["sigma"]
    abi.add_factory(d, cp)
    source = case.get("source", "short")
    f = abi.factory_defaults({"short": abi.FACTORY_SHORT_PULSE, "focus": abi.FACTORY_FOCUSED_PULSE,
                              "plane": abi.FACTORY_PLANE_WAVE}[source])
    f.d, f.eps, f.om0, f.amp = p["d_src"], _medium_eps(poles), 1.0, p["amp"]
    f.length, f.width, f.phase, f.tshift = p["length"], p["width"], p["phase"], p["tshift"]
    f.zshift = 0.0 if source == "focus" else (p["d_src"] - 0.5 * (grid[2] + 1)) * DX
    if source == "plane":
        f.h[0], f.h[1], f.h[2] = 0.3 * p["amp"], p["amp"], 0.0
        f.k[0], f.k[1], f.k[2] = p["tilt"] * 2 * math.pi / (grid[0] * DX), 0.0, p["om"]
        f.ramp, f.h_bg[0], f.e_bg[1] = 0.5, 0.01, 0.02
    abi.add_factory(d, f)
    if case.get("plasma"):
        c = abi.factory_defaults(abi.FACTORY_PLASMA_CURRENT)
        c.em, c.gamma, c.rho_bg = 0.8, 0.2, 0.01
        abi.add_factory(d, c)
        d.plasma, d.plasma_k, d.plasma_nu, d.plasma_mpa, d.plasma_wion = 1, 3, 1e-3, 1e-5, 0.5
    return d


def _grid(case):
    return case["nx"], case["ny"], case["nz"]


def _batch_runs(case, seed):
    """Per run: (grid, numbers).  Sizes belong to the case, the pulses to the seed."""
    r = random.Random(case["sizes"])
    out = []
    for q in range(case["runs"]):
        n = r.randint(case["nmin"], case["nmax"])
        sub = {"solver": "nonlin", "prec": case["prec"], "steps": case["steps"], "warm": 0}
        p = _numbers(sub, int(seed) * 64 + q, 6, (n, n, n))
        p["tshift"] = 0.4 * p["length"]  # a batch's clock starts at 0: the peak comes early
        out.append((sub, (n, n, n), p))
    return out


def _smooth(shape, r, terms=4):
    """A smooth periodic field on the interior, about [-1, 1]: a few low Fourier modes."""
    ax = [np.arange(n) * (2 * math.pi / n) for n in shape]
    f = np.zeros(shape)
    for _ in range(terms):
        k = [r.randint(1, 3) for _ in range(3)]
        ph = [r.uniform(0, 2 * math.pi) for _ in range(3)]
        f += (np.cos(k[0] * ax[0] + ph[0])[:, None, None] * np.cos(k[1] * ax[1] + ph[1])[None, :, None]
              * np.cos(k[2] * ax[2] + ph[2])[None, None, :]) / terms
    return f


def _state_fields(case, seed):
    """Interior E and B of a simple solver: smooth fields, E_x offset from zero (fdtd-nl needs D > 0)."""
    r = random.Random(int(seed) * 31 + 5)
    out = {n: 0.3 * _smooth(_grid(case), r) for n in FIELDS}
    out["Ex"] += 1.0
    return out


def _eps_cells(case, seed):
    """Per-cell permittivity in [1, 2.25] of the gradient case (interior)."""
    r = random.Random(int(seed) * 7 + 3)
    return 1.625 + 0.625 * np.clip(_smooth(_grid(case), r), -1, 1)


SETUP = """
globals {{ grid-x {nx} grid-y {ny} grid-z {nz} grid-dx {dx!r} grid-dy {dx!r} grid-dz {dx!r} dt {dt!r}
          T-total 1000000 }}
fieldsim {{
  fdtd-plrc-nonlin {{ eps 1 chi {chi!r}  L1eps 1.1 L1Om2 4 L1delta 0.005 L2eps 0 L2Om2 1 L3eps 0 L3Om2 1
                     cpml_border {{ d 6 kappaMax 15 aMax 0.25 sigmaMax {sigma!r} }}
                     short_pulse_inject {{ d 8 length {length!r} width {width!r} om0 1 amp {amp!r} eps {eps!r}
                                          TShift {tshift!r} ZShift {zshift!r} Phase {phase!r} }} }}
  single_periodic
}}
"""


def _setup_numbers(case, seed):
    p = _numbers({"steps": case["steps"], "warm": 0}, seed, 6, _grid(case))
    p["tshift"] = 0.5 * p["length"]  # the driver's clock starts at 0: the peak comes early
    return p


# ---- the work ------------------------------------------------------------------------------


def _pinned(grid, names):
    shape = tuple(n + 2 for n in reversed(grid))
    return {n: torch.empty(shape, dtype=torch.float64, pin_memory=True) for n in names}


def _names(case):
    return FIELDS[:3] if case.get("fields") == "E" else FIELDS


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pulse":
        grid = _grid(case)
        p = _numbers(case, seed, case["cpml"], grid)
        s = abi.Solver(_desc(case, p, grid, POLES[case["poles"]], case["cpml"]))
        s.set_time(p["start"])
        s.step(case["warm"])  # the pulse is on its way
        return {"case": case, "solver": s, "time": p["start"] + case["warm"], "host": _pinned(grid, _names(case))}
    if kind == "batch":
        runs = _batch_runs(case, seed)
        b = abi.Batch([_desc(sub, p, grid, POLES[1], 6) for sub, grid, p in runs])
        b.tune("structure", case["structure"])
        return {"case": case, "batch": b, "views": [b.run(q) for q in range(len(runs))],
                "host": [_pinned(grid, FIELDS) for _, grid, _ in runs]}
    if kind == "adjoint":
        grid = _grid(case)
        p = _numbers(case, seed, 6, grid)
        s = abi.Solver(_desc(case, p, grid, POLES[case["poles"]], 6))
        full = np.pad(_eps_cells(case, seed), 1, constant_values=1.0)
        s.set("Eps", full)
        return {"case": case, "solver": s, "time": p["start"], "plane": p["d_src"] + 6}
    if kind == "state":
        d = abi.desc_defaults()
        d.nx, d.ny, d.nz = _grid(case)
        d.dx = d.dy = d.dz = DX
        d.dt = DT
        d.solver = SOLVERS[case["solver"]]
        d.eps, d.chi = 1.2, 0.05
        for q in range(3):
            d.d_eps2[q], d.d_om2[q] = 0.2 * (q + 1), 0.5 + q
        s = abi.Solver(d)
        for n, f in _state_fields(case, seed).items():
            s.set(n, np.pad(f, 1, mode="wrap"))
        return {"case": case, "solver": s, "host": _pinned(_grid(case), FIELDS)}
    p = _setup_numbers(case, seed)
    text = SETUP.format(nx=case["nx"], ny=case["ny"], nz=case["nz"], dx=DX, dt=DT, eps=_medium_eps(POLES[1]),
                        zshift=(8 - 0.5 * (case["nz"] + 1)) * DX,
                        **{k: p[k] for k in ("chi", "sigma", "length", "width", "amp", "tshift", "phase")})
    return {"case": case, "sim": abi.HostSimulation(text)}


def _read(solver, host):
    for h in [solver.fetch_async(n, t.numpy()) for n, t in host.items()]:
        h.wait()
    return host


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "pulse":
        s, out = state["solver"], {}
        s.set_time(state["time"])
        calls = case["steps"] // case["a_call"]
        watch = calls // case["energies"] if case["energies"] and calls >= case["energies"] else 0
        if case["energies"] and not watch:  # one call for many steps, cut where the diagnostic reads
            part = case["steps"] // case["energies"]
            out["energy"] = []
            for _ in range(case["energies"]):
                s.step(part)
                out["energy"].append(s.energy())
        else:
            for q in range(calls):
                s.step(case["a_call"])
                if watch and (q + 1) % watch == 0:
                    out.setdefault("energy", []).append(s.energy())
        out.update(_read(s, state["host"]))
        return out
    if kind == "batch":
        state["batch"].step(case["steps"])
        return [_read(v, h) for v, h in zip(state["views"], state["host"])]
    if kind == "adjoint":
        s = state["solver"]
        s.set_time(state["time"])
        J, deps, dchi = s.adjoint_grad(state["plane"], DX * DX * DT, case["steps"], case["every"])
        return {"J": J, "dJ_deps": deps, "dJ_dchi": dchi}
    if kind == "state":
        state["solver"].step(case["steps"])
        return _read(state["solver"], state["host"])
    state["sim"].run(case["steps"])
    return {n: state["sim"].get(n) for n in FIELDS}


def work(case):
    kind = case["kind"]

    def stepping(grid, w, poles, d, one_d, steps, words=12):
        nx, ny, nz = grid
        cells = nx * ny * nz
        layer = 2 * d * (nx * ny if one_d else nx * ny + ny * nz + nx * nz)
        return (cells * (words * w + 96 * poles) + 8 * w * layer) * steps, cells * steps * (90 + 45 * poles)

    def boxes(grid, n):
        return 8 * n * (grid[0] + 2) * (grid[1] + 2) * (grid[2] + 2)

    if kind == "pulse":
        w = {"fp64": 8, "fp32_bulk": 4, "fp32_res": 16 / 3}[case["prec"]]
        b, f = stepping(_grid(case), w, case["poles"], case["cpml"], case["cpml_1d"], case["steps"])
        if case["plasma"]:
            b += case["nx"] * case["ny"] * case["nz"] * 8 * 8 * case["steps"]  # density and current, read and written
        b += boxes(_grid(case), len(_names(case)))
    elif kind == "batch":
        b = f = 0
        for _, grid, _ in _batch_runs(case, 0):
            x, y = stepping(grid, 8 if case["prec"] == "fp64" else 4, 1, 6, False, case["steps"])
            b, f = b + x + boxes(grid, 6), f + y
    elif kind == "adjoint":
        # forward, the forward again for the history, and the reverse step: the adjoints of E, B and
        # the accumulators read and written, E read, the permittivity and its gradient
        b, f = stepping(_grid(case), 8, case["poles"], 6, False, case["steps"])
        cells = case["nx"] * case["ny"] * case["nz"]
        b = 2 * b + (cells * 8 * (12 + 3 + 1 + 2) + cells * 96 * case["poles"]) * case["steps"] + boxes(_grid(case), 1)
        f *= 4
    elif kind == "state":
        words = 12 + (36 if case["solver"] == "disp" else 0)
        b, f = stepping(_grid(case), 8, 0, 0, True, case["steps"], words)
        b += boxes(_grid(case), 6)
    else:
        b, f = stepping(_grid(case), 8, 1, 6, False, case["steps"])
        b += boxes(_grid(case), 6)
    return {"bytes": b, "flops": f}


# ---- the same in plain torch float64 ---------------------------------------------------------


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.asarray(a), dtype=torch.float64, device=_dev())


def _line(v, dim):
    shape = [1, 1, 1]
    shape[dim] = -1
    return _t(v).reshape(shape)


def _faddeeva(z):
    """w(z), Im z >= 0: the trapezoid rule with step 1/2 and, below Im z = 2 pi, the residue of the
    poles it passes (Matta and Reichel, Math. Comp. 25, 1971)."""
    h = 0.5
    s = 1 / z
    for q in range(1, 13):
        s = s + 2 * math.exp(-(q * h) ** 2) * z / (z * z - (q * h) ** 2)
    low = z.imag < math.pi / h
    zl = torch.where(low, z, torch.full_like(z, 1j))
    return 1j * h / math.pi * s + torch.where(low, 2 * torch.exp(-zl * zl) / (1 - torch.exp(-2j * math.pi / h * zl)), 0 * zl)


class _ShortPulse:
    """The closed-form short pulse on one plane: E_x, or (B_x, B_y)."""

    def __init__(self, p, eps, grid):
        self.c = math.sqrt(1 / eps)
        self.T, self.width = p["length"], p["width"]
        self.zr = 0.5 * self.width ** 2 / self.c
        self.p, self.grid = p, grid
        zero = torch.zeros(1, dtype=torch.float64, device=_dev())
        self.amp = p["amp"] / float(self.efield(zero, 0.0, 0.0, 0.0).real[0])

    def _parts(self, r2, z, t, phase):
        T, c, tb = self.T, self.c, 0.5 * self.T
        q = complex(z, self.zr)
        tp = (t - z / c) - r2 / (2 * c * q)
        sides = []
        for sgn in (-1, 1):  # the two Faddeeva arguments and what their reflection adds
            a = sgn * 1j * tb + tp / T
            flip = a.imag < 0
            e = torch.where(flip, -sgn * 2j * tp * tb / T - tp * tp / T ** 2, 0 * tp)
            sides.append((_faddeeva(torch.where(flip, -a, a)), flip, torch.exp(e)))
        return q, tp, tb, np.exp(2j * phase), sides

    @staticmethod
    def _sum(A, e0, B, C, D, sides):
        (wn, fn, en), (wp, fp, ep) = sides
        S = torch.where(fn, 2 * A * C * en, 0 * wn) + torch.where(fp, 2 * A * D * ep, 0 * wp)
        C, D = torch.where(fn, -C, C), torch.where(fp, -D, D)
        return S + A * e0 * (B + C * wn - D * wp)

    def efield(self, r2, z, t, phase):
        T, c, zr = self.T, self.c, self.zr
        r2 = r2.to(torch.complex128)
        q, tp, tb, ei, sides = self._parts(r2, z, t, phase)
        rt, rpt = zr / q, -zr / q ** 2
        rpi = math.sqrt(math.pi) * rt
        tz = -1 / c - r2 / (2 * c * q * q)
        A = np.exp(-1j * phase) / (rpi * T ** 4)
        B = rt * T * (1j * (1 + ei) * rpt * T ** 2
                      - rt * (T * ((-1j - 2 * tb) + ei * (-1j + 2 * tb)) + 2j * (1 + ei) * tp) * tz)
        C = 1j * ei * rpi * (T * tb + 1j * tp) * (rpt * T ** 2 + 2j * rt * T * tb * tz - 2 * rt * tp * tz)
        D = rpi * (T * tb - 1j * tp) * (1j * rpt * T ** 2 + 2 * rt * (T * tb - 1j * tp) * tz)
        return -1j * self._sum(A, math.exp(-tb * tb), B, C, D, sides)

    def bfield(self, x, y, z, t, phase, bx):
        T, c, zr = self.T, self.c, self.zr
        x, y = x.to(torch.complex128), y.to(torch.complex128)
        r2 = x * x + y * y
        q, tp, tb, ei, sides = self._parts(r2, z, t, phase)
        rt, rpt, rppt = zr / q, -zr / q ** 2, 2 * zr / q ** 3
        sp = math.sqrt(math.pi)
        rpi = sp * rt
        tz, tzz = -1 / c + r2 / (2 * c * q * q), -r2 / (c * q ** 3)
        tx, ty, txx = -x / (c * q), -y / (c * q), -1 / (c * q)
        ap, an = T * tb + 1j * tp, T * tb - 1j * tp
        br = T * ((-1j - 2 * tb) + ei * (-1j + 2 * tb)) + 2j * (1 + ei) * tp
        e0 = math.exp(-tb * tb)
        A = np.exp(-1j * phase) / (sp * T ** 4)
        if bx:
            return 1j * self._sum(A, e0, -tx * ty * rt * T * br, -tx * ty * 2 * ei * rpi * ap * ap,
                                  -tx * ty * 2 * rpi * an * an, sides)
        Bb = self._sum(A, e0, -tx * tx * rt * T * br + 1j * T ** 2 * txx * (1 + ei) * rt * T,
                       -tx * tx * 2 * ei * rpi * ap * ap + 1j * T ** 2 * txx * ei * rpi * ap,
                       -tx * tx * 2 * rpi * an * an + 1j * T ** 2 * txx * rpi * (-T * tb + 1j * tp), sides)
        DB = 2 * T * (2j * (1 + ei) * rpt * T ** 2 * tz
                      - rt * (T * ((-1j - 2 * tb) + ei * (-1j + 2 * tb)) * tz * tz
                              + 1j * (1 + ei) * (2 * tp * tz * tz - T ** 2 * tzz)))
        r4 = rt * T ** 4
        DC = ei * rpi * (rppt * r4 + 2j * rt * ap * (2 * rpt * T ** 2 * tz + rt * (
            2j * T * tb * tz * tz - 2 * tp * tz * tz + T ** 2 * tzz))) / rt ** 2
        DD = rpi * (rppt * r4 - 2 * rt * an * (2j * rpt * T ** 2 * tz + rt * (
            2 * T * tb * tz * tz - 2j * tp * tz * tz + 1j * T ** 2 * tzz))) / rt ** 2
        Bd = self._sum(A / 2, e0, DB, DC, DD, sides)
        return 1j * (Bd - Bb)

    def _axes(self, sx, sy):
        nx, ny, _ = self.grid
        x = (torch.arange(1, nx + 1, dtype=torch.float64, device=_dev()) + sx - 0.5 * (nx + 1)) * DX
        y = (torch.arange(1, ny + 1, dtype=torch.float64, device=_dev()) + sy - 0.5 * (ny + 1)) * DX
        return torch.broadcast_tensors(x[:, None], y[None, :])

    def sheet(self, time, magnetic):
        """(J_x, J_y) of the E current (magnetic False) or of the H current at a step."""
        p = self.p
        ph, cz = 2 * math.pi * p["phase"], 0.5 * (self.grid[2] + 1)
        zs = (p["d_src"] - cz) * DX
        k = p["d_src"] - 1
        if magnetic:
            x, y = self._axes(0.5, 0.0)
            e = self.efield(x * x + y * y, (k - cz) * DX - zs, time * DT - p["tshift"], ph)
            return None, self.amp * e.real / DX
        z, t = (k - 0.5 - cz) * DX - zs, (time - 0.5) * DT - p["tshift"]
        bx = self.bfield(*self._axes(0.0, 0.5), z, t, ph, True)
        by = self.bfield(*self._axes(0.5, 0.0), z, t, ph, False)
        return self.amp * by.real / DX, self.amp * bx.real / DX


class _Focused:
    """The focused pulse: an angular spectrum on the transverse grid, a Gaussian envelope in time."""

    def __init__(self, p, eps, grid):
        nx, ny, nz = grid
        self.p, self.v = p, math.sqrt(1 / eps)
        k = math.sqrt(eps)
        cz = 0.5 * (nz + 1)
        self.z = {"E": (p["d_src"] - 1 - cz) * DX, "B": (p["d_src"] - 1.5 - cz) * DX}
        kx = _t(2 * math.pi * (np.arange(nx) - nx // 2) / (nx * DX))[:, None]
        ky = _t(2 * math.pi * (np.arange(ny) - ny // 2) / (ny * DX))[None, :]
        kp2 = kx * kx + ky * ky
        live = kp2 < k * k
        kz = torch.sqrt(torch.where(live, k * k - kp2, torch.ones_like(kp2)))
        A = torch.where(live, torch.exp(-kp2 * p["width"] ** 2 / 4), torch.zeros_like(kp2))
        amps = {"ex": (A, "E", 0.5, 0.0), "bx": (-kx * ky * A / kz, "B", 0.0, 0.5),
                "by": (A * (kz * kz + kx * kx) / kz, "B", 0.5, 0.0)}
        self.u = {}
        for n, (g, where, sx, sy) in amps.items():
            x = (_t(np.arange(1, nx + 1)) + sx - 0.5 * (nx + 1)) * DX
            y = (_t(np.arange(1, ny + 1)) + sy - 0.5 * (ny + 1)) * DX
            G = g * torch.exp(1j * kz * self.z[where])
            self.u[n] = torch.exp(1j * x[:, None] * kx[:, 0]) @ G @ torch.exp(1j * ky[0][:, None] * y) / A.sum()

    def sheet(self, time, magnetic):
        p = self.p
        t = (time if magnetic else time - 0.5) * DT - p["tshift"]
        s = t - self.z["E" if magnetic else "B"] / self.v
        env = p["amp"] * math.exp(-s * s / p["length"] ** 2)
        ph = np.exp(-1j * (t - 2 * math.pi * p["phase"]))
        if magnetic:
            return None, env * (self.u["ex"] * ph).real / DX
        return env * (self.u["by"] * ph).real / DX, env * (self.u["bx"] * ph).real / DX


class _Plane:
    """The ramped plane wave with background fields."""

    def __init__(self, p, eps, grid):
        self.p, self.grid = p, grid
        self.k = np.array([p["tilt"] * 2 * math.pi / (grid[0] * DX), 0.0, p["om"]])
        self.h = np.array([0.3 * p["amp"], p["amp"], 0.0])
        e = np.cross(self.k, self.h)
        self.e = -e * np.linalg.norm(self.h) / np.linalg.norm(e) / math.sqrt(eps)
        self.om = np.linalg.norm(self.k) / math.sqrt(eps)

    def sheet(self, time, magnetic):
        nx, ny, _ = self.grid
        i, j, l = _t(np.arange(1, nx + 1))[:, None], _t(np.arange(1, ny + 1))[None, :], self.p["d_src"] - 1
        out = []
        for d in range(2):
            half = [0.5] * 3 if not magnetic else [0.0] * 3
            half[d] = 0.0 if not magnetic else 0.5
            pos = (self.k[0] * (i + half[0]) + self.k[1] * (j + half[1]) + self.k[2] * (l + half[2])) * DX \
                + self.om * DT * (time if magnetic else time - 0.5)
            bg = ((0.01, 0.0) if not magnetic else (0.0, 0.02))[d]
            f = (self.e if magnetic else self.h)[d] * torch.sin(pos) + bg
            out.append(torch.where(pos < 0.5, f * pos / 0.5, f) / DX)
        return out[1], out[0]


def _cpml_lines(n, d, sigma, one_d):
    """kappa of the E and H side on 0 .. n + 1, and b, c of both (zero outside the layers)."""
    high = n + 1
    kE, kH = np.ones(n + 2), np.ones(n + 2)
    cube = lambda x: 1 + 14 * x ** 3  # noqa: E731
    if one_d:
        for i in range(d):
            kE[i + 1], kH[i] = cube(1 - i / d), cube(1 - (i + 0.5) / d)
            kE[high - i - 1], kH[high - i - 1] = cube(1 - i / d), cube(1 - (i + 0.5) / d)
    else:
        for i in range(d + 1):
            kE[i], kH[high - i] = cube(1 - i / d), cube(1 - i / d)
        for i in range(d):
            kH[i], kE[high - i] = cube(1 - (i + 0.5) / d), cube(1 - (i + 0.5) / d)
    tables = []
    for side in (0, 1):
        b, c = np.zeros(n + 2), np.zeros(n + 2)
        for q in range(d):
            x = 1 - (q - 0.5 * side) / d
            s, kap, a = x ** 3 * sigma, 1 + 14 * x ** 3, 0.25 * (1 - x)
            bb = math.exp(-(s / kap + a) * DT)
            for at in (1 - side + q, n - q):
                b[at], c[at] = bb, s * (bb - 1) / (kap * (s + kap * a))
        tables.append((b, c))
    return kE, kH, tables


class _Yee:
    """FDTD with the PLRC poles, the Kerr solve, CPML, sheets and plasma on interior cells.  With an
    open z boundary the arrays span k = 0 .. nz + 1 in z and E outside 1 .. nz, B outside 0 .. nz
    stay zero.  The state is a tuple of tensors; a step returns a new one (autograd-safe)."""

    def __init__(self, case, p, grid, poles, d_cpml, eps_cells=None, chi=None):
        self.case, self.p, self.grid = case, p, grid
        self.nonlin = case["solver"] == "nonlin"
        xy, one_d = case.get("xy", False), case.get("cpml_1d", False)
        self.cut = [slice(1, -1), slice(1, -1), slice(None) if xy else slice(1, -1)]
        self.shape = (grid[0], grid[1], grid[2] + (2 if xy else 0))
        self.kp = p["d_src"] - (0 if xy else 1)
        self.dims = (2,) if one_d else (0, 1, 2)
        self.ikE, self.ikH, self.bc = [], [], []
        for q in range(3):
            kE, kH, tab = _cpml_lines(grid[q], d_cpml, p["sigma"], one_d)
            if q not in self.dims:
                kE, kH = np.ones(grid[q] + 2), np.ones(grid[q] + 2)
            self.ikE.append(_line(1 / (kE * DX), q)[self._at(q)])
            self.ikH.append(_line(1 / (kH * DX), q)[self._at(q)])
            self.bc.append([[_line(v, q)[self._at(q)] for v in bc] for bc in tab])
        self.mE = self.mB = None
        if xy:
            k = np.arange(grid[2] + 2)
            self.mE, self.mB = _line((k >= 1) & (k <= grid[2]), 2), _line(k <= grid[2], 2)
        eps_l = _medium_eps(poles)
        self.source = {"short": _ShortPulse, "focus": _Focused, "plane": _Plane}[case.get("source", "short")](p, eps_l, grid)
        self.poles, chi0s, xi0s = [], 0.0, 0.0
        for de, om2, dl in poles:
            beta = math.sqrt(om2 - dl * dl)
            ph = complex(dl, -beta)
            g = de * om2 / beta
            cr = np.exp(-ph * DT)
            c0 = 1j * g * (cr - 1) / ph
            x0 = 1j * g * (cr * (ph * DT + 1) - 1) / (ph * ph * DT)
            self.poles.append((complex(cr), complex((c0 - x0) * (1 - cr)), complex(x0 * (1 - cr))))
            chi0s, xi0s = chi0s + c0.real, xi0s + x0.real
        eps = 1.0 if eps_cells is None else eps_cells
        self.denom, self.numer = eps + chi0s - xi0s, eps - xi0s
        self.chi = p["chi"] if chi is None else chi

    def _at(self, q):
        s = [slice(None)] * 3
        s[q] = self.cut[q]
        return tuple(s)

    def zero(self):
        z = lambda: torch.zeros(self.shape, dtype=torch.float64, device=_dev())  # noqa: E731
        n = 6 + 4 * len(self.dims) + (4 if self.case.get("plasma") else 0)
        psi = [torch.zeros(self.shape, dtype=torch.complex128, device=_dev()) for _ in range(3 * len(self.poles))]
        return tuple([z() for _ in range(n)] + psi)

    def step(self, S, time):
        S = list(S)
        E, B, aux = S[0:3], S[3:6], 6
        diff = {}
        for d in range(3):
            for q in range(3):
                if q != d:
                    diff[d, q] = B[q] - torch.roll(B[q], 1, d)
        J = [0.0, 0.0, 0.0]
        for d in self.dims:
            (b, c), c0, c1 = self.bc[d][0], (d + 1) % 3, (d + 2) % 3
            S[aux] = b * S[aux] - c * diff[d, c1] / DX
            S[aux + 1] = b * S[aux + 1] + c * diff[d, c0] / DX
            J[c0], J[c1], aux = J[c0] + S[aux], J[c1] + S[aux + 1], aux + 2
        denom, numer = self.denom, self.numer
        n_plasma = 6 + 4 * len(self.dims)
        if self.case.get("plasma"):
            inten = E[0] ** 2 + E[1] ** 2 + E[2] ** 2
            n, m = 0.5 * DT * 1e-3, DT * 1e-5
            S[n_plasma] = (S[n_plasma] * (1 + n * inten) + m * inten ** 3) / (1 - n * inten)
            sg = 0.5 * DT * (1e-5 * 0.5 * inten ** 2)
            denom, numer = denom + sg, numer - sg
            for q in range(3):
                at = n_plasma + 1 + q
                S[at] = (S[at] * (1 - 0.1 * DT) - 0.8 * DT * E[q] * (S[n_plasma] + 0.01)) / (1 + 0.1 * DT)
                J[q] = J[q] + S[at]
        J = self._sheet(J, time, False, self.kp)
        curl = [diff[1, 2] * self.ikE[1] - diff[2, 1] * self.ikE[2], diff[2, 0] * self.ikE[2] - diff[0, 2] * self.ikE[0],
                diff[0, 1] * self.ikE[0] - diff[1, 0] * self.ikE[1]]
        at = n_plasma + (4 if self.case.get("plasma") else 0)
        psum = [0.0, 0.0, 0.0]
        for cr, dd, dx in self.poles:
            for q in range(3):
                acc = dd * E[q] + S[at]
                psum[q], S[at], at = psum[q] + acc.real, dx * E[q] + cr * acc, at + 1
        f = numer
        if self.nonlin:
            f = numer + self.chi * (E[0] ** 2 + E[1] ** 2 + E[2] ** 2)
        new = [(f * E[q] + DT * (curl[q] + J[q]) + psum[q]) / denom for q in range(3)]
        if self.nonlin:
            # E' = s C with s = 1 / (1 + A |E'|^2): A |C|^2 s^3 + s = 1; the last step carries the derivative
            aq = self.chi / denom * (new[0] ** 2 + new[1] ** 2 + new[2] ** 2)
            s = torch.ones_like(new[0])
            with torch.no_grad():
                for _ in range(8):
                    s = s - (aq * s ** 3 + s - 1) / (3 * aq * s * s + 1)
            s = s - (aq * s ** 3 + s - 1) / (3 * aq * s * s + 1).detach()
            new = [s * v for v in new]
        if self.mE is not None:
            new = [v * self.mE for v in new]
        for d in range(3):
            for q in range(3):
                if q != d:
                    diff[d, q] = torch.roll(new[q], -1, d) - new[q]
        M = [0.0, 0.0, 0.0]
        for d in self.dims:
            (b, c), c0, c1 = self.bc[d][1], (d + 1) % 3, (d + 2) % 3
            S[aux] = b * S[aux] + c * diff[d, c1] / DX
            S[aux + 1] = b * S[aux + 1] - c * diff[d, c0] / DX
            M[c0], M[c1], aux = M[c0] + S[aux], M[c1] + S[aux + 1], aux + 2
        M = self._sheet(M, time, True, self.kp - 1)
        curl = [diff[2, 1] * self.ikH[2] - diff[1, 2] * self.ikH[1], diff[0, 2] * self.ikH[0] - diff[2, 0] * self.ikH[2],
                diff[1, 0] * self.ikH[1] - diff[0, 1] * self.ikH[0]]
        B = [B[q] + DT * (curl[q] + M[q]) for q in range(3)]
        if self.mB is not None:
            B = [v * self.mB for v in B]
        S[0:6] = new + B
        return tuple(S)

    def _sheet(self, J, time, magnetic, k):
        out = list(J)
        for q, v in enumerate(self.source.sheet(time, magnetic)):
            if v is not None:
                add = torch.zeros(self.shape, dtype=torch.float64, device=_dev())
                add[:, :, k] = v
                out[q] = out[q] + add
        return out

    def boxes(self, S):
        """E and B over the storage box, x fastest."""
        open_z = self.mE is not None
        return {n: _box(S[q], open_z) for q, n in enumerate(FIELDS)}

    def energy(self, S):
        tot = 0.0
        for v in S[:6]:
            v = v[:, :, 1:-1] if self.mE is not None else v
            tot += float((v * v).sum())
        return tot * DX ** 3


def _box(v, open_z=False):
    v = torch.cat([v[-1:], v, v[:1]], 0)
    v = torch.cat([v[:, -1:], v, v[:, :1]], 1)
    if not open_z:
        v = torch.cat([v[:, :, -1:], v, v[:, :, :1]], 2)
    return v.permute(2, 1, 0).contiguous()


def _simple_exact(case, seed):
    f = {n: _t(a) for n, a in _state_fields(case, seed).items()}
    E, B = [f[n] for n in FIELDS[:3]], [f[n] for n in FIELDS[3:]]
    P = [[torch.zeros_like(E[0]) for _ in range(3)] for _ in range(3)]
    Pp = [[torch.zeros_like(E[0]) for _ in range(3)] for _ in range(3)]
    kind = case["solver"]

    def curl(F, shift):
        def diff(q, d):
            g = torch.roll(F[q], shift, d)
            return (F[q] - g if shift > 0 else g - F[q]) / DX
        return [diff(2, 1) - diff(1, 2), diff(0, 2) - diff(2, 0), diff(1, 0) - diff(0, 1)]

    for _ in range(case["steps"]):
        c = curl(B, 1)
        if kind == "plain":
            E = [E[q] + DT * c[q] for q in range(3)]
        elif kind == "nl":
            e2 = E[0] ** 2 + E[1] ** 2 + E[2] ** 2
            D = [(1.2 + 0.05 * e2) * E[q] + DT * c[q] for q in range(3)]
            d2 = D[0] ** 2 + D[1] ** 2 + D[2] ** 2
            s = torch.full_like(d2, 1 / 1.2)  # E = s D: 0.05 |D|^2 s^3 + 1.2 s = 1
            for _ in range(12):
                s = s - (0.05 * d2 * s ** 3 + 1.2 * s - 1) / (0.15 * d2 * s * s + 1.2)
            E = [s * v for v in D]
        else:
            for q in range(3):
                tot = old = 0.0
                for n in range(3):
                    a = DT * DT * (0.5 + n)
                    new = (2 - a) * P[n][q] - Pp[n][q] + a * 0.2 * (n + 1) * E[q]
                    tot, old, Pp[n][q], P[n][q] = tot + new, old + P[n][q], P[n][q], new
                E[q] = E[q] + old - tot + DT * c[q]
        c = curl(E, -1)
        B = [B[q] - DT * c[q] for q in range(3)]
    return {n: _box(v) for n, v in zip(FIELDS, E + B)}


def _adjoint_exact(case, seed):
    from torch.utils.checkpoint import checkpoint

    grid = _grid(case)
    p = _numbers(case, seed, 6, grid)
    eps = _t(_eps_cells(case, seed)).requires_grad_(True)
    chi = torch.tensor(p["chi"], dtype=torch.float64, device=_dev(), requires_grad=True)
    plane, part = p["d_src"] + 6, 5

    def some(t0, n, eps, chi, *S):
        y = _Yee(case, p, grid, POLES[case["poles"]], 6, eps, chi)
        y.source = first.source
        J = 0.0
        for t in range(t0, t0 + n):
            S = y.step(S, t)
            J = J + sum((S[q][:, :, plane - 1] ** 2).sum() for q in range(3))
        return (J,) + tuple(S)

    first = _Yee(case, p, grid, POLES[case["poles"]], 6)
    S, J = first.zero(), 0.0
    for t in range(0, case["steps"], part):
        n = min(part, case["steps"] - t)
        got = checkpoint(some, p["start"] + t, n, eps, chi, *S, use_reentrant=False)
        J, S = J + got[0], got[1:]
    J = J * (DX * DX * DT)
    J.backward()
    full = np.pad(eps.grad.cpu().numpy(), 1)
    return {"J": float(J), "dJ_deps": full, "dJ_dchi": float(chi.grad) if chi.grad is not None else 0.0}


def exact(case, seed):
    kind = case["kind"]
    if kind == "state":
        return _simple_exact(case, seed)
    if kind == "adjoint":
        return _adjoint_exact(case, seed)
    with torch.no_grad():
        if kind == "batch":
            out = []
            for sub, grid, p in _batch_runs(case, seed):
                y = _Yee(sub, p, grid, POLES[1], 6)
                S = y.zero()
                for t in range(case["steps"]):
                    S = y.step(S, t)
                out.append(y.boxes(S))
            return out
        if kind == "setup":
            sub = {"solver": "nonlin"}
            y = _Yee(sub, _setup_numbers(case, seed), _grid(case), POLES[1], 6)
            S = y.zero()
            for t in range(case["steps"]):
                S = y.step(S, t)
            return {n: np.ascontiguousarray(v.cpu().numpy().transpose(2, 1, 0)) for n, v in y.boxes(S).items()}
        grid = _grid(case)
        if grid[0] * grid[1] * grid[2] > 40_000_000:
            return None
        p = _numbers(case, seed, case["cpml"], grid)
        y = _Yee(case, p, grid, POLES[case["poles"]], case["cpml"])
        S = y.zero()
        for t in range(case["warm"]):
            S = y.step(S, p["start"] + t)
        out = {}
        n = case["energies"]
        calls = case["steps"] // case["a_call"]
        if n:
            part = case["steps"] // n if calls < n else calls // n * case["a_call"]
        done = part * n if n and calls < n else calls * case["a_call"]
        for t in range(done):
            S = y.step(S, p["start"] + case["warm"] + t)
            if n and (t + 1) % part == 0:
                out.setdefault("energy", []).append(y.energy(S))
        b = y.boxes(S)
        out.update({q: b[q] for q in _names(case)})
        return out
