"""The pass path on an open z (single_xy_periodic), where it takes a step as the two fused halves or as
one kernel: the fused path's bits, ghosts of z included, with z ghosts set mid-run while a B half is
owed, and in runs that a tuning call moves between the routes."""
import numpy as np
import pytest

from mpulse_amd import abi, configs

pytestmark = pytest.mark.gpu

FIELDS = ("Ex", "Ey", "Bx", "Bz", "PsiR1y")
# (grid, precision, layers, poles): both sides of the rule's lines -- with layers, no poles, at 3 * 2^21 cells;
# with layers and a pole at 2^24 cells and at whole z tiles; layers along z alone (negative); without layers at 2^22 cells, by poles and whole z tiles
CASES = [((66, 61, 70), abi.PREC_FP64, 4, 1), ((49, 64, 65), abi.PREC_FP32_RES, 3, 1), ((66, 64, 64), abi.PREC_FP32_BULK, 4, 1),
         ((30, 29, 65), abi.PREC_FP64, 4, 0), ((182, 185, 187), abi.PREC_FP64, 4, 0), ((170, 171, 173), abi.PREC_FP64, 4, 0),
         ((256, 256, 256), abi.PREC_FP64, 5, 1), ((255, 256, 256), abi.PREC_FP64, 5, 1),
         ((162, 161, 163), abi.PREC_FP32_BULK, 0, 1), ((162, 161, 163), abi.PREC_FP32_RES, 0, 0),
         ((96, 64, 64), abi.PREC_FP64, -4, 1), ((96, 64, 65), abi.PREC_FP64, -4, 1), ((60, 50, 40), abi.PREC_FP64, -4, 0),
         ((128, 129, 128), abi.PREC_FP32_BULK, -4, 0), ((127, 128, 128), abi.PREC_FP32_RES, -4, 0),
         ((152, 152, 192), abi.PREC_FP32_RES, 0, 1), ((152, 152, 190), abi.PREC_FP32_RES, 0, 1)]


def make(grid, prec, layers, poles, path):
    d, _ = configs.plrc_kerr_pulse(64, max(abs(layers), 3), 5.0, 4, 3e9, 0, d_src=8, nz=grid[2], precision=prec, path=path,
                                   boundary=abi.BOUNDARY_XY_PERIODIC, poles=((1.1, 4.0, 0.005),) * poles)
    d.nx, d.ny = grid[:2]
    d.factories[1].tshift = 3.0
    if layers < 0:
        d.factories[0].kind = abi.FACTORY_CPML_1D
    if not layers:
        d.factories[0] = abi.Factory.from_buffer_copy(d.factories[1])
        d.n_factories = 1
    return d


def run(grid, prec, layers, poles, path, switch):
    rng = np.random.default_rng(11)
    out = []
    with abi.Solver(make(grid, prec, layers, poles, path)) as s:
        for q, steps in enumerate((1, 7, 6, 3)):
            s.step(steps)
            if q == 1 and switch:
                s.tune(*switch)  # a B half is owed here
            if q == 2:  # fields with ghosts of their own at both ends of z
                for n in ("Ey", "Bx"):
                    f = s.get(n)
                    for k in (0, -1):
                        f[1:-1, 1:-1, k] += rng.uniform(-1e-3, 1e-3, f[1:-1, 1:-1, k].shape)
                    s.set(n, f)
            if q != 1:
                out.append({n: s.get(n)[1:-1, 1:-1] for n in FIELDS})
    return out


@pytest.mark.parametrize("grid,prec,layers,poles", CASES)
def test_same_bits(grid, prec, layers, poles):
    print(f"case: pass route, open z, {grid} precision {prec} layers {layers} poles {poles}", flush=True)
    want = run(grid, prec, layers, poles, abi.PATH_FUSED, None)
    assert np.linalg.norm(want[-1]["Ey"]) > 0 and np.linalg.norm(want[-1]["Bx"][:, :, 0]) > 0
    for switch in (None, ("march_seg", 5), ("pass_kernel", 1)):
        got = run(grid, prec, layers, poles, abi.PATH_PASS, switch)
        for w, g in zip(want, got):
            for n in FIELDS:
                assert np.array_equal(w[n], g[n]), (switch, n)
