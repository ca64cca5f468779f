"""The pass path takes a step in one kernel or as the two fused halves, by size, storage form and
layers: the fused path's bits on either side of each line of the rule, with a read in between,
and in a run that a tuning call moves from the halves to the one kernel."""
import numpy as np
import pytest

from mpulse_amd import abi, configs

pytestmark = pytest.mark.gpu

FIELDS = ("Ex", "Ey", "Ez", "Bx", "By", "Bz", "PsiR1x")
# (grid, precision, layers, plasma) on both sides of the lines at 2^18 and 3 * 2^16 cells
CASES = [((64, 64, 64), abi.PREC_FP64, 5, False), ((65, 64, 64), abi.PREC_FP64, 5, False),
         ((64, 64, 64), abi.PREC_FP32_BULK, 5, False), ((64, 65, 64), abi.PREC_FP32_BULK, 5, False),
         ((48, 64, 64), abi.PREC_FP32_RES, 5, False), ((49, 64, 64), abi.PREC_FP32_RES, 5, False),
         ((66, 61, 70), abi.PREC_FP64, 0, False), ((66, 61, 70), abi.PREC_FP32_BULK, 0, False),
         ((66, 61, 70), abi.PREC_FP64, 4, True), ((30, 31, 33), abi.PREC_FP64, 4, True)]


def make(grid, prec, layers, plasma, path):
    d, _ = configs.plrc_kerr_pulse(64, max(layers, 4), 5.0, 4, 3e9, 0, d_src=8, nz=grid[2], precision=prec, path=path)
    d.nx, d.ny = grid[:2]
    d.factories[1].tshift = 3.0
    if not layers:
        d.factories[0] = abi.Factory.from_buffer_copy(d.factories[1])
        d.n_factories = 1
    if plasma:
        c = abi.factory_defaults(abi.FACTORY_PLASMA_CURRENT)
        c.em, c.gamma, c.rho_bg = 0.8, 0.2, 0.01
        abi.add_factory(d, c)
        d.plasma, d.plasma_k, d.plasma_nu, d.plasma_mpa, d.plasma_wion = 1, 3, 1e-3, 1e-5, 0.5
    return d


@pytest.mark.parametrize("grid,prec,layers,plasma", CASES)
def test_same_bits(grid, prec, layers, plasma):
    print(f"case: pass route {grid} precision {prec} layers {layers} plasma {plasma}", flush=True)
    ref = []
    for path, tuning in ((abi.PATH_FUSED, None), (abi.PATH_PASS, None), (abi.PATH_PASS, ("march_seg", 5))):
        with abi.Solver(make(grid, prec, layers, plasma, path)) as s:
            for q, steps in enumerate((1, 20, 19, 2)):
                s.step(steps)
                if q == 1 and tuning:
                    s.tune(*tuning)  # a B half is owed here
                if q in (0, 2, 3):
                    got = {n: s.get(n) for n in FIELDS}
                    if path == abi.PATH_FUSED:
                        ref.append(got)
                    for n in FIELDS:
                        assert np.array_equal(got[n], ref[{0: 0, 2: 1, 3: 2}[q]][n]), (path, tuning, q, n)
    assert np.linalg.norm(ref[-1]["Ey"]) > 0
