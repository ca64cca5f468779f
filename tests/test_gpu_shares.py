"""The fused kernels' block order with shares of equal work (layers present, 2048 tiles or more):
every cell once, so the bits of the plain orders, whose shares are equal tiles -- bands of one row
of tiles, of several, of all; forwards and backwards; one and two planes per thread; layers that
are thin, unequal in number by dimension, or fill the box."""
import numpy as np
import pytest

from mpulse_amd import abi, configs

pytestmark = pytest.mark.gpu

FIELDS = ("Ex", "Ey", "Ez", "Bx", "By", "Bz", "PsiR1x")
CASES = [((70, 130, 65), 3, abi.PREC_FP64), ((257, 33, 60), 10, abi.PREC_FP32_BULK),
         ((40, 211, 70), 18, abi.PREC_FP32_RES), ((9, 31, 2000), 4, abi.PREC_FP64)]


@pytest.mark.parametrize("grid,d_cpml,prec", CASES)
def test_same_bits(grid, d_cpml, prec):
    print(f"case: shares {grid} layers of {d_cpml} precision {prec}", flush=True)
    ref = None
    for tuning in ({"tile_order": 0}, {}, {"tile_band": 1}, {"tile_band": 7, "b_reverse": 0}, {"tile_band": 1000},
                   {"march_b": 2, "tile_band": 4}):
        d, _ = configs.plrc_kerr_pulse(64, d_cpml, 5.0, 4, 3e9, 0, d_src=min(d_cpml + 2, grid[2] // 2), nz=grid[2],
                                       precision=prec, path=abi.PATH_FUSED)
        d.nx, d.ny = grid[:2]
        d.factories[1].tshift = 3.0
        with abi.Solver(d) as s:
            for k, v in tuning.items():
                s.tune(k, v)
            s.step(25)
            got = {n: s.get(n) for n in FIELDS}
        if ref is None:
            ref = got
            assert np.linalg.norm(ref["Ey"]) > 0
        for n in FIELDS:
            assert np.array_equal(got[n], ref[n]), (tuning, n)
