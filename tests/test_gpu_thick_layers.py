"""CPML layers thicker than the box on the reference-structured path and in stepSchemeInit: the layer
kernels stay inside the grid, and E and B agree with the fused path, which visits interior cells only."""
import numpy as np
import pytest

from mpulse_amd import abi, configs

pytestmark = pytest.mark.gpu

FIELDS = ("Ex", "Ey", "Ez", "Bx", "By", "Bz")


@pytest.mark.parametrize("init", [False, True])
@pytest.mark.parametrize("boundary", [abi.BOUNDARY_PERIODIC, abi.BOUNDARY_XY_PERIODIC])
@pytest.mark.parametrize("grid,d_cpml", [((39, 2, 66), 4), ((3, 5, 40), 6), ((20, 17, 3), 5), ((1, 1, 9), 7)])
def test_reference_path_agrees_with_the_fused(grid, d_cpml, boundary, init):
    print(f"case: layers of {d_cpml} in {grid} boundary {boundary} init {init}", flush=True)
    got = []
    for path in (abi.PATH_FUSED, abi.PATH_REFERENCE):
        d, _ = configs.plrc_kerr_pulse(grid[0], d_cpml, 5.0, 4, 3e9, 0, d_src=min(8, max(2, grid[2] // 2)), nz=grid[2],
                                       path=path, boundary=boundary)
        d.ny = grid[1]
        rng = np.random.default_rng(3)
        with abi.Solver(d) as s:
            for n in FIELDS:
                s.set(n, np.pad(rng.uniform(-0.1, 0.1, grid), 1, mode="wrap"))
            if init:
                s.step_init()
            s.step(20)
            got.append({n: s.get(n)[1:-1, 1:-1, 1:-1] for n in FIELDS})
    for n in FIELDS:
        assert np.linalg.norm(got[1][n] - got[0][n]) <= 1e-12 * np.linalg.norm(got[0][n]), n
