"""CPML layers where their handling can go wrong (GPU): layers that meet or overlap in a short
dimension (a cell then belongs to both faces of it), layers that end inside a 64-cell z tile, on
its edge or one past it, every row of a tile in a layer, one dimension's faces only -- float64
against the oracle (1e-12), the float32 forms and the pass path against the fused float64 /
fused path bit for bit where they must agree."""
import numpy as np
import pytest

from mpulse_amd import abi, configs
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

FIELDS = ("Ex", "Ey", "Ez", "Bx", "By", "Bz", "PsiR1x")
GRIDS = [((11, 9, 64), 6), ((9, 12, 65), 5), ((40, 16, 13), 7), ((13, 70, 130), 3), ((20, 21, 192), 10)]


def make(grid, d_cpml, prec, path, one_d=False):
    d, _ = configs.plrc_kerr_pulse(64, d_cpml, 5.0, 4, 3e9, 0, d_src=min(8, grid[2] // 2), nz=grid[2],
                                   precision=prec, path=path)
    d.nx, d.ny = grid[:2]
    d.factories[1].tshift = 6.0
    if one_d:
        d.factories[0].kind = abi.FACTORY_CPML_1D
    return d


@pytest.mark.parametrize("path", [abi.PATH_FUSED, abi.PATH_PASS])
@pytest.mark.parametrize("one_d", [False, True])
@pytest.mark.parametrize("grid,d_cpml", GRIDS)
def test_against_oracle(grid, d_cpml, one_d, path):
    print(f"case: layers of {d_cpml} in {grid} one_d {one_d} path {path}", flush=True)
    d = make(grid, d_cpml, abi.PREC_FP64, path, one_d)
    o = Oracle(d)
    with abi.Solver(d) as s:
        for steps in (40, 31):
            s.step(steps)
            o.step(steps)
            for n in FIELDS:
                got, ref = s.get(n), o.get(n)
                assert np.linalg.norm(ref) > 0, n
                assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(ref), n
        for name, face in (("CPMLPsiEx", abi.UP), ("CPMLPsiBy", abi.DOWN)):
            got, ref = s.get_layer(name, face)[0], o.get_layer(name, face)[0]
            inner = (slice(1, -1), slice(1, -1), slice(1, -1))  # a fused path's layer ghosts stay at zero
            assert np.linalg.norm((got - ref)[inner]) <= 1e-12 * np.linalg.norm(ref), name
    o.close()


@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_FP32_BULK, abi.PREC_FP32_RES])
@pytest.mark.parametrize("grid,d_cpml", GRIDS)
def test_shapes_agree(grid, d_cpml, prec):
    """One and several planes per thread, block orders and the pass path: the same bits."""
    print(f"case: layers of {d_cpml} in {grid} precision {prec}", flush=True)
    ref = None
    shapes = [(abi.PATH_FUSED, {}), (abi.PATH_FUSED, {"march_b": 2}), (abi.PATH_FUSED, {"march_b": 4, "march_e": 2}),
              (abi.PATH_FUSED, {"tile_order": 0}), (abi.PATH_FUSED, {"tile_order": 1, "tile_band": 3}),
              (abi.PATH_FUSED, {"tile_band": 2, "b_reverse": 0}), (abi.PATH_PASS, {}),
              (abi.PATH_PASS, {"march_rows": 3, "march_seg": 4}), (abi.PATH_PASS, {"march_rows": 7, "march_seg": 3})]
    for path, tuning in shapes:
        with abi.Solver(make(grid, d_cpml, prec, path)) as s:
            for k, v in tuning.items():
                s.tune(k, v)
            s.step(45)
            got = {n: s.get(n) for n in FIELDS}
        if ref is None:
            ref = got
        for n in FIELDS:
            assert np.array_equal(got[n], ref[n]), (path, tuning, n)
