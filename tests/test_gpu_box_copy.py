"""Reads and writes of grids (GPU): what is set comes back as the storage form holds it, over the
whole storage box, in every precision, for fields and accumulator parts, and a periodic
dimension's ghosts read as the periodic images whether or not a step was taken."""
import numpy as np
import pytest

from mpulse_amd import abi, configs

pytestmark = pytest.mark.gpu


def images(a, periodic):
    a = a.copy()
    for d, per in enumerate(periodic):
        if per:
            m = np.moveaxis(a, d, 0)
            m[0], m[-1] = m[-2], m[1]
    return a


@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_FP32_BULK, abi.PREC_FP32_RES])
@pytest.mark.parametrize("boundary", [abi.BOUNDARY_PERIODIC, abi.BOUNDARY_XY_PERIODIC])
@pytest.mark.parametrize("grid", [(9, 7, 63), (8, 12, 64), (200, 33, 1300)])  # the last in several slabs
def test_set_get_fetch(prec, boundary, grid):
    print(f"case: set/get precision {prec} boundary {boundary} grid {grid}", flush=True)
    d, _ = configs.plrc_kerr_pulse(grid[0], 2, 5.0, 4, 1e9, 0, d_src=4, nz=grid[2], precision=prec, boundary=boundary)
    d.ny = grid[1]
    rng = np.random.default_rng(3)
    form = {abi.PREC_FP64: lambda x: x, abi.PREC_FP32_BULK: lambda x: x.astype(np.float32).astype(np.float64)}.get(prec)
    with abi.Solver(d) as s:
        periodic = (True, True, boundary == abi.BOUNDARY_PERIODIC)
        for n in ("Ex", "Ez", "By"):  # several slots of one residual word
            a = rng.standard_normal(s.shape) * 10.0 ** rng.integers(-6, 3, s.shape)
            s.set(n, a)
            got = s.get(n)
            if form is not None:
                assert np.array_equal(got, images(form(a), periodic)), n
            else:
                assert np.abs(got / images(a, periodic) - 1).max() < 2.0 ** -33, n
                some = [tuple(rng.integers(1, e - 1) for e in s.shape) for _ in range(50)]
                assert all(got[c] == abi.store_round(a[c], prec) for c in some), n
            assert np.array_equal(s.fetch(n).transpose(2, 1, 0), got), n
        for n in ("PsiR1x", "PsiI1z"):  # accumulators: float64 in every form, as stored
            a = rng.standard_normal(s.shape)
            s.set(n, a)
            assert np.array_equal(s.get(n), a), n
