"""A batched run whose accumulator block passes 4 GiB (storage cell 2^26.4 and beyond): the fused
and the x-march structure open with the batched fused E kernel, whose accumulator addresses must
hold there too -- the bits of the same run on its own."""
import numpy as np
import pytest

from mpulse_amd import abi, configs

pytestmark = pytest.mark.gpu

GRID = (9, 3000, 3000)


def make(path):
    d, _ = configs.plrc_kerr_pulse(24, 4, 5.0, 4, 3e9, 0, d_src=8, nz=GRID[2], precision=abi.PREC_FP32_BULK, path=path)
    d.nx, d.ny = GRID[:2]
    d.n_factories = 0
    return d


def fill(solver):
    n = [g + 2 for g in GRID]
    rng = np.random.default_rng(7)
    x, y, z = (rng.uniform(-1.0, 1.0, m) for m in n)
    solver.set("Ey", x[:, None, None] * y[None, :, None] * z)


@pytest.mark.parametrize("structure", [0, 2])
def test_same_bits_past_4_gib(structure):
    print(f"case: batch of one run {GRID}, structure {structure}", flush=True)
    with abi.Solver(make(abi.PATH_FUSED)) as s:
        fill(s)
        s.step(1)
        s.step(2)
        want = {n: s.get(n) for n in ("Ey", "PsiI1y")}
    assert np.linalg.norm(want["PsiI1y"][-2]) > 0
    with abi.Batch([make(abi.PATH_SWEEP)]) as b:
        b.tune("structure", structure)
        fill(b.run(0))
        b.step(1)  # the second call opens with accumulators in place
        b.step(2)
        b.sync()
        for n, w in want.items():
            assert np.array_equal(b.run(0).get(n), w), n
