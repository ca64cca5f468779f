"""A batch whose structure changes between calls: every structure reads the field, accumulator and
layer sets that the one before it left, after odd and even numbers of steps."""
import numpy as np
import pytest

from mpulse_amd import abi, configs
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

FIELDS = ("Ex", "Ey", "Ez", "Bx", "By", "Bz")
ORDER = ((1, 3), (0, 5), (2, 5), (1, 1), (2, 2), (0, 1))  # (structure, steps)


def runs(prec):
    out = []
    for nx, ny, nz in ((21, 26, 33), (30, 19, 70)):
        d, _ = configs.plrc_kerr_pulse(nx, 4, 6.0, 5, 3e9, 0, d_src=7, precision=prec, path=abi.PATH_SWEEP, nz=nz)
        d.ny = ny
        out.append(d)
    return out


def start(d, seed):
    """E and B over the storage box, ghosts the periodic images, so that all layers work at once"""
    rng = np.random.default_rng(seed)
    return {n: np.pad(rng.uniform(-1e-2, 1e-2, (d.nx, d.ny, d.nz)).astype(np.float32).astype(np.float64), 1, mode="wrap")
            for n in FIELDS}


# float64: the order of the sums; float32: 17 steps of two roundings of 2^-24 (2e-6), five times that
@pytest.mark.parametrize("prec,bound", [(abi.PREC_FP64, 1e-12), (abi.PREC_FP32_BULK, 1e-5)])
def test_structure_changes_in_a_running_batch(prec, bound):
    print(f"case: batch structure changes, precision {prec}", flush=True)
    descs = runs(prec)
    for _ in range(3):  # leave the allocator's free blocks out of order
        with abi.Solver(descs[1]), abi.Solver(descs[0]):
            pass
    with abi.Batch(descs) as b:
        for r, d in enumerate(descs):
            for n, f in start(d, r).items():
                b.run(r).set(n, f)
        for structure, steps in ORDER:
            b.tune("structure", structure)
            b.step(steps)
        b.sync()
        for r, d in enumerate(descs):
            o = Oracle(d)
            for n, f in start(d, r).items():
                o.set(n, f)
            o.step(sum(s for _, s in ORDER))
            v = b.run(r)
            for group in (FIELDS[:3], FIELDS[3:]):
                w = np.concatenate([o.get(n).ravel() for n in group])
                g = np.concatenate([v.get(n).ravel() for n in group])
                assert np.linalg.norm(g - w) <= bound * np.linalg.norm(w), (r, group)
            for side in "EB":
                for direction in range(6):
                    for c in "xyz":
                        name = f"CPMLPsi{side}{c}"
                        inner = (slice(1, -1), slice(1, -1), slice(1, -1))  # these paths leave a layer's ghosts at zero
                        w, g = o.get_layer(name, direction)[0][inner], v.get_layer(name, direction)[0][inner]
                        assert np.linalg.norm(g - w) <= bound * np.linalg.norm(w), (r, name, direction)
            o.close()
