"""Source sheets of many steps from one launch (GPU): the layers and the fields after one call
for many steps equal those of one call per step bit for bit -- windows of the slots a solver
keeps, a last window that is shorter -- and the layers equal the oracle's, so the mirrored
quarter of the short pulse is checked on even and odd cross-sections."""
import numpy as np
import pytest

from mpulse_amd import abi, configs
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

FIELDS = ("Ex", "Ey", "Ez", "Bx", "By", "Bz")
LAYERS = ("IncidentEJx", "IncidentEJy", "IncidentHJx", "IncidentHJy")


def sources(nx, ny, path, kind):
    d, _ = configs.plrc_kerr_pulse(nx, 4, 6.0, 4, 2e9, 0, d_src=7, nz=20, path=path)
    d.ny = ny
    d.factories[1].tshift = 5.0
    if kind != "pulse":
        f = abi.factory_defaults(abi.FACTORY_PLANE_WAVE)
        f.d = 7 if kind == "shared" else 9  # the pulse's plane (the later source's values stand) or its own
        f.h[0], f.h[1] = 0.3, 1.0
        f.k[0], f.k[2] = 0.2, 1.1
        abi.add_factory(d, f)
    return d


@pytest.mark.parametrize("path", [abi.PATH_FUSED, abi.PATH_PASS])
@pytest.mark.parametrize("nx,ny,kind", [(14, 17, "pulse"), (15, 16, "pulse"), (12, 13, "two"), (13, 12, "shared")])
def test_many_steps_a_call(path, nx, ny, kind):
    steps = 75  # more than two full windows of at most 32 steps
    print(f"case: sheets {nx}x{ny} {kind} path {path}", flush=True)
    d = sources(nx, ny, path, kind)
    o = Oracle(d)
    o.step(steps)
    with abi.Solver(d) as a, abi.Solver(d) as b:
        a.step(steps)
        for _ in range(steps):
            b.step(1)
        for n in FIELDS:
            x, y = a.get(n), b.get(n)
            assert np.array_equal(x, y), n
            ref = o.get(n)
            assert np.linalg.norm(x - ref) <= 1e-12 * np.linalg.norm(ref), n
        for n in LAYERS:
            x, y, ref = a.get_layer(n, abi.DOWN)[0], b.get_layer(n, abi.DOWN)[0], o.get_layer(n, abi.DOWN)[0]
            assert np.array_equal(x, y), n
            assert np.abs(x - ref).max() <= 1e-12 * max(np.abs(ref).max(), 1e-300), n
    o.close()
