"""The pass path's tests once more with every step in the one kernel, whatever the size: the route that the
solver chooses by itself takes small runs with layers as the two fused halves."""
import pytest

from mpulse_amd import abi
from test_gpu_cpml_layers import test_against_oracle, test_shapes_agree  # noqa: F401
from test_gpu_pass import *  # noqa: F401,F403

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def one_kernel(monkeypatch):
    create = abi.Solver.__init__

    def init(self, desc):
        create(self, desc)
        if desc.path == abi.PATH_PASS:
            self.tune("pass_kernel", 1)

    monkeypatch.setattr(abi.Solver, "__init__", init)
