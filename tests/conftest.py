import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
TESTS = os.path.dirname(os.path.abspath(__file__))
if TESTS not in sys.path:
    sys.path.insert(0, TESTS)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")
    config.addinivalue_line("markers", "slow: long CPU run")


def pytest_collection_modifyitems(config, items):
    # a GPU test that cannot reach a GPU must fail loudly, never fall back
    pass


@pytest.fixture(scope="session")
def ora():
    import oracle_bind
    return oracle_bind.load()


@pytest.fixture(params=["one launch", "launch per step"])
def route(request, monkeypatch):
    """Both routes of a time loop that fits the chip: the launch that takes all
    steps, and (for every handle the test makes) a launch per step."""
    if request.param == "one launch":
        return
    from hyperelasticsolver_amd.adjoint import Adjoint, BatchAdjoint
    from hyperelasticsolver_amd.batched import Batch
    from hyperelasticsolver_amd.solver import Solver

    def per_step(init):
        def make(self, *args, **kw):
            init(self, *args, **kw)
            assert self.team(-1) == 0
        return make

    for kind in (Solver, Batch, Adjoint, BatchAdjoint):
        monkeypatch.setattr(kind, "__init__", per_step(kind.__init__))
