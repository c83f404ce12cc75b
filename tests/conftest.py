import os
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an AMD GPU (MI355X) and the built HIP library")
    config.addinivalue_line("markers", "slow: long-running parity case")


def gpu_available() -> bool:
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:
        return False


@pytest.fixture(scope="session")
def hip():
    """The suite library, initialised on device 0 (GPU tests only)."""
    if not gpu_available():
        pytest.skip("no GPU")
    from tealeaf_amd.abi import lib
    L = lib()
    L.tlhip_init(0)
    return L


@pytest.fixture(scope="session")
def oracle():
    from oracle.pyoracle import load_oracle
    return load_oracle()


@pytest.fixture(params=["chip", "launches"])
def loops(request, monkeypatch):
    """Driver tests on small grids run both ways that the loops have: on the
    chip, where such grids run by default, and launch by launch, as larger
    grids run."""
    if request.param == "launches":
        from tealeaf_amd.problem import Problem
        init = Problem.__init__

        def launches(self, *args, **kw):
            init(self, *args, **kw)
            self.set_on_chip(False)

        monkeypatch.setattr(Problem, "__init__", launches)
    return request.param
