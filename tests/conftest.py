"""Test configuration: the ``gpu`` marker and import paths.

``-m "not gpu"`` runs on any host (oracle, golden fixtures, ROM generator, the
C ABI's exports); ``-m gpu`` needs an MI355X and the built native libraries.
"""

import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))


@pytest.fixture(params=["chosen", "lanes"])
def step_kernel(request, monkeypatch):
    """Runs a test's plain steps twice: by the kernel the library chooses (one
    console per wave up to 32,768 consoles) and by the lane kernel, which the
    library falls back to."""
    if request.param == "lanes":
        from nesle_amd import abi

        create = abi.Batch.__init__

        def create_in_lanes(self, *args, **kwargs):
            create(self, *args, **kwargs)
            self.set_lane_kernel(True)

        monkeypatch.setattr(abi.Batch, "__init__", create_in_lanes)
    return request.param


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a GPU (MI355X) and the built HIP library")
