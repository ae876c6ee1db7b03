import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")


@pytest.fixture(autouse=True)
def _tiles_by_size():
    """Every test starts from the tiles that a program gets without setting any,
    whatever the tests before it set."""
    from qtnh_amd import ops
    ops.tune_circuit()
