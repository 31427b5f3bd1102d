import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through libehip's C ABI)")


def launched_only(system):
    """Keeps a system's solves off the resident loops, which take most systems
    of at most 262 144 rows, for tests of the launched and recorded ones."""
    import ctypes as C
    from elmerfem_amd import _lib
    assert _lib.load().ehip_internal_resident(system._h, C.c_int(1)) == 0


@pytest.fixture(scope="session")
def ehip():
    """libehip initialised on device 0.  GPU tests fail (not skip) when the
    library or the device is missing: they run only where a GPU is."""
    from elmerfem_amd import _lib
    return _lib.init(0)
