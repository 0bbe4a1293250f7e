import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through the HIP C-ABI library)")


@pytest.fixture(scope="session")
def pkg():
    import __graft_entry__
    return __graft_entry__.load_package()


@pytest.fixture(scope="session")
def O():
    from oracle import oracle
    return oracle


@pytest.fixture(scope="session")
def gpu(pkg):
    pkg.native.init(0)
    return pkg


@pytest.fixture
def launched(gpu):
    """launched(f): f()'s result and the names of the kernels that this thread launched meanwhile."""
    import ctypes
    lib = gpu.native.lib()
    names = lib._ZN2cj12launch_namesEv
    names.restype = ctypes.c_char_p

    def record(f):
        lib._ZN2cj18launch_names_resetEv()
        try:
            out = f()
        finally:
            seen = names().decode().split(" + ")
        return out, seen

    return record
