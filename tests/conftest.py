import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP library)")


@pytest.fixture(scope="session")
def oracle():
    from oracle import oracle_py
    oracle_py.lib()
    return oracle_py


@pytest.fixture(scope="session")
def engine():
    import cltem_amd
    e = cltem_amd.Engine(0)
    yield e
    e.close()


@pytest.fixture(autouse=True)
def kernels_by_rule(request):
    """Each test finds the session's engine with no kernel variant forced or tuned by another."""
    yield
    if "engine" in request.fixturenames:
        e = request.getfixturevalue("engine")
        for kernel in (0, 1):
            e.set_kernel_variant(kernel, -1)
