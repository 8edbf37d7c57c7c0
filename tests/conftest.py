import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
for sub in ("oracle", "tests"):
    p = os.path.join(ROOT, sub)
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device) and the built libgpupi.so")
    config.addinivalue_line("markers", "slow: larger sizes")


@pytest.fixture(scope="session")
def oracle():
    import oracle_ffi
    oracle_ffi.lib()
    return oracle_ffi


@pytest.fixture(scope="session")
def shared_context():
    import gpupi_amd
    c = gpupi_amd.Context()
    yield c
    c.close()


@pytest.fixture
def ctx(shared_context):
    """The session's context, with the crossover that a fresh one has (tests
    that move it leave it somewhere else)."""
    import gpupi_amd
    from helpers import DEFAULT_NTT_MIN_LIMBS
    gpupi_amd.check(shared_context.set_ntt_threshold(DEFAULT_NTT_MIN_LIMBS), "set_ntt_threshold")
    return shared_context
