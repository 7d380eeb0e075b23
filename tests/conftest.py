import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "oracle")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP library on cuda:0)")


@pytest.fixture(scope="session")
def orc():
    import oracle
    return oracle.Oracle()


# Default of the option "mlt_wave_chains" (Ctx::mlt_wave_chains).
MLT_WAVE_CHAINS = 28672


@pytest.fixture(autouse=True)
def shipped_chain_limit(request):
    """Whatever a test sets it to, the next one gets the session's context with
    the number of chains up to which a wave runs each as it is shipped."""
    yield
    if "ctx" in request.fixturenames:
        request.getfixturevalue("ctx").set_option("mlt_wave_chains", MLT_WAVE_CHAINS)


@pytest.fixture(scope="session")
def ctx():
    from barnacle_amd import native
    c = native.Context(0)
    yield c
    c.close()
