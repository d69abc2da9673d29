import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

GOLDEN = os.path.join(ROOT, "tests", "golden")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and the built libbtrc_hip.so")


@pytest.fixture(scope="session")
def _session_ctx():
    import btrc_amd
    c = btrc_amd.Context(0)
    c.default_tuning = c.get_tuning()
    yield c
    c.close()


@pytest.fixture
def ctx(_session_ctx):
    """one context for the whole session; every test starts from the box
    filter, a fresh context's tuning and the cache switched off"""
    c = _session_ctx
    c.set_filter("box")
    c.set_tuning(**c.default_tuning)
    c.nrc_configure(enabled=0, train_depth=0)
    yield c


@pytest.fixture(scope="session")
def golden():
    return GOLDEN
