import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for sub in ("", "oracle", "tests", "thirring-rhmc_amd"):
    p = os.path.join(ROOT, sub)
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and the built HIP library")
    config.addinivalue_line("markers", "slow: longer CPU test")


@pytest.fixture(autouse=True)
def _default_dslash_shapes(request):
    """A GPU test that pins Dslash shapes leaves none of them to the next."""
    yield
    G = sys.modules.get("thirring_hip")
    if request.node.get_closest_marker("gpu") and G is not None and G._lib is not None:
        G.dslash_clear_config()
