import os
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if REPO not in sys.path:
    sys.path.insert(0, REPO)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP) GPU and the built libfsk_decode.so")


def pytest_collection_modifyitems(config, items):
    import torch
    if torch.cuda.is_available():
        return
    skip = pytest.mark.skip(reason="no HIP GPU in this environment")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


@pytest.fixture(params=["direct", "split"])
def both_routes(request):
    """Calls of short sequences as they are routed, on the direct kernel, and
    again with every call on the split kernels."""
    from fasterkernels_amd import native as nat
    nat.set_option("direct", int(request.param == "direct"))
    yield
    nat.set_option("direct", 1)
