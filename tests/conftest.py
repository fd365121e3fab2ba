import gc
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def scalar_oracle():
    from oracle import scalar
    scalar.build()
    return scalar


@pytest.fixture(autouse=True)
def _no_garbage_of_earlier_tests(request):
    """Tests that compare the allocator's counters around a call begin without reference cycles of earlier tests, whose tensors the
    collector may free in between."""
    if "no_alloc" in request.node.nodeid:
        gc.collect()
