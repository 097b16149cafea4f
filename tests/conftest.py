import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TESTS = os.path.dirname(os.path.abspath(__file__))
for p in (ROOT, TESTS):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through the C ABI on device 0)")


def pytest_collection_modifyitems(config, items):
    # The drop-in drivers hold the reference's own main.cpp: without its sources
    # build() leaves them out, and their tests cannot run.  Where the sources are,
    # a missing driver stays a failure.
    from __graft_entry__ import REFERENCE_SOURCE

    drivers = os.path.join(ROOT, "capaz_amd", "adapter", "_bin")
    if os.path.isfile(REFERENCE_SOURCE):
        return
    for item in items:
        if item.path.name == "test_dropin.py":
            model = item.callspec.params["model"]
            if not os.path.exists(os.path.join(drivers, f"capaz_dropin_{model}")):
                item.add_marker(pytest.mark.skip(reason="the drop-in driver is built from the reference's sources, "
                                                        "which are not here"))


@pytest.fixture(autouse=True)
def _announce(request):
    if request.node.get_closest_marker("gpu"):
        print(f"\n[case] {request.node.nodeid}", flush=True)
    yield
