import os
import sys

import pytest

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))
PKG = os.path.join(ROOT, "rhmc-on-gpu_amd")
for p in (PKG, os.path.join(ROOT, "oracle"), os.path.join(ROOT, "tests")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through the HIP C ABI)")
    config.addinivalue_line("markers", "slow: longer CPU test")


def pytest_collection_modifyitems(items):
    # the tests that compile the reference's sources look for its directory, which may be empty
    import build_ref
    if not build_ref.have_reference():
        skip = pytest.mark.skip(reason="reference sources not present")
        for item in items:
            if item.name == "test_reference_links_against_library":
                item.add_marker(skip)
