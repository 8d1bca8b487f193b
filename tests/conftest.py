import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X; run through the C ABI on the device")


def pytest_collection_modifyitems(items):
    """The reference's own programs are built from its source tree; where that tree is absent and nothing was built
    from it beforehand, the tests that run them have nothing to run."""
    suite = os.path.join(ROOT, "tests", "reference_programs", "build", "suite")
    tree = os.environ.get("TIRAMISU_REFERENCE_TREE", "/root/reference")
    if os.path.isdir(suite) or os.path.isdir(os.path.join(tree, "tests")):
        return
    for item in items:
        if item.path.name == "test_reference_suite.py":
            item.add_marker(pytest.mark.skip(reason="no reference tree at %s, and nothing built from one" % tree))


@pytest.fixture(scope="session")
def programs_dir():
    return os.path.join(ROOT, "tests", "programs")


@pytest.fixture(scope="session")
def product_programs_dir():
    return os.path.join(ROOT, "tiramisu_amd", "programs")
