import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

import __graft_entry__ as entry  # noqa: E402


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def pkg():
    return entry.load_package()


@pytest.fixture(scope="session")
def oracle():
    return entry.load_oracle()


@pytest.fixture(scope="session")
def golden_dir():
    return os.path.join(ROOT, "tests", "golden")


@pytest.fixture(params=["as_planned", "part_by_part"])
def launches(request, pkg):
    """A test twice: as the planner has it, which runs most layers of a test's size in one launch; and without launches that do
    the work of several, so that they run the pre-pass and the lookup kernels of large layers."""
    if request.param == "part_by_part":
        pkg.ops.set_merged_launches(-1)
    try:
        assert (pkg.ops.conv2d_direct_plan((1, 32, 32, 16), (3, 3, 16, 32)) is None) == (request.param == "part_by_part")
        yield request.param
    finally:
        pkg.ops.set_merged_launches(0)
