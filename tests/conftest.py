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


# Tests about layers that lutgemm_mx_kernel runs out of pre-expanded rows: the planner may have it make its rows itself
# there, which tests/test_gpu_matrix_rows.py is about.
PRE_EXPANDED_ROWS = ("test_gpu_matrix_sums", "test_strided_pixel_groups_stay_in_the_workspace",
                     "test_matrix_core_kernel_where_it_was_measured_faster")


@pytest.fixture(autouse=True)
def _pre_expanded_rows(request):
    if request.module.__name__ not in PRE_EXPANDED_ROWS and request.function.__name__ not in PRE_EXPANDED_ROWS:
        yield
        return
    ops = entry.load_package().ops
    ops.set_matrix_rows(1)
    try:
        yield
    finally:
        ops.set_matrix_rows(0)
