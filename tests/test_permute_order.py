"""Host-only test of the permutes' tile order: tests/permute_order_check.cpp."""
from host_check import run_check


def test_permute_order(tmp_path):
    run_check(tmp_path, "permute_order_check.cpp")
