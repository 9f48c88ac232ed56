"""Host-only test of the split path's plans: tests/split_plan_check.cpp."""
from host_check import run_check


def test_split_plan_lists(tmp_path):
    print(run_check(tmp_path, "split_plan_check.cpp"))
