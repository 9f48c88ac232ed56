"""Host-only test of the boxes of (T) sums: tests/triples_boxes_check.cpp."""
from host_check import run_check


def test_boxes(tmp_path):
    run_check(tmp_path, "triples_boxes_check.cpp")
