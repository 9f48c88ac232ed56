"""Host-only test of the table planner's choice of tiles: tests/tile_choice_check.cpp."""
from host_check import run_check


def test_tile_choice(tmp_path):
    run_check(tmp_path, "tile_choice_check.cpp")
