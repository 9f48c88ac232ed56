"""Host-only test of a single contraction's plan: tests/single_plan_check.cpp."""
import pytest

from host_check import run_check


@pytest.mark.parametrize("pinned", [None, 0, 5, 18])
def test_single_plan(tmp_path, monkeypatch, pinned):
    if pinned is None:
        monkeypatch.delenv("SIPGPU_GEMM_CONFIG", raising=False)
        run_check(tmp_path, "single_plan_check.cpp")
    else:
        monkeypatch.setenv("SIPGPU_GEMM_CONFIG", str(pinned))
        run_check(tmp_path, "single_plan_check.cpp", str(pinned))
