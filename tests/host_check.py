"""Compiles a host-only C++ check against the built library and runs it."""
import os
import subprocess

from aces4_amd import sipgpu as sg

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def run_check(tmp_path, source, *args):
    exe = str(tmp_path / source.replace(".cpp", ""))
    cmd = [HIPCC, "-O1", "-std=c++17", "-I", os.path.join(HERE, "..", "aces4_amd", "csrc"), "-x",
           "hip", os.path.join(HERE, source), "-x", "none", sg.LIB_PATH, "-o", exe,
           "-Wl,-rpath," + os.path.dirname(sg.LIB_PATH)]
    subprocess.run(cmd, check=True, capture_output=True, timeout=300)
    r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "all ok" in r.stdout, r.stdout + r.stderr
    return r.stdout
