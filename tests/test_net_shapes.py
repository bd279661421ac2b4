"""Split of the network's weight gradients (csrc/net_shapes.hpp), compiled for the host."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "magnum.af_amd", "csrc")


def test_weight_gradient_sums_are_no_longer(tmp_path):
    exe = tmp_path / "net_shapes_check"
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, os.path.join(HERE, "net_shapes_check.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    if r.returncode != 0:
        pytest.fail(r.stderr)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
