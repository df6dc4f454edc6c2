"""The pressure-ratio power of the HLLC shear factor (csrc/device/powu.hpp,
pow_ratio), built for the host and checked against long-double powl with the
bounds of powu."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pow_ratio_matches_libm(tmp_path):
    exe = tmp_path / "pow_ratio_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", str(exe),
                    os.path.join(HERE, "pow_ratio_check.cpp")], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    rel, ab = float(out[0]), float(out[1])
    assert rel < 32.0, rel
    assert ab <= 2.3e-16, ab
    assert [float(v) for v in out[2:]] == [1.0, 1.0, 0.0, 0.5, 0.0]
