"""The indicator's density power (csrc/device/powu.hpp, pow_pos), built for the
host and checked against long-double powl."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pow_pos_within_one_ulp(tmp_path):
    exe = tmp_path / "pow_pos_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", str(exe),
                    os.path.join(HERE, "pow_pos_check.cpp")], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    assert float(out[0]) <= 1.0, out[0]
    assert [float(v) for v in out[1:5]] == [1.0, 2.0, 0.0, 1.0]  # 1^y, an exact power, 0^y, overflow
    assert out[5:] == ["1", "1", "1"]  # negative base, NaN, whole exponents and limits
