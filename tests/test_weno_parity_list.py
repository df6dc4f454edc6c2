"""The mirror-symmetric WENO list (csrc/host/parity_weno.hpp) against the dense rows
of every substencil, derivative and point, for both dimensions and both rules,
and its refusal of tables without the symmetry."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HOST = os.path.join(HERE, "..", "kfvm-kokkos_amd", "csrc", "host")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_list_equals_dense_rows(tmp_path):
    exe = tmp_path / "weno_parity_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-fconstexpr-ops-limit=200000000", "-I", HOST, "-o", str(exe),
                    os.path.join(HERE, "weno_parity_check.cpp")] +
                   [os.path.join(HOST, f) for f in ("weights.cpp", "common.cpp", "problems.cpp")] +
                   ["-lquadmath"], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout
