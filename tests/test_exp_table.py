"""exp_table (csrc/exp_table.hpp), the exponential of the every-token masses, against 80-bit arithmetic on the host."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_error(tmp_path):
    if np.finfo(np.longdouble).nmant < 63:
        pytest.skip("no 80-bit long double")
    exe = str(tmp_path / "exp_error")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "exp_error.cpp")], check=True)
    ulp, one = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
    # the last addition rounds by half a unit; before it: t q and the table's rest, each below a hundredth
    assert float(ulp) < 0.53 and one == "1", ulp
