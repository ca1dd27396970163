"""Scalar code shared by kernels and host propagators (csrc/gdp_arith.h), on
the CPU: the candidate bounds against the reference's formulas, bit for bit,
and the decision of a round's launch to run."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("driver", ["arith_driver", "round_runs_driver"])
def test_native(tmp_path, driver):
    exe = tmp_path / driver
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I",
                    os.path.join(REPO, "gpu-domain-propagator_amd", "csrc"), "-o", str(exe),
                    os.path.join(REPO, "tests", "native", driver + ".cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
