"""What the process shares of pinned host memory, on the CPU: the lock of the
staging of bulk copies (csrc/gdp_copy_pool.h) and the pool of blocks
(csrc/gdp_host_blocks.h)."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("driver", ["staging_lock_driver", "host_blocks_driver"])
def test_native(tmp_path, driver):
    exe = tmp_path / driver
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-Wall", "-I",
                    os.path.join(REPO, "gpu-domain-propagator_amd", "csrc"), "-o", str(exe),
                    os.path.join(REPO, "tests", "native", driver + ".cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
