"""The order of a launch's work-groups, checked on the host (tests/work_order_test.cpp).  No GPU needed."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "flash_attn_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("work_order") / "work_order_test")
    subprocess.check_call(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-std=c++17", "-O1",
                           "-I", CSRC, os.path.join(HERE, "work_order_test.cpp"), "-o", exe])
    return exe


@pytest.mark.parametrize("check", ["bijection", "places", "shared_heads"])
def test_work_order(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
