"""What launches of few rows work out on the host and unpack in the kernel (tests/few_rows_test.cpp).  No GPU needed."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_arguments_and_order(tmp_path):
    exe = str(tmp_path / "few_rows_test")
    subprocess.check_call(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-std=c++17", "-O1", "-I",
                           os.path.join(os.path.dirname(HERE), "flash_attn_amd", "csrc"), os.path.join(HERE, "few_rows_test.cpp"), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
