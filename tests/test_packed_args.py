"""The arguments that the tiled kernels get, packed and unpacked on the host (tests/packed_args_test.cpp), and their size in the code
as it was built.  No GPU needed."""
import os
import re
import subprocess

import launch_recorder as lr
import machine_code as mc

HERE = os.path.dirname(os.path.abspath(__file__))
LIBRARY = os.path.join(mc.ROOT, "flash_attn_amd", "lib", "libflash_attn_mi355.so")


def test_round_trip(tmp_path):
    exe = str(tmp_path / "packed_args_test")
    subprocess.check_call(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-std=c++17", "-O1", "-I",
                           os.path.join(os.path.dirname(HERE), "flash_attn_amd", "csrc"), os.path.join(HERE, "packed_args_test.cpp"), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


def test_arguments_are_few():
    """112 bytes at most, hidden arguments included, for every kernel without ALiBi, dropout and debug outputs, and for decode below the
    line from which on its launches get more on purpose."""
    seen = 0
    for name, fields in mc.metadata(LIBRARY).items():
        m = re.match(r".*fwd_(?:pp_)?kernelILi\d+E(?:Li\d+E)?Li(\d+)EEE", name)
        if (m and not int(m[1]) & (lr.ALIBI | lr.DROPOUT | lr.STAMP | lr.EVERY)) or "decode_split_kernel" in name or "combine_kernel" in name:
            seen += 1
            assert fields["kernarg_segment_size"] <= 112, (name, fields["kernarg_segment_size"])
    assert seen > 100


def test_decode_addresses_wait_for_no_bit_field():
    """What the first addresses of the decode kernel need has words of its own where there is room for them: without ALiBi nothing but
    shift counts, which shifts take as they are, is cut out of a word before the first request."""
    seen = 0
    for name, body in mc.kernels(LIBRARY):
        if re.match(r".*decode_split_kernelILi\d+ELb0E", name):
            seen += 1
            first = next(i for i, (m, _) in enumerate(body) if m.startswith("global_load"))
            assert not [x for x in body[:first] if x[0].startswith("s_bfe")], name
    assert seen == 12


def argument_lines(body):
    """64-byte lines of the arguments that scalar loads ask for before the first wait for scalar loads, and behind it."""
    first, later, waited = set(), set(), False
    for m, text in body:
        if m.startswith("s_load_dword"):
            target, base, offset = (x.strip() for x in text.split(",")[:3])
            if base != "s[0:1]":
                continue
            words = int(m.removeprefix("s_load_dword").removeprefix("x") or 1)
            lines = range(int(offset, 0) // 64, (int(offset, 0) + 4 * words - 1) // 64 + 1)
            (later if waited else first).update(lines)
            if mc.registers(target) & {("s", 0), ("s", 1)}:
                break
        elif m == "s_waitcnt" and "lgkmcnt" in text:
            waited = True
    return first, later


def test_no_line_of_the_arguments_comes_late():
    """No tiled kernel asks for a line of its arguments for the first time once it has waited for others (ALiBi and dropout together, the
    instances that serve every request and the instrumented twins apart)."""
    seen = 0
    for name, body in mc.kernels(LIBRARY):
        m = re.match(r".*fwd_(?:pp_)?kernelILi\d+E(?:Li\d+E)?Li(\d+)EEE", name)
        if not m or int(m[1]) & (lr.STAMP | lr.EVERY) or int(m[1]) & (lr.ALIBI | lr.DROPOUT) == lr.ALIBI | lr.DROPOUT:
            continue
        seen += 1
        first, later = argument_lines(body)
        assert later <= first, (name, first, later)
    assert seen > 100
