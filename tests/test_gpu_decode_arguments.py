"""Decode launches on both sides of the line from which on they get the longer arguments: 4 MiB of visible keys and values."""
import os

import pytest

import machine_code as mc
from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu
from launch_recorder import call, record

LINE = 4 << 20
LENGTHS = [8, 31, 32, 40, 63, 64, 100, 128]
HEADS = [(8, 8), (16, 8)]  # query heads, K/V heads
OPTIONS = [dict(), dict(alibi=True), dict(window=(999, -1))]


def keys_at_the_line(Hk, d):
    return -(-LINE // (4 * d * Hk))


def kernel(H, Hk, Nk, d, **options):
    launch, = (x for x in record([call(1, H, Hk, 1, Nk, d, num_splits=0, **options)])[0]["launches"] if "combine" not in x["kernel"])
    return launch["kernel"]


def test_route():
    for d in LENGTHS:
        for H, Hk in HEADS:
            for alibi in (False, True):
                Nk = keys_at_the_line(Hk, d)
                assert "decode_split_kernel" in kernel(H, Hk, Nk - 1, d, alibi=alibi)
                assert "decode_stream_kernel" in kernel(H, Hk, Nk, d, alibi=alibi)
    # the keys that a window leaves
    assert "decode_split_kernel" in kernel(8, 8, 9000, 128, window=(1022, -1))
    assert "decode_stream_kernel" in kernel(8, 8, 9000, 128, window=(1023, -1))


def test_sizes():
    sizes = {f["kernarg_segment_size"] for n, f in mc.metadata(os.path.join(mc.ROOT, "flash_attn_amd", "lib", "libflash_attn_mi355.so")).items() if "decode_stream_kernel" in n}
    assert sizes == {192}


@pytest.mark.gpu
@pytest.mark.parametrize("d", LENGTHS)
@pytest.mark.parametrize("H,Hk", HEADS)
def test_both_sides(fa, oracle, H, Hk, d):
    import torch

    for options in OPTIONS:
        for Nk in (keys_at_the_line(Hk, d) - 1, keys_at_the_line(Hk, d)):
            q, k, v = randn_f16_gpu((1, H, 1, d), 1), randn_f16_gpu((1, Hk, Nk, d), 2), randn_f16_gpu((1, Hk, Nk, d), 3)
            mine = {x: y for x, y in options.items() if x != "alibi"}
            theirs = dict(mine)
            if "alibi" in options:
                slopes = torch.linspace(0.0, 0.2, H)
                mine["alibi_slopes"], theirs["slopes"] = slopes.cuda(), slopes.numpy()
            kr, vr = (t.repeat_interleave(H // Hk, dim=1) for t in (k, v))
            O, L = oracle_forward_batched(oracle, q, kr, vr, **theirs)
            check_o_lse(*fa.flash_forward_splitkv(q, k, v, **mine), O, L, f"Nk {Nk} {options}")
