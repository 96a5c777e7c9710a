"""Unmasked d = 64 launches of many heads take 256-row work-groups: bit for bit the results of the 128-row ones (which
kernel_hint = 1 asks for), whole and ragged row counts, key counts that differ, grouped heads; and the oracle on a head."""
import pytest

from helpers import check_o_lse, randn_f16_gpu, to_f32_np

pytestmark = pytest.mark.gpu


# (the rule takes them from 1024 keys on; tests/test_launch_geometry.py holds these shapes against it)
SHAPES = [(32, 32, 32, 256, 1024), (32, 32, 8, 225, 1055), (16, 32, 32, 512, 1088), (16, 32, 32, 449, 1030), (3, 28, 28, 3329, 2049)]
CHUNKS = [(16, 32, 32, 512, 1024), (16, 32, 8, 481, 1090), (3, 28, 28, 3329, 1025), (13, 40, 40, 512, 1087)]


@pytest.mark.parametrize("B,H,Hk,Nq,Nk", SHAPES)
def test_tall_blocks(fa, oracle, B, H, Hk, Nq, Nk):
    import torch

    q, k, v = randn_f16_gpu((B, H, Nq, 64), 1), randn_f16_gpu((B, Hk, Nk, 64), 2), randn_f16_gpu((B, Hk, Nk, 64), 3)
    o, lse = fa.flash_forward(q, k, v)
    o4, lse4 = fa.flash_forward(q, k, v, kernel_hint=1)
    assert torch.equal(o, o4) and torch.equal(lse, lse4)
    O, L = oracle.attention_forward(*(to_f32_np(t[-1:, -1:]) for t in (q, k, v)))
    check_o_lse(o[-1:, -1:], lse[-1:, -1:], O, L, "last head")


@pytest.mark.parametrize("B,H,Hk,Nq,Nk", CHUNKS)
def test_tall_blocks_and_slice_chunks_of_long_key_ranges(fa, oracle, B, H, Hk, Nq, Nk):
    """Slice counts that do and do not divide into chunks of sixteen."""
    test_tall_blocks(fa, oracle, B, H, Hk, Nq, Nk)
