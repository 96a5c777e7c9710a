"""Narrow work-groups of the 64-column bucket, whose waves work out the scores of their next tile beside the exponentials of the present
one: one to five tiles per wave with ragged ends, tiles that only some waves have, every mask and row alignment, a first tile past key 0,
rows without a key."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu
from launch_recorder import call, form, record

# keys: one, two, three, four and five tiles for the first wave, the last wave's count one lower or the last tile ragged
KEYS = [200, 257, 320, 512, 513, 700, 769, 960, 1025, 1100, 1279]
LENGTHS = [64, 63, 56, 48, 33]
MASKS = [dict(), dict(causal=True), dict(window=(300, 40)), dict(causal=True, alibi=True)]
# a window of four or five tiles per wave whose first tile is not key 0's: left keys, keys
WIDE = [(900, 1279), (1000, 1300), (1101, 1500)]


def test_route():
    for d in LENGTHS:
        for mask in MASKS:
            for r in record([call(1, 3, 3, 70, Nk, d, **mask) for Nk in KEYS]):
                assert form(r["launches"][0]) == "narrow"
        for r in record([call(1, 3, 3, 70, Nk, d, window=(left, 40)) for left, Nk in WIDE] + [call(1, 3, 3, 900, 850, d, causal=True)]):
            assert form(r["launches"][0]) == "narrow"


@pytest.mark.gpu
@pytest.mark.parametrize("d", LENGTHS)
@pytest.mark.parametrize("mask", MASKS)
def test_scores_ahead(fa, oracle, d, mask):
    import torch

    kw = {x: mask[x] for x in mask if x != "alibi"}
    mine, theirs = dict(kw), dict(kw)
    if "alibi" in mask:
        slopes = torch.tensor([0.25, 0.01, 0.0])
        mine["alibi_slopes"], theirs["slopes"] = slopes.cuda(), slopes.numpy()
    for Nk in KEYS:
        q, k, v = randn_f16_gpu((1, 3, 70, d), 1), randn_f16_gpu((1, 3, Nk, d), 2), randn_f16_gpu((1, 3, Nk, d), 3)
        k[..., -200:, :] *= 3  # the maximum rises towards the last tiles
        O, L = oracle_forward_batched(oracle, q, k, v, **theirs)
        check_o_lse(*fa.flash_forward(q, k, v, **mine), O, L, f"Nk {Nk}")


@pytest.mark.gpu
@pytest.mark.parametrize("d", LENGTHS)
def test_wide_windows_and_rows_without_keys(fa, oracle, d):
    for Nq, Nk, mask in [(70, Nk, dict(window=(left, 40))) for left, Nk in WIDE] + [(900, 850, dict(causal=True))]:
        q, k, v = randn_f16_gpu((1, 3, Nq, d), 1), randn_f16_gpu((1, 3, Nk, d), 2), randn_f16_gpu((1, 3, Nk, d), 3)
        O, L = oracle_forward_batched(oracle, q, k, v, **mask)
        check_o_lse(*fa.flash_forward(q, k, v, **mask), O, L, f"Nq {Nq} Nk {Nk}")
