"""Narrow work-groups, whose waves fetch Q like the first rows of a K tile: row blocks of one to 32 rows, every kind of row length and
alignment, one and several tiles per wave, folded heads, dropout."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu
from launch_recorder import call, form, record

LENGTHS = [8, 9, 16, 31, 32, 33, 40, 63, 64, 65, 80, 95, 96, 97, 104, 112, 113, 127, 128]
ROWS = [2, 31, 32, 33, 61]
KEYS = [130, 270, 600]  # one tile for some waves, for all of them, several


def test_route():
    for d in LENGTHS:
        calls = [call(1, 17, 17, Nq, Nk, d) for Nq in ROWS for Nk in KEYS if 17 * ((Nq + 31) // 32) > 64 or Nk > 192]
        assert all(form(r["launches"][0]) == "narrow" for r in record(calls)), d


@pytest.mark.gpu
@pytest.mark.parametrize("d", LENGTHS)
def test_rows(fa, oracle, d):
    for Nq in ROWS:
        for Nk in KEYS:
            q, k, v = randn_f16_gpu((1, 17, Nq, d), 1), randn_f16_gpu((1, 17, Nk, d), 2), randn_f16_gpu((1, 17, Nk, d), 3)
            O, L = oracle_forward_batched(oracle, q, k, v)
            check_o_lse(*fa.flash_forward(q, k, v), O, L, f"Nq {Nq} Nk {Nk}")


@pytest.mark.gpu
@pytest.mark.parametrize("d", [31, 64, 80, 100, 128])
def test_folded_and_dropout(fa, oracle, d):
    import torch

    q, k, v = randn_f16_gpu((1, 12, 7, d), 4), randn_f16_gpu((1, 3, 600, d), 5), randn_f16_gpu((1, 3, 600, d), 6)
    kr, vr = (t.repeat_interleave(4, dim=1).contiguous() for t in (k, v))
    O, L = oracle_forward_batched(oracle, q, kr, vr, causal=True)
    check_o_lse(*fa.flash_forward(q, k, v, causal=True), O, L, "folded")
    p = 0.2
    keep = torch.from_numpy(oracle.dropout_keep_mask(9, 0, p, 1, 12, 7, 600))
    O, L = oracle_forward_batched(oracle, q, kr, vr, causal=True, keep_mask=keep, p_drop=p)
    check_o_lse(*fa.flash_forward(q, k, v, causal=True, dropout_p=p, seed=9), O, L, "dropout")
