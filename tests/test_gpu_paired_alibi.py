"""Paired work-groups with ALiBi, whose halves walk every other tile from the last to the first: odd and even tile counts, rows that end
inside a wave, every row alignment, windows and causal masks, one and two work-groups per CU, against the oracle."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu
from launch_recorder import call, form, record

# B, H, Hk, Nq, Nk, d, masks, form
CASES = [
    (1, 16, 16, 677, 677, 64, dict(window=(129, 0)), "paired"), (1, 16, 16, 677, 677, 64, dict(window=(128, 0)), "plain"),  # 4 | 5 tiles
    (1, 16, 16, 650, 650, 128, dict(window=(384, 0)), "paired"), (1, 16, 16, 650, 650, 128, dict(window=(383, 0)), "plain"),  # d > 96: 8
    (1, 17, 17, 1290, 1290, 100, dict(causal=True), "paired"), (1, 20, 20, 1100, 1100, 31, dict(causal=True), "paired"),
    (1, 30, 30, 300, 300, 80, dict(causal=True, window=(135, -1)), "paired"), (1, 34, 34, 290, 290, 96, dict(causal=True, window=(130, -1)), "paired"),
    (1, 12, 3, 900, 1300, 72, dict(window=(500, 0)), "paired"), (1, 12, 12, 1300, 900, 40, dict(window=(400, 0)), "paired"),  # rows without a key
    (1, 32, 32, 1160, 1160, 32, dict(causal=True), "paired"), (1, 30, 30, 1283, 1283, 112, dict(causal=True), "paired"),  # 257 to 512 work-groups
    (1, 30, 30, 1283, 1283, 64, dict(window=(500, 0)), "plain"),                     # as many under a window
    (1, 16, 16, 677, 677, 64, dict(window=(200, 100)), "plain"),                     # keys right of the row
]


def test_forms():
    calls = [call(B, H, Hk, Nq, Nk, d, causal=m.get("causal", False), window=m.get("window", (-1, -1)), alibi=True) for B, H, Hk, Nq, Nk, d, m, _ in CASES]
    assert [form(r["launches"][0]) for r in record(calls)] == [c[-1] for c in CASES]


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,Nq,Nk,d,masks", [c[:-1] for c in CASES if c[-1] == "paired"])
def test_paired_alibi(fa, oracle, B, H, Hk, Nq, Nk, d, masks):
    import torch

    q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
    kr, vr = (t.repeat_interleave(H // Hk, dim=1).contiguous() for t in (k, v))
    slopes = oracle.alibi_slopes(H)
    O, L = oracle_forward_batched(oracle, q, kr, vr, slopes=slopes, **masks)
    o, lse = fa.flash_forward(q, k, v, alibi_slopes=torch.from_numpy(slopes).cuda(), **masks)
    check_o_lse(o, lse, O, L, "paired, ALiBi")
