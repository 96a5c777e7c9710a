"""Rows of at most D - 16 elements in the head-dim bucket of D columns: instances without the last k-step of Q K^T, in every
launch form that has them, with row lengths on both sides of the line."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu
from launch_recorder import FOLD, FULL_D, call, form, record

SHORT = 2048  # variant bit of fwd_kernel.h

LENGTHS = [(64, 33), (64, 40), (64, 47), (64, 48), (64, 49), (96, 65), (96, 72), (96, 80), (96, 81), (128, 97), (128, 104), (128, 111),
           (128, 112), (128, 113), (128, 120)]
SLOPES = [0.5, 0.03, 0.0]
# form, rows, keys, entry point's arguments
FORMS = [("narrow", 97, 700, dict()),
         ("narrow", 130, 200, dict(causal=True)),
         ("paired", 140, 1740, dict(num_splits=2, causal=True)),
         ("paired", 140, 1740, dict(num_splits=3, p=0.2)),
         ("plain", 130, 300, dict(kernel_hint=1, causal=True)),
         ("plain", 130, 300, dict(kernel_hint=1, window=(70, 0), alibi=True)),
         ("plain", 130, 300, dict(kernel_hint=1, alibi=True)),
         ("plain", 130, 300, dict(kernel_hint=1, p=0.2)),
         ("plain", 130, 300, dict(kernel_hint=1, causal=True, p=0.2, alibi=True)),
         ("plain", 130, 300, dict(kernel_hint=1, window=(70, 40), p=0.2, alibi=True)),
         ("8-wave", 300, 330, dict(kernel_hint=2, causal=True)),
         ("8-wave", 300, 330, dict(kernel_hint=2, p=0.2, alibi=True))]


def forms(d):
    return [f for f in FORMS if d > 96 or f[0] != "8-wave"]


def test_route():
    """Every form of the list is the one that is launched, and leaves the k-step out up to the line and not beyond."""
    cases = [(D, d, f) for D, d in LENGTHS for f in forms(d)]
    for (D, d, f), r in zip(cases, record([call(1, 3, 3, f[1], f[2], d, **f[3]) for _, d, f in cases])):
        launch = r["launches"][0]
        assert form(launch) == f[0], (d, f)
        assert (launch["variant"] & SHORT != 0) == (d <= D - 16), (d, f)
    for d in (32, 64, 96, 128, 16, 31):  # rows of the bucket's width, the smallest bucket
        assert record([call(1, 3, 3, 130, 300, d, kernel_hint=1)])[0]["launches"][0]["variant"] & SHORT == 0
    folded = record([call(2, 8, 2, 5, 3000, 80, num_splits=3)])[0]["launches"][0]["variant"]
    assert folded & FOLD and not folded & (SHORT | FULL_D)


@pytest.mark.gpu
@pytest.mark.parametrize("D,d", LENGTHS)
def test_shorter_rows(fa, oracle, D, d):
    import torch

    B, H = 1, 3
    for i, (name, Nq, Nk, kw) in enumerate(forms(d)):
        q, k, v = randn_f16_gpu((B, H, Nq, d), 3 * i + 1), randn_f16_gpu((B, H, Nk, d), 3 * i + 2), randn_f16_gpu((B, H, Nk, d), 3 * i + 3)
        # the last eight columns decide: a column left out or taken twice shows in every score
        q[..., -8:] *= 3
        options = {x: kw[x] for x in ("causal", "window") if x in kw}
        mine = {x: kw[x] for x in ("causal", "window", "kernel_hint", "num_splits") if x in kw}
        if "alibi" in kw:
            options["slopes"] = torch.tensor(SLOPES).numpy()
            mine["alibi_slopes"] = torch.tensor(SLOPES, device="cuda")
        if "p" in kw:
            options.update(p_drop=kw["p"], keep_mask=torch.from_numpy(oracle.dropout_keep_mask(9, 0, kw["p"], B, H, Nq, Nk)))
            mine.update(dropout_p=kw["p"], seed=9)
        O, L = oracle_forward_batched(oracle, q, k, v, **options)
        run = fa.flash_forward_splitkv if "num_splits" in kw else fa.flash_forward
        check_o_lse(*run(q, k, v, **mine), O, L, f"{name} {kw}")
