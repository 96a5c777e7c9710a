"""Dropout bits where the tiled kernels take them from their tables of 64 Philox calls (512 keys): key ranges that cross a
table's end, in every order in which the launch forms walk the key tiles -- one after the other, every other one (paired),
every fourth one (narrow), from the last to the first (ALiBi left of the row), from the middle (windows, the later of
several splits) -- held bit by bit against the CPU replica, and the output against the oracle with those bits."""
import numpy as np
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu

pytestmark = pytest.mark.gpu


WALKS = [  # (the last field: what the launch is, which tests/test_launch_geometry.py holds the rules to)
    (1, 2, 130, 1090, 64, {}, "narrow"),                                    # two stages per wave
    (1, 2, 700, 1090, 100, dict(causal=True), "narrow"),                    # one stage per wave
    (2, 4, 1090, 1090, 96, dict(causal=True), "narrow"),                    # two rounds of work-groups
    (1, 11, 1090, 1090, 64, dict(causal=True), "paired"), (1, 20, 800, 800, 100, dict(causal=True), "paired"),
    (3, 30, 600, 600, 63, dict(causal=True), "plain"),                      # a work-group's tiles one after the other, odd rows
    (3, 30, 520, 1030, 96, dict(window=(300, 0)), "plain"),                 # starts inside a table
    (3, 30, 600, 600, 64, dict(causal=True, alibi=True), "plain"),          # from the last tile to the first
    (1, 3, 1100, 1100, 128, dict(causal=True, kernel_hint=2), "8-wave"),
    (1, 3, 300, 1100, 128, dict(window=(700, 0), kernel_hint=2), "8-wave"), # waves that start later than others
    (1, 2, 40, 1600, 72, dict(num_splits=3), "paired"),                     # splits that begin and end inside a table
]


@pytest.mark.parametrize("B,H,Nq,Nk,d,kw,form", WALKS)
def test_keep_decisions_across_call_tables(fa, oracle, B, H, Nq, Nk, d, kw, form):
    import torch
    kw = dict(kw)
    okw = {k: v for k, v in kw.items() if k in ("causal", "window")}
    q, k, v = [randn_f16_gpu((B, H, n, d), 17 + i) for i, n in enumerate((Nq, Nk, Nk))]
    if kw.pop("alibi", False):
        sl = oracle.alibi_slopes(H)
        kw["alibi_slopes"], okw["slopes"] = torch.from_numpy(sl).cuda(), sl
    p, seed, off = 0.3, 2 ** 35 + 11, 5
    keep = oracle.dropout_keep_mask(seed, off, p, B, H, Nq, Nk)
    if "num_splits" in kw:  # (that entry point does not dump the bits)
        o, lse = fa.flash_forward_splitkv(q, k, v, dropout_p=p, seed=seed, offset=off, **kw)
    else:
        o, lse, km = fa.flash_forward(q, k, v, dropout_p=p, seed=seed, offset=off, return_keep_mask=True, **kw)
        i, j = np.arange(Nq)[:, None] + Nk - Nq, np.arange(Nk)[None, :]
        vis = np.ones((Nq, Nk), bool)
        if kw.get("causal"):
            vis &= j <= i
        if "window" in kw:
            vis &= (i - j <= kw["window"][0]) & (j - i <= kw["window"][1])
        assert np.array_equal(km.cpu().numpy()[..., vis], keep[..., vis])
        o2, _ = fa.flash_forward(q, k, v, dropout_p=p, seed=seed, offset=off, **kw)
        assert torch.equal(o, o2)
    O, L = oracle_forward_batched(oracle, q, k, v, keep_mask=torch.from_numpy(keep), p_drop=p, **okw)
    check_o_lse(o, lse, O, L, f"{B, H, Nq, Nk, d, kw}")
