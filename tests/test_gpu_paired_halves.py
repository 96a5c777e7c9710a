"""Paired work-groups: eight waves in two halves that take every other key tile.  Row counts at the edges of a wave and of a
work-group, odd and even tile counts (the masks leave from one tile up), whole and split, every row alignment and folded
heads, against the oracle."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nq,G,d", [(33, 1, 128), (128, 1, 64), (129, 1, 96), (200, 1, 31), (140, 1, 100), (135, 1, 80),
                                    (20, 2, 128), (30, 4, 72), (64, 2, 40), (5, 1, 32)])
@pytest.mark.parametrize("kw", [dict(), dict(causal=True), dict(causal=True, window=(390, -1)), dict(window=(300, 120))])
def test_paired_halves(fa, oracle, Nq, G, d, kw):
    B, Hk, Nk = 1, 2, 1740
    q, k, v = randn_f16_gpu((B, Hk * G, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
    kr, vr = (t.repeat_interleave(G, dim=1).contiguous() for t in (k, v))
    O, L = oracle_forward_batched(oracle, q, kr, vr, **kw)
    for S in (2, 3):
        check_o_lse(*fa.flash_forward_splitkv(q, k, v, num_splits=S, **kw), O, L, f"split {S}")


# (tests/test_launch_geometry.py holds these three lists against the rule)
UNSPLIT = [(1, 17, 1290, 100), (1, 20, 900, 112), (1, 20, 1100, 31), (1, 11, 1090, 64)]


@pytest.mark.parametrize("B,H,N,d", UNSPLIT)
def test_paired_halves_unsplit(fa, oracle, B, H, N, d):
    """Unsplit causal launches of 64 to 256 work-groups, too many rows for the narrow instances."""
    q, k, v = (randn_f16_gpu((B, H, N, d), s) for s in (4, 5, 6))
    O, L = oracle_forward_batched(oracle, q, k, v, causal=True)
    check_o_lse(*fa.flash_forward(q, k, v, causal=True), O, L, "unsplit")


@pytest.mark.parametrize("Nq,d", [(33, 128), (129, 96), (140, 100), (200, 31), (128, 64)])
def test_paired_halves_dropout(fa, oracle, Nq, d):
    import torch

    B, H, Nk, p = 1, 2, 1740, 0.2
    q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, H, Nk, d), 2), randn_f16_gpu((B, H, Nk, d), 3)
    keep = torch.from_numpy(oracle.dropout_keep_mask(9, 0, p, B, H, Nq, Nk))
    O, L = oracle_forward_batched(oracle, q, k, v, causal=True, keep_mask=keep, p_drop=p)
    check_o_lse(*fa.flash_forward_splitkv(q, k, v, num_splits=3, causal=True, dropout_p=p, seed=9), O, L, "dropout")


UNSPLIT_DROPOUT = [(1, 20, 700, 128, dict(causal=True)), (1, 11, 1090, 64, dict(causal=True)),
                   (1, 20, 900, 100, dict(causal=True, window=(390, -1))), (1, 16, 1100, 96, dict(window=(600, 0))),
                   (1, 34, 800, 31, dict(causal=True))]


@pytest.mark.parametrize("B,H,N,d,kw", UNSPLIT_DROPOUT)
def test_paired_halves_unsplit_dropout(fa, oracle, B, H, N, d, kw):
    """Whole launches with dropout, under a mask and under a window, and the decisions that the two halves store."""
    import torch

    p = 0.2
    q, k, v = (randn_f16_gpu((B, H, N, d), s) for s in (4, 5, 6))
    keep = torch.from_numpy(oracle.dropout_keep_mask(9, 0, p, B, H, N, N))
    O, L = oracle_forward_batched(oracle, q, k, v, keep_mask=keep, p_drop=p, **kw)
    o, lse = fa.flash_forward(q, k, v, dropout_p=p, seed=9, **kw)
    check_o_lse(o, lse, O, L, "unsplit dropout")
    o1, lse1, stored = fa.flash_forward(q, k, v, dropout_p=p, seed=9, return_keep_mask=True, **kw)
    assert torch.equal(o1, o) and torch.equal(lse1, lse)
    i, j = torch.arange(N).view(-1, 1), torch.arange(N).view(1, -1)
    visible = (j <= i) & (i - j <= (kw.get("window", (N,))[0] if kw.get("window", (-1,))[0] >= 0 else N))
    assert torch.equal(stored.cpu()[..., visible], keep[..., visible])


@pytest.mark.parametrize("Nq,d", [(33, 128), (140, 100), (128, 64)])
def test_paired_halves_windowed_dropout(fa, oracle, Nq, d):
    import torch

    B, H, Nk, p, kw = 1, 2, 1740, 0.2, dict(causal=True, window=(390, -1))
    q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, H, Nk, d), 2), randn_f16_gpu((B, H, Nk, d), 3)
    keep = torch.from_numpy(oracle.dropout_keep_mask(9, 0, p, B, H, Nq, Nk))
    O, L = oracle_forward_batched(oracle, q, k, v, keep_mask=keep, p_drop=p, **kw)
    check_o_lse(*fa.flash_forward_splitkv(q, k, v, num_splits=3, dropout_p=p, seed=9, **kw), O, L, "windowed dropout")


FOLLOWING = [(1, 28, 28, 1283, 1283, 100, 0.0), (2, 12, 4, 1700, 1921, 40, 0.0), (1, 26, 26, 1281, 1300, 64, 0.2), (1, 24, 24, 1925, 1870, 72, 0.0)]


@pytest.mark.parametrize("B,H,Hk,Nq,Nk,d,p", FOLLOWING)
def test_paired_halves_one_after_the_other(fa, oracle, B, H, Hk, Nq, Nk, d, p):
    """Causal launches of 257 to 512 work-groups, two of them one after the other on a CU; rows that see no key among them."""
    import torch

    q, k, v = randn_f16_gpu((B, H, Nq, d), 4), randn_f16_gpu((B, Hk, Nk, d), 5), randn_f16_gpu((B, Hk, Nk, d), 6)
    kr, vr = (t.repeat_interleave(H // Hk, dim=1).contiguous() for t in (k, v))
    okw, kw = dict(causal=True), dict(causal=True)
    if p:
        kw.update(dropout_p=p, seed=9)
        okw.update(keep_mask=torch.from_numpy(oracle.dropout_keep_mask(9, 0, p, B, H, Nq, Nk)), p_drop=p)
    O, L = oracle_forward_batched(oracle, q, kr, vr, **okw)
    o, lse = fa.flash_forward(q, k, v, **kw)
    check_o_lse(o, lse, O, L, "two paired work-groups per CU")
    assert all(torch.equal(a, b) for a, b in zip(fa.flash_forward(q, k, v, **kw), (o, lse)))
