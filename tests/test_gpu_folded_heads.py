"""Few query rows per head with grouped K/V heads: the heads of a K/V head run as the rows of one problem.  Row counts at
the edges of a wave's 32 rows, of the 64 up to which heads are folded and of a 128-row work-group, each mask, whole and
split, against the oracle; and the split workspace, whose layout does not show any of this."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nq,G,d", [(2, 2, 64), (3, 8, 80), (31, 3, 31), (32, 4, 128), (33, 4, 96), (43, 3, 100),
                                    (64, 2, 64), (64, 8, 32), (65, 4, 128)])
@pytest.mark.parametrize("kw", [dict(), dict(causal=True), dict(causal=True, window=(70, -1)), dict(window=(300, 11))])
def test_folded_heads(fa, oracle, Nq, G, d, kw):
    import torch

    B, Hk, Nk = 2, 2, 700
    H = Hk * G
    q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
    kr, vr = (t.repeat_interleave(G, dim=1).contiguous() for t in (k, v))
    O, L = oracle_forward_batched(oracle, q, kr, vr, **kw)
    check_o_lse(*fa.flash_forward(q, k, v, **kw), O, L, "whole")
    for S in (0, 3):
        o, lse, (op, lp) = fa.flash_forward_splitkv(q, k, v, num_splits=S, return_partials=True, **kw)
        check_o_lse(o, lse, O, L, f"split {S}")
        if op is None:
            continue
        assert op.shape == (B, H, lp.shape[2], Nq, d)
        # the workspace holds every head's own partial results: merged by hand they are the result (fp32 throughout)
        torch.testing.assert_close(torch.logsumexp(lp, dim=2), lse, rtol=0, atol=1e-5)
        w = torch.exp(lp - lse.unsqueeze(2)).unsqueeze(-1)
        torch.testing.assert_close((w * op).sum(dim=2).half(), o, rtol=2e-3, atol=1e-4)


def test_folded_heads_with_empty_splits(fa, oracle):
    """A left window shorter than a split: most splits see no key of any row and only fill their part of the workspace."""
    B, Hk, G, Nq, Nk, d = 1, 2, 4, 40, 1500, 72
    q, k, v = randn_f16_gpu((B, Hk * G, Nq, d), 4), randn_f16_gpu((B, Hk, Nk, d), 5), randn_f16_gpu((B, Hk, Nk, d), 6)
    kr, vr = (t.repeat_interleave(G, dim=1).contiguous() for t in (k, v))
    kw = dict(causal=True, window=(50, -1))
    O, L = oracle_forward_batched(oracle, q, kr, vr, **kw)
    check_o_lse(*fa.flash_forward_splitkv(q, k, v, num_splits=12, **kw), O, L, "empty splits")
