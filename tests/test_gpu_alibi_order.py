"""ALiBi where no visible key lies right of its row: the key tiles are walked from the last to the first.  One to seven
tiles, whole and ragged, under a causal mask, a window and a split, with slopes that move the row maximum by far more
than a tile's scores do, of either sign, against the oracle."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nk,d", [(33, 64), (64, 32), (65, 96), (129, 128), (200, 72), (448, 64)])
@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("kw", [dict(causal=True), dict(window=(70, 0))])
def test_alibi_from_the_last_tile(fa, oracle, Nk, d, kw, p):
    import torch

    B, H = 1, 4
    q, k, v = (randn_f16_gpu((B, H, Nk, d), s) for s in (1, 2, 3))
    slopes = torch.tensor([1.5, 0.25, 0.004, -0.05], dtype=torch.float32, device="cuda")
    gkw, okw = dict(kw, alibi_slopes=slopes), dict(kw, slopes=slopes.cpu().numpy())
    if p > 0:
        gkw.update(dropout_p=p, seed=5)
        okw.update(p_drop=p, keep_mask=torch.from_numpy(oracle.dropout_keep_mask(5, 0, p, B, H, Nk, Nk)))
    O, L = oracle_forward_batched(oracle, q, k, v, **okw)
    check_o_lse(*fa.flash_forward(q, k, v, kernel_hint=1, **gkw), O, L, "whole")
    check_o_lse(*fa.flash_forward_splitkv(q, k, v, num_splits=2, **gkw), O, L, "split")
