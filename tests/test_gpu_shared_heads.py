"""Grouped K/V heads whose count fills no whole rounds of eight: part of a launch's head slices is dealt out by K/V head, the rest
one after the other (set_slice_order).  Every launch form, against the oracle."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Hk,Nq,Nk,d,p,kw", [
    (1, 44, 11, 140, 300, 64, 0.0, dict()),                        # 32-row work-groups
    (3, 36, 9, 300, 300, 64, 0.0, dict()), (3, 36, 9, 290, 290, 96, 0.2, dict(causal=True)),
    (1, 27, 9, 70, 900, 31, 0.2, dict(num_splits=3)), (1, 22, 11, 130, 2000, 64, 0.0, dict(num_splits=3)),  # the latter paired
    (1, 20, 10, 700, 700, 128, 0.0, dict(causal=True, kernel_hint=2)),  # 8-wave kernel
    (5, 20, 5, 1, 700, 64, 0.2, dict(num_splits=1)),
])
def test_ragged_counts_of_shared_heads(fa, oracle, B, H, Hk, Nq, Nk, d, p, kw):
    import torch

    q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
    okw = dict(causal=kw.get("causal", False))
    if p:
        kw = dict(kw, dropout_p=p, seed=7, offset=8)
        okw.update(keep_mask=torch.from_numpy(oracle.dropout_keep_mask(7, 8, p, B, H, Nq, Nk)), p_drop=p)
    kr, vr = (t.repeat_interleave(H // Hk, dim=1).contiguous() for t in (k, v))
    O, L = oracle_forward_batched(oracle, q, kr, vr, **okw)
    call = fa.flash_forward_splitkv if "num_splits" in kw else fa.flash_forward
    check_o_lse(*call(q, k, v, **kw), O, L, f"{B} {H} {Hk} {Nq} {Nk} {d} {kw}")
