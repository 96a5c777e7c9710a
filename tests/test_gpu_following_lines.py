"""Causal launches of 257 to 512 work-groups: from which number of keys on they are paired, by head dimension, number and dropout,
and launches right at the lines against the oracle."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu
from launch_recorder import call, form, record

# H, keys at the line, d, p (one sequence; H ceil(N / 128) work-groups)
LINES = [(44, 704, 32, 0.0), (44, 704, 40, 0.0), (64, 704, 64, 0.0), (40, 960, 80, 0.0), (40, 1104, 128, 0.0),      # up to 384 of them
         (40, 960, 31, 0.1), (60, 608, 64, 0.1), (60, 608, 96, 0.1), (60, 640, 100, 0.1),
         (40, 1184, 64, 0.0), (32, 1600, 96, 0.0), (34, 1600, 72, 0.0), (36, 1760, 80, 0.0), (30, 1856, 128, 0.0), (42, 1856, 64, 0.0), (50, 1280, 64, 0.1)]  # more


def test_lines():
    calls = [call(1, H, H, n, n, d, p, causal=True) for H, N, d, p in LINES for n in (N - 1, N)]
    forms = [form(r["launches"][0]) for r in record(calls)]
    groups = [c["H"] * -(-c["Nq"] // 128) for c in calls]
    assert all(256 < g <= 512 or f == "plain" for g, f in zip(groups, forms)), list(zip(calls, groups, forms))
    for i, line in enumerate(LINES):
        if groups[2 * i] == groups[2 * i + 1] <= 512:
            assert forms[2 * i:2 * i + 2] == ["plain", "paired"], (line, groups[2 * i], forms[2 * i:2 * i + 2])


@pytest.mark.gpu
@pytest.mark.parametrize("H,N,d,p", [(48, 704, 40, 0.0), (48, 703, 64, 0.0), (44, 960, 96, 0.0), (36, 1184, 31, 0.0), (60, 608, 64, 0.1), (56, 640, 128, 0.1)])
def test_at_the_lines(fa, oracle, H, N, d, p):
    import torch

    q, k, v = (randn_f16_gpu((1, H, N, d), s) for s in (4, 5, 6))
    okw, kw = dict(causal=True), dict(causal=True)
    if p:
        kw.update(dropout_p=p, seed=9)
        okw.update(keep_mask=torch.from_numpy(oracle.dropout_keep_mask(9, 0, p, 1, H, N, N)), p_drop=p)
    O, L = oracle_forward_batched(oracle, q, k, v, **okw)
    check_o_lse(*fa.flash_forward(q, k, v, **kw), O, L, "at the line")
