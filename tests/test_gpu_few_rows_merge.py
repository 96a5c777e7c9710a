"""Launches of few rows whose last work-group merges the partial results: which ones they are, that they are one launch, and their results, in
rows of every whole bucket."""
import ctypes as C

import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu
from launch_recorder import call, record

ROWS = 1 << 12

# B, H, Hk, Nq, Nk, d, splits, launches
LINES = [
    (4, 32, 8, 1, 4000, 128, 8, 1), (7, 16, 4, 1, 4000, 128, 9, 2), (25, 4, 1, 1, 4000, 96, 8, 1), (25, 4, 1, 1, 4000, 96, 9, 2),  # eight splits
    (1, 32, 8, 1, 4000, 64, 8, 1), (1, 32, 8, 1, 4000, 64, 9, 2), (2, 32, 8, 1, 4000, 32, 8, 1), (2, 32, 8, 1, 4000, 32, 9, 2),
    (6, 8, 8, 4, 4000, 64, 4, 1), (6, 8, 8, 5, 4000, 64, 4, 2), (12, 8, 4, 2, 4000, 128, 4, 1), (12, 8, 4, 3, 4000, 128, 4, 2),    # four rows
    (8, 32, 8, 1, 4000, 100, 4, 2), (8, 32, 8, 1, 4000, 120, 4, 2), (4, 32, 8, 1, 4000, 40, 8, 2), (4, 32, 8, 1, 4000, 31, 8, 2),  # whole buckets
]


def recorded(cases, missing=0):
    return record([dict(call(*c[:6], num_splits=c[6]), entry="splitkv", split_counters=0xB00000, split_counters_len=c[0] * c[1] - missing)
                   for c in cases])


def test_lines():
    for c, r in zip(LINES, recorded(LINES)):
        assert r["rc"] == 0 and r["splits"] == c[6] and r["launches"][0]["variant"] & ROWS and len(r["launches"]) == c[7], (c, r)


def test_words():
    """A word per query head, however many of them share a slice; with one less, a launch of its own."""
    cases = [c for c in LINES if c[7] == 1] + [(2, 16, 16, 1, 4000, 64, 8, 1), (2, 16, 8, 1, 4000, 64, 8, 1)]
    assert [len(r["launches"]) for r in recorded(cases)] == [1] * len(cases)
    assert [len(r["launches"]) for r in recorded(cases, missing=1)] == [2] * len(cases)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,Nq,d,S", [(8, 32, 8, 1, 128, 4), (6, 16, 4, 1, 128, 8), (8, 32, 8, 1, 96, 4), (20, 8, 2, 1, 96, 5), (8, 16, 8, 2, 96, 3), (16, 6, 6, 3, 128, 2),
                                           (1, 32, 8, 1, 64, 8), (2, 8, 8, 4, 64, 5), (1, 32, 8, 1, 32, 8), (3, 8, 4, 2, 32, 6)])
def test_one_launch(fa, oracle, B, H, Hk, Nq, d, S):
    """Against the oracle, and the same bits as the merge by a launch of its own, call after call; the counters end at zero.  A last tile of three
    keys, and splits of unequal length."""
    import torch
    from flash_attn_amd import binding

    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    counters = torch.zeros(B * H, dtype=torch.int32, device="cuda")
    for Nk in (S * 256, S * 384 - 125):
        r, = recorded([(B, H, Hk, Nq, Nk, d, S)])
        assert r["launches"][0]["variant"] & ROWS and len(r["launches"]) == 1
        q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
        kr, vr = (t.repeat_interleave(H // Hk, dim=1).contiguous() for t in (k, v))
        O, L = oracle_forward_batched(oracle, q, kr, vr, causal=True)
        res = []
        for given in (0, B * H):
            o, lse = torch.empty_like(q), torch.empty((B, H, Nq), device="cuda")
            ws = torch.full((B * H * S * Nq * d,), float("nan"), device="cuda"), torch.full((B * H * S * Nq,), float("nan"), device="cuda")
            p = binding.make_params(q, k, v, o, lse, None, True, (-1, -1), None, 0.0, 0, 0, S, *ws)
            p.split_counters, p.split_counters_len = (counters.data_ptr() if given else None), given
            for _ in range(3):
                assert fa.lib().flash_forward_splitkv(C.byref(p), stream) == 0
            torch.cuda.synchronize()
            assert not counters.any()
            check_o_lse(o, lse, O, L, f"{Nk} keys, {given} counters")
            res.append((o, lse))
        assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
