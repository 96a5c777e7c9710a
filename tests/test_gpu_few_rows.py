"""Launches of few rows per slice: 32-row work-groups that read K and V once, whole or in splits, and up to 512 rows in splits whose row
blocks share the tiles.  The lines of the rule, and every instance on both sides of them against the oracle: rows shorter than
their bucket at any alignment, folded heads under a causal mask, tiles that not every wave has, a last tile that is not whole,
counters given and not."""
import ctypes as C

import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu
from launch_recorder import KV_ONCE, NARROW, call, record

ROWS, MANY_ROWS = 1 << 12, 1 << 13

# B, H, Hk, Nq, Nk, d, splits asked for -> splits, variant bits
LINES = [
    (1, 32, 8, 1, 1920, 64, 0, 8, ROWS), (4, 32, 8, 1, 8192, 128, 0, 8, ROWS), (1, 32, 8, 1, 32768, 128, 0, 32, ROWS),
    (32, 32, 8, 1, 4096, 128, 0, 1, ROWS), (18, 32, 8, 1, 512, 64, 0, 1, ROWS), (17, 32, 8, 1, 512, 64, 1, 1, ROWS),
    (33, 32, 8, 1, 4096, 128, 1, 1, 0), (15, 32, 8, 1, 4096, 128, 1, 1, 0), (32, 32, 8, 1, 511, 128, 1, 1, 0),
    (1, 32, 8, 1, 2048, 128, 16, 16, 0), (1, 32, 8, 1, 32768, 128, 33, 33, 0), (16, 32, 8, 1, 16384, 128, 0, 4, 0),
    (30, 8, 8, 8, 3000, 128, 0, 1, ROWS), (30, 8, 8, 33, 3000, 128, 1, 1, 0),
    (2, 8, 8, 64, 4096, 128, 0, 8, ROWS | MANY_ROWS), (2, 8, 8, 33, 4096, 128, 0, 8, ROWS | MANY_ROWS), (2, 8, 8, 32, 4096, 64, 0, 16, ROWS),
    (1, 32, 4, 16, 8192, 128, 0, 16, ROWS | MANY_ROWS), (1, 32, 32, 128, 16384, 128, 0, 8, 0), (1, 32, 32, 128, 4096, 128, 2, 2, ROWS | MANY_ROWS),
    (1, 4, 4, 512, 4096, 128, 0, 4, ROWS | MANY_ROWS), (1, 4, 4, 513, 4096, 128, 3, 3, 0), (3, 2, 1, 448, 2752, 128, 0, 3, ROWS | MANY_ROWS),
    (1, 12, 2, 100, 7000, 100, 5, 5, 0), (2, 8, 8, 100, 8000, 64, 4, 4, 0), (1, 2, 2, 128, 4096, 64, 11, 11, 0),
]


def test_lines():
    for (B, H, Hk, Nq, Nk, d, asked, S, bits), r in zip(LINES, record([dict(call(B, H, Hk, Nq, Nk, d, num_splits=asked), entry="splitkv")
                                                                     for B, H, Hk, Nq, Nk, d, asked, _, _ in LINES])):
        assert r["rc"] == 0 and r["splits"] == S, (B, H, Hk, Nq, Nk, d, r)
        launch = r["launches"][0]
        assert launch["variant"] & (ROWS | MANY_ROWS) == bits, (B, H, Hk, Nq, Nk, d, launch)
        if bits:
            folds = Nq <= 64 and Hk < H
            rows, slices = (Nq * (H // Hk), B * Hk) if folds else (Nq, B * H)
            assert launch["variant"] & NARROW and not launch["variant"] & KV_ONCE
            assert launch["groups"] == slices * ((rows + 31) // 32) * S and len(r["launches"]) == (2 if S > 1 else 1)
    # features and hints stay with the forms that serve them
    for kw in (dict(p=0.1), dict(alibi=True), dict(window=(100, -1)), dict(window=(-1, 3)), dict(kernel_hint=1)):
        r, = record([call(2, 8, 8, 20, 4096, 64, num_splits=16, **kw)])
        assert not r["launches"][0]["variant"] & ROWS, kw


@pytest.mark.gpu
@pytest.mark.parametrize("d", [8, 31, 32, 40, 64, 72, 96, 100, 128])
@pytest.mark.parametrize("B,H,Hk,Nq,Nk,S,causal", [
    (1, 32, 8, 1, 6200, 24, False),   # heads as rows
    (2, 16, 8, 2, 4099, 12, True),    # folded heads; a last tile of three keys
    (3, 16, 16, 32, 1025, 4, True),   # all rows of a work-group; the last split has one key
    (12, 12, 12, 5, 700, 1, True),    # whole: eleven tiles, the last not whole
    (9, 32, 16, 16, 513, 1, True),    # whole, folded
    (2, 8, 8, 33, 3000, 8, True),     # more than one row block, the last with one row
    (1, 16, 4, 30, 3001, 12, True),   # the same folded, 120 rows
    (2, 4, 4, 128, 1600, 6, False),
    (1, 6, 3, 200, 1900, 4, True),    # query heads that share K and V, and row blocks of eight neighbours split over the order's end
])
def test_few_rows(fa, oracle, B, H, Hk, Nq, Nk, S, causal, d):
    r, = record([dict(call(B, H, Hk, Nq, Nk, d, causal=causal, num_splits=S), entry="splitkv")])
    G = H // Hk
    rows = Nq * G if Nq <= 64 else Nq
    if rows > 32 or d > 64 or S == 1 or d <= 32:
        assert r["launches"][0]["variant"] & ROWS
    q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
    kr, vr = (t.repeat_interleave(G, dim=1).contiguous() for t in (k, v))
    O, L = oracle_forward_batched(oracle, q, kr, vr, causal=causal)
    check_o_lse(*fa.flash_forward_splitkv(q, k, v, num_splits=S, causal=causal), O, L, "splits")
    if S == 1:
        check_o_lse(*fa.flash_forward(q, k, v, causal=causal), O, L, "whole")


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,Nq,d,S", [(1, 32, 8, 1, 31, 24), (1, 32, 8, 1, 128, 8), (8, 16, 8, 2, 100, 4), (1, 32, 8, 1, 64, 12)])
def test_merge_by_the_last_work_group(fa, B, H, Hk, Nq, d, S):
    """The same bits whoever merges, call after call, and counters that end at zero; partial results of an earlier call do not matter."""
    import torch
    from flash_attn_amd import binding

    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    counters = torch.zeros(B * H, dtype=torch.int32, device="cuda")
    for Nk in (S * 256, S * 256 - 200):
        q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
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
            res.append((o, lse))
        assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
        assert torch.isfinite(res[0][0]).all() and torch.isfinite(res[0][1]).all()
