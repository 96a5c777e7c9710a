"""The instrumented twins of launches of few rows, whole and in splits, with a split that has no key, merging in the launch, and of paired work-groups
with ALiBi: the same results bit by bit, and a row of ordered stamps from each work-group."""
import ctypes as C

import numpy as np
import pytest

from helpers import randn_f16_gpu
from launch_recorder import ALIBI, PAIR, STAMP, call, record

ROWS = 1 << 12

# B, H, Hk, Nq, Nk, splits
SHAPES = [(2, 16, 16, 5, 2000, 8), (2, 32, 16, 3, 1500, 8), (1, 16, 16, 41, 2000, 8), (1, 16, 8, 20, 2000, 8), (20, 32, 8, 1, 600, 1)]
DIMS = [31, 32, 40, 63, 64, 72, 96, 100, 112, 128]


def recorded(shapes, d, **kw):
    return record([dict(call(B, H, Hk, Nq, Nk, d, num_splits=S, causal=True), entry="splitkv", stage_stamps_out=0xC00000, **kw)
                   for B, H, Hk, Nq, Nk, S in shapes])


def test_forms():
    for d in DIMS:
        for (B, H, Hk, Nq, Nk, S), r in zip(SHAPES, recorded(SHAPES, d)):
            launch = r["launches"][0]
            assert launch["variant"] & ROWS and launch["variant"] & STAMP and r["stamp_bytes"] == 72 * launch["groups"], (d, B, Nq, launch)


def check(st, Nk):
    t = st.cpu().numpy()
    assert (t[:, 0] > 0).all() and (np.diff(t[:, :7], axis=1) >= 0).all()
    assert ((t[:, 6] - t[:, 0]) < 100_000_000).all() and (t[:, 7] >> 32).max() <= (Nk + 63) // 64


@pytest.mark.gpu
@pytest.mark.parametrize("d", DIMS)
@pytest.mark.parametrize("B,H,Hk,Nq,Nk,S", SHAPES)
def test_few_rows(fa, B, H, Hk, Nq, Nk, S, d):
    import torch

    q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
    o0, l0 = fa.flash_forward_splitkv(q, k, v, num_splits=S, causal=True)
    o, l, st = fa.flash_forward_splitkv(q, k, v, num_splits=S, causal=True, return_stage_stamps=True)
    assert torch.equal(o, o0) and torch.equal(l, l0) and torch.isfinite(o).all()
    check(st, Nk)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [32, 64, 96, 128])
def test_merged_in_the_launch(fa, d):
    import torch
    from flash_attn_amd import binding

    B, H, Hk, Nq, Nk, S = 8, 32, 8, 1, 1500, 4
    r, = recorded([(B, H, Hk, Nq, Nk, S)], d, split_counters=0xB00000, split_counters_len=B * H)
    assert r["launches"][0]["variant"] & ROWS and len(r["launches"]) == 1
    q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
    counters = torch.zeros(B * H, dtype=torch.int32, device="cuda")
    st = torch.zeros((r["launches"][0]["groups"], fa.FLASH_STAMP_WORDS), dtype=torch.int64, device="cuda")
    o, lse = torch.empty_like(q), torch.empty((B, H, Nq), device="cuda")
    ws = torch.empty(B * H * S * Nq * d, device="cuda"), torch.empty(B * H * S * Nq, device="cuda")
    p = binding.make_params(q, k, v, o, lse, None, True, (-1, -1), None, 0.0, 0, 0, S, *ws)
    p.split_counters, p.split_counters_len, p.stage_stamps_out = counters.data_ptr(), B * H, st.data_ptr()
    assert fa.lib().flash_forward_splitkv(C.byref(p), C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    o0, l0 = fa.flash_forward_splitkv(q, k, v, num_splits=S, causal=True)
    assert torch.equal(o, o0) and torch.equal(lse, l0) and not counters.any()
    check(st, Nk)


@pytest.mark.gpu
@pytest.mark.parametrize("H,N,d,masks", [(16, 677, 64, dict(window=(129, 0))), (17, 1290, 100, dict(causal=True)), (20, 1100, 31, dict(causal=True)), (30, 300, 80, dict(causal=True, window=(135, -1))),
                                         (34, 290, 96, dict(causal=True, window=(130, -1))), (32, 1160, 32, dict(causal=True)), (16, 650, 128, dict(window=(384, 0)))])
def test_paired_alibi(fa, H, N, d, masks):
    import torch

    r, = record([dict(call(1, H, H, N, N, d, alibi=True, **masks), stage_stamps_out=0xC00000)])
    assert r["launches"][0]["variant"] & (ALIBI | PAIR | STAMP) == ALIBI | PAIR | STAMP
    q, k, v = (randn_f16_gpu((1, H, N, d), s) for s in (1, 2, 3))
    slopes = torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)], device="cuda")
    o0, l0 = fa.flash_forward(q, k, v, alibi_slopes=slopes, **masks)
    o, l, st = fa.flash_forward(q, k, v, alibi_slopes=slopes, return_stage_stamps=True, **masks)
    assert torch.equal(o, o0) and torch.equal(l, l0) and torch.isfinite(o).all()
    check(st, N)
