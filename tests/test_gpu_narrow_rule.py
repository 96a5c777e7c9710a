"""Launches on both sides of the lines that the rule for the 32-row work-groups draws (fwd_uses_narrow): tile counts, work-group
counts, windows and row lengths around them, every feature combination in every head-dim bucket, against the oracle."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu

pytestmark = pytest.mark.gpu


# (the last field: what the launch is, which tests/test_launch_geometry.py holds the rule to)
LINES = [
    (2, 4, 192, 64, dict(), "plain"), (2, 4, 193, 64, dict(), "narrow"),       # up to 64 groups of 32 rows: 3 | 4 tiles
    (2, 3, 300, 64, dict(window=(100, 0)), "plain"), (2, 3, 300, 64, dict(window=(140, 0)), "narrow"),  # 4 | 5 under a window
    (1, 33, 64, 64, dict(), "plain"), (1, 33, 65, 64, dict(), "narrow"),       # more of them: 1 | 2 tiles
    (1, 12, 600, 64, dict(window=(60, 0)), "narrow"),                          # also under a window
    (1, 17, 128, 100, dict(), "plain"), (1, 17, 129, 100, dict(), "narrow"),   # row shorter than the widest bucket: 2 | 3
    (1, 4, 320, 80, dict(), "narrow"), (1, 4, 321, 80, dict(causal=True), "narrow"),  # rows shorter than their buckets
    (1, 2, 576, 100, dict(), "narrow"), (1, 2, 577, 100, dict(causal=True), "narrow"), (1, 2, 577, 112, dict(), "narrow"),
    (1, 48, 192, 32, dict(), "plain"), (1, 33, 256, 32, dict(), "narrow"),     # more than the CUs, at two per CU: 3 | 4 tiles
    (2, 32, 256, 32, dict(causal=True), "narrow"), (1, 32, 272, 32, dict(), "narrow"),
    (1, 32, 256, 128, dict(), "narrow"), (1, 33, 256, 128, dict(), "plain"),   # 256 | 264 groups
    (1, 12, 832, 64, dict(causal=True), "narrow"), (1, 12, 833, 96, dict(causal=True), "narrow"),  # two rounds, causal
    (1, 13, 700, 64, dict(causal=True), "narrow"), (1, 14, 700, 64, dict(causal=True), "paired"),  # 11 tiles: 286 | 308 groups
    (1, 20, 640, 96, dict(causal=True), "narrow"), (1, 21, 640, 96, dict(causal=True), "paired"),  # 10 tiles: 400 | 420 groups
    (1, 18, 576, 31, dict(causal=True), "narrow"),                             # 324 groups at two per CU, any alignment
]


@pytest.mark.parametrize("B,H,N,d,kw,form", LINES)
def test_around_the_lines(fa, oracle, B, H, N, d, kw, form):
    q, k, v = (randn_f16_gpu((B, H, N, d), s) for s in (1, 2, 3))
    O, L = oracle_forward_batched(oracle, q, k, v, **kw)
    check_o_lse(*fa.flash_forward(q, k, v, **kw), O, L, f"{B} {H} {N} {d} {kw}")


@pytest.mark.parametrize("d", [31, 40, 64, 72, 96, 99, 112, 128])
@pytest.mark.parametrize("alibi,p", [(True, 0.0), (False, 0.2), (True, 0.2)])
def test_features_in_every_bucket(fa, oracle, d, alibi, p):
    import torch

    B, H, N = 1, 3, 700  # 66 groups of 32 rows, 11 tiles
    q, k, v = (randn_f16_gpu((B, H, N, d), s) for s in (4, 5, 6))
    kw, okw = dict(causal=True), dict(causal=True)
    if alibi:
        sl = oracle.alibi_slopes(H)
        kw, okw = dict(kw, alibi_slopes=torch.from_numpy(sl).cuda()), dict(okw, slopes=sl)
    if p:
        keep = oracle.dropout_keep_mask(7, 8, p, B, H, N, N)
        kw, okw = dict(kw, dropout_p=p, seed=7, offset=8), dict(okw, keep_mask=torch.from_numpy(keep), p_drop=p)
    O, L = oracle_forward_batched(oracle, q, k, v, **okw)
    check_o_lse(*fa.flash_forward(q, k, v, **kw), O, L, f"d {d} {sorted(kw)}")


ROUNDS = [  # all narrow
    (2, 65, 65, 140, 2010, 32, 0.0, dict()), (1, 54, 54, 600, 2049, 24, 0.0, dict(causal=True)),  # 128-row work-groups past the CUs
    (2, 130, 65, 50, 4100, 32, 0.0, dict()),                                     # folded, a second round at two per CU
    (1, 9, 9, 930, 1540, 64, 0.0, dict()), (1, 9, 9, 930, 1540, 40, 0.2, dict()),  # K and V in L2
    (1, 11, 11, 900, 2000, 50, 0.0, dict(window=(-1, 30))),                      # later work-groups with fewer keys
    (1, 8, 8, 300, 2000, 128, 0.0, dict(window=(900, 20))), (1, 8, 4, 300, 2000, 100, 0.2, dict(window=(900, -1))),  # one stage per wave:
    (1, 4, 4, 700, 400, 128, 0.0, dict(causal=True)), (1, 4, 4, 700, 450, 96, 0.2, dict(causal=True)),  # tiles and rows without a key
    (1, 14, 14, 1001, 1001, 96, 0.0, dict(causal=True)), (1, 6, 6, 1288, 772, 128, 0.2, dict(causal=True)),  # 448 and 246 that see a key
    (1, 7, 7, 290, 130, 72, 0.0, dict(window=(40, -1))), (1, 13, 13, 1213, 2304, 112, 0.0, dict(causal=True)),
]


@pytest.mark.parametrize("B,H,Hk,Nq,Nk,d,p,kw", ROUNDS)
def test_more_rounds_and_one_stage_loops(fa, oracle, B, H, Hk, Nq, Nk, d, p, kw):
    import torch

    q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
    okw = dict(kw)
    if p:
        kw = dict(kw, dropout_p=p, seed=7, offset=8)
        okw.update(keep_mask=torch.from_numpy(oracle.dropout_keep_mask(7, 8, p, B, H, Nq, Nk)), p_drop=p)
    kr, vr = (t.repeat_interleave(H // Hk, dim=1).contiguous() for t in (k, v))
    O, L = oracle_forward_batched(oracle, q, kr, vr, **okw)
    check_o_lse(*fa.flash_forward(q, k, v, **kw), O, L, f"{B} {H} {Hk} {Nq} {Nk} {d} {kw}")
