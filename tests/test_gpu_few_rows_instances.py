"""Launches of few rows, heads shorter than their bucket: the instance goes by row length and alignment as in the other forms, and its requests
are non-temporal from 22 MiB of K and V on (rows_read_once).  Both sides of that line against the oracle."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu
from launch_recorder import FOLD, FULL_D, NARROW, VEC, call, record

SHORT, ROWS, CACHED = 1 << 11, 1 << 12, 1 << 13
DIMS = [16, 31, 33, 40, 48, 56, 65, 72, 80, 88, 97, 100, 112, 120]
SPLITS = 8


def bucket(d):
    return -(-d // 32) * 32


def sizes(d):
    """Keys of 32 slices right below and at the line."""
    line = -(-(22 << 20) // (4 * 32 * d))
    return [(line - 1, CACHED), (line, 0)]


def shape(folded):
    return (2, 32, 16, 3) if folded else (2, 16, 16, 5)


@pytest.mark.parametrize("folded", [False, True])
def test_instances(folded):
    B, H, Hk, Nq = shape(folded)
    calls, wanted = [], []
    for d in DIMS + [32, 64, 96, 128]:
        bits = NARROW | ROWS | (FOLD if folded else 0)
        if d == bucket(d):
            calls.append(call(B, H, Hk, Nq, 2000, d, num_splits=SPLITS))
            wanted.append(bits | VEC | FULL_D)
            continue
        bits |= VEC if d % 8 == 0 and d > 32 else 0
        bits |= SHORT if not folded and d > 32 and d <= bucket(d) - 16 else 0
        for Nk, cached in sizes(d):
            calls.append(call(B, H, Hk, Nq, Nk, d, num_splits=SPLITS))
            wanted.append(bits | cached)
    found = [r["launches"][0]["variant"] for r in record(calls)]
    assert found == wanted, [(c["d"], c["Nk"], f, w) for c, f, w in zip(calls, found, wanted) if f != w]


def test_whole_launches():
    """The same line, and ordinary requests below 160 slices."""
    for d, B, Nk, cached in [(40, 20, 901, CACHED), (40, 20, 902, 0), (40, 19, 2000, CACHED), (31, 20, 1163, 0), (112, 20, 321 + 191, 0), (64, 17, 600, 0), (128, 17, 600, 0)]:
        r, = record([call(B, 32, 8, 1, Nk, d)])
        assert r["launches"][0]["variant"] & (ROWS | CACHED) == ROWS | cached, (d, B, Nk)


@pytest.mark.gpu
@pytest.mark.parametrize("folded", [False, True])
@pytest.mark.parametrize("d", DIMS)
def test_few_rows_of_shorter_heads(fa, oracle, d, folded):
    B, H, Hk, Nq = shape(folded)
    for Nk, _ in sizes(d):
        q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
        kr, vr = (t.repeat_interleave(H // Hk, dim=1).contiguous() for t in (k, v))
        O, L = oracle_forward_batched(oracle, q, kr, vr, causal=True)
        check_o_lse(*fa.flash_forward_splitkv(q, k, v, num_splits=SPLITS, causal=True), O, L, f"{Nk} keys")
