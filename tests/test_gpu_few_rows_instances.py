"""Launches of few rows, heads shorter than their bucket: the instance goes by row length and alignment as in the other forms.  Against the
oracle."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu
from launch_recorder import FOLD, FULL_D, NARROW, VEC, call, record

SHORT, ROWS, MANY_ROWS = 1 << 11, 1 << 12, 1 << 13
DIMS = [16, 31, 33, 40, 48, 56, 65, 72, 80, 88, 97, 100, 112, 120]
SPLITS = 8
SHAPES = [(2, 16, 16, 5), (2, 32, 16, 3), (1, 16, 16, 41), (1, 16, 8, 20)]  # B, H, Hk, Nq: up to 32 rows and more, the second and the last folded


def bucket(d):
    return -(-d // 32) * 32


@pytest.mark.parametrize("B,H,Hk,Nq", SHAPES)
def test_instances(B, H, Hk, Nq):
    wanted = []
    for d in DIMS:
        bits = NARROW | ROWS | (FOLD if Hk < H else 0) | (MANY_ROWS if Nq * (H // Hk) > 32 or d < 32 else 0)
        if d > 32:
            bits |= (VEC if d % 8 == 0 else 0) | (SHORT if Hk == H and d <= bucket(d) - 16 else 0)
        wanted.append(bits)
    found = [r["launches"][0]["variant"] for r in record([call(B, H, Hk, Nq, 2000, d, num_splits=SPLITS) for d in DIMS])]
    assert found == wanted, list(zip(DIMS, found, wanted))


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,Nq", SHAPES)
@pytest.mark.parametrize("d", DIMS)
def test_few_rows_of_shorter_heads(fa, oracle, d, B, H, Hk, Nq):
    Nk = 2000  # a last tile of 16 keys
    q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
    kr, vr = (t.repeat_interleave(H // Hk, dim=1).contiguous() for t in (k, v))
    O, L = oracle_forward_batched(oracle, q, kr, vr, causal=True)
    check_o_lse(*fa.flash_forward_splitkv(q, k, v, num_splits=SPLITS, causal=True), O, L)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [31, 40, 64, 96, 100, 128])
def test_last_split_of_one_key(fa, oracle, d):
    B, H, Nq, Nk, S = 3, 16, 32, 3 * 384 + 1, 4
    r, = record([dict(call(B, H, H, Nq, Nk, d, causal=True, num_splits=S), entry="splitkv")])
    assert r["launches"][0]["variant"] & ROWS and r["splits"] == S
    q, k, v = randn_f16_gpu((B, H, Nq, d), 1), randn_f16_gpu((B, H, Nk, d), 2), randn_f16_gpu((B, H, Nk, d), 3)
    O, L = oracle_forward_batched(oracle, q, k, v, causal=True)
    check_o_lse(*fa.flash_forward_splitkv(q, k, v, num_splits=S, causal=True), O, L)
