"""Windows that end at the row: from how many key tiles on a launch is paired, one and two work-groups per CU, and launches at the
lines against the oracle."""
import pytest

from helpers import check_o_lse, oracle_forward_batched, randn_f16_gpu
from launch_recorder import call, form, record

# H, N, d, window, causal, p, form (one sequence)
CASES = [
    (16, 677, 64, (129, 0), False, 0.0, "paired"), (16, 677, 64, (128, 0), False, 0.0, "plain"),   # 4 | 5 tiles
    (17, 600, 112, (129, -1), True, 0.0, "paired"), (17, 600, 99, (128, 0), False, 0.0, "plain"),
    (16, 1025, 31, (200, 0), False, 0.0, "paired"), (32, 300, 96, (130, 0), False, 0.0, "paired"),
    (16, 677, 128, (383, 0), False, 0.0, "plain"), (16, 677, 128, (384, 0), False, 0.0, "paired"),  # d = 128: 8
    (16, 677, 64, (129, 0), False, 0.1, "plain"), (16, 677, 64, (129, 1), False, 0.0, "plain"),     # dropout, keys right of the row
    (40, 1241, 40, (257, 0), False, 0.0, "paired"), (40, 1241, 64, (256, 0), False, 0.0, "plain"),  # 257 to 400 work-groups: 6 | 7
    (40, 1280, 64, (300, 0), False, 0.0, "paired"), (41, 1280, 64, (300, 0), False, 0.0, "plain"),  # 400 | 410 of them
    (40, 1241, 72, (400, 0), False, 0.0, "plain"), (40, 1241, 32, (400, 0), False, 0.0, "plain"),
]


def test_forms():
    calls = [call(1, H, H, N, N, d, p, causal=causal, window=window) for H, N, d, window, causal, p, _ in CASES]
    assert [form(r["launches"][0]) for r in record(calls)] == [c[-1] for c in CASES]


@pytest.mark.gpu
@pytest.mark.parametrize("H,N,d,window,causal,p", [c[:-1] for c in CASES if c[-1] == "paired"])
def test_paired_windows(fa, oracle, H, N, d, window, causal, p):
    q, k, v = (randn_f16_gpu((1, H, N, d), s) for s in (4, 5, 6))
    O, L = oracle_forward_batched(oracle, q, k, v, causal=causal, window=window)
    check_o_lse(*fa.flash_forward(q, k, v, causal=causal, window=window), O, L, "paired, window")
