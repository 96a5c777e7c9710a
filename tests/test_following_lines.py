"""Causal launches of 417 to 512 work-groups: the lines from which on they are paired, one key below and at each, both launches inside the range of work-groups
that the line is for.  No GPU needed."""
from launch_recorder import call, form, record

# H, keys at the line, d (one sequence; H ceil(N / 128) work-groups)
LINES = [(33, 1856, 64), (33, 1856, 40), (34, 1856, 31), (31, 1856, 96), (32, 1856, 88), (33, 1760, 80), (35, 1760, 72), (34, 1856, 112)]


def test_lines():
    calls = [call(1, H, H, n, n, d, causal=True) for H, N, d in LINES for n in (N - 1, N)]
    groups = [c["H"] * -(-c["Nq"] // 128) for c in calls]
    assert all(416 < g <= 512 for g in groups) and groups[::2] == groups[1::2], groups
    forms = [form(r["launches"][0]) for r in record(calls)]
    assert forms == ["plain", "paired"] * len(LINES), list(zip(calls, forms))
