"""Which launches are paired at the edges of the rule: five or six tiles, and dropout with 325 to 384 work-groups.  No GPU needed."""
from launch_recorder import call, form, record

# B, H, N, d, p, keywords, form
CASES = [
    (1, 32, 320, 64, 0.0, dict(causal=True, alibi=True), "plain"), (1, 32, 321, 64, 0.0, dict(causal=True, alibi=True), "paired"),    # ALiBi, no window that cuts
    (6, 8, 320, 96, 0.0, dict(window=(300, 0), alibi=True), "plain"), (1, 30, 300, 80, 0.0, dict(window=(135, 0), alibi=True), "paired"),
    (3, 8, 900, 112, 0.0, dict(window=(192, 0)), "plain"), (3, 8, 900, 112, 0.0, dict(window=(193, 0)), "paired"),                    # 192 work-groups: 5 | 6 tiles
    (2, 8, 900, 112, 0.0, dict(window=(192, 0)), "paired"), (3, 8, 900, 96, 0.0, dict(window=(192, 0)), "paired"),                    # 128; other buckets
    (7, 8, 704, 128, 0.2, dict(causal=True), "plain"), (6, 9, 704, 128, 0.2, dict(causal=True), "paired"),                            # 336 | 324 work-groups
    (6, 8, 895, 80, 0.1, dict(causal=True), "plain"), (6, 8, 896, 80, 0.1, dict(causal=True), "paired"), (7, 8, 704, 64, 0.2, dict(causal=True), "paired"),
]


def test_forms():
    found = [form(r["launches"][0]) for r in record([call(B, H, H, N, N, d, p, **kw) for B, H, N, d, p, kw, _ in CASES])]
    assert found == [c[-1] for c in CASES], [(c, f) for c, f in zip(CASES, found) if f != c[-1]]
