"""The library's own split counts of launches of few rows: where the form takes fewer splits than the estimate, and where it leaves the estimate's
count.  No GPU needed."""
from launch_recorder import call, record

ROWS = 1 << 12

# B, H, Hk, Nq, Nk, d -> splits, form of few rows
CASES = [
    (1, 32, 8, 1, 1920, 64, 8, True), (8, 16, 2, 1, 1739, 64, 14, False),       # d = 64, 256 keys per split: four rows, eight splits and merged in the launch
    (1, 64, 8, 4, 1728, 64, 14, False), (4, 8, 2, 1, 3587, 64, 29, False),
    (6, 8, 1, 1, 31104, 64, 31, True), (8, 64, 8, 1, 5941, 64, 8, False),       # one work-group per CU by the estimate, or two
    (13, 32, 4, 1, 5210, 96, 9, False), (12, 16, 4, 1, 4992, 96, 5, True), (16, 16, 4, 1, 4992, 96, 4, True), (9, 16, 2, 1, 4992, 96, 13, True),
    (4, 32, 8, 1, 8192, 128, 8, True), (26, 16, 2, 1, 5656, 128, 4, True),      # other dimensions
    (9, 16, 2, 1, 24960, 40, 14, True), (2, 64, 8, 1, 12250, 80, 16, True), (6, 8, 2, 4, 5000, 32, 20, True),
    (1, 4, 4, 100, 6000, 31, 16, True), (2, 4, 4, 134, 9971, 31, 16, False),    # more than 32 rows, d < 32: 256 work-groups
    (1, 4, 4, 100, 6000, 32, 24, True),
    (8, 4, 1, 9, 1306, 128, 11, False), (1, 4, 4, 50, 3072, 128, 24, False), (3, 2, 2, 48, 5300, 128, 21, True), (1, 4, 4, 65, 3072, 128, 12, True),  # two row blocks, 256 keys
]


def test_counts():
    found = [(r["splits"], bool(r["launches"][0]["variant"] & ROWS)) for r in
             record([dict(call(*c[:6], num_splits=0), entry="splitkv", is_causal=int(c[3] > 1)) for c in CASES])]
    assert found == [c[6:] for c in CASES], [(c, f) for c, f in zip(CASES, found) if f != c[6:]]
