"""Who merges the partial results of launches of few rows: a launch of its own has one row per work-group and takes four waves for it from
17 splits on, whatever the split launch looked like."""
import pytest

from launch_recorder import call, record

COUNTERS = dict(split_counters=0xB00000, split_counters_len=4096)


# rows of a slice: heads of a K/V head, folded heads, rows of one head
@pytest.mark.parametrize("given", [{}, COUNTERS], ids=["no counters", "counters"])
def test_waves_behind_the_split_launch(given):
    cases = [(1, 32, 8, 1, 32768, 128, 32), (6, 4, 1, 1, 12288, 80, 32), (2, 32, 4, 1, 26396, 32, 30), (1, 32, 8, 1, 10048, 100, 27), (4, 16, 8, 3, 7000, 96, 18),
             (3, 4, 4, 8, 10881, 100, 18), (3, 4, 4, 8, 10881, 100, 17), (4, 4, 4, 17, 9000, 128, 16), (8, 16, 8, 6, 3000, 64, 12)]
    for c, r in zip(cases, record([dict(call(*c[:6], num_splits=c[6]), entry="splitkv", **given) for c in cases])):
        B, H, Hk, Nq, Nk, d, S = c
        assert r["rc"] == 0 and len(r["launches"]) == 2, (c, r)
        merge = r["launches"][1]
        waves = 4 if merge["split_count"] > 16 else 1
        assert f"combine_kernelILi{waves}E" in merge["kernel"] and merge["groups"] == (B * H * Nq if waves == 4 else -(-B * H * Nq // 4)), (c, merge)
