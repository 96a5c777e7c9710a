"""What the library launches against the buffers it told the caller to bring, without a GPU (tests/launch_recorder.py)."""
import numpy as np

from launch_recorder import ALIBI, DROPOUT, EVERY, FOLD, FULL_D, KV_ONCE, NARROW, PAIR, STAMP, call, form, record

STAMPS = 0x900000  # a stage-stamp buffer


def random_calls(seed, n, **fixed):
    """Calls of both entry points over every head-dim bucket, mask, feature and kernel hint, few and many rows, grouped heads."""
    rng = np.random.default_rng(seed)
    calls = []
    while len(calls) < n:
        Hk = int(rng.choice([1, 2, 4, 8]))
        B, H = int(rng.integers(1, 30)), Hk * int(rng.choice([1, 1, 2, 3, 4, 8]))
        Nq = int(rng.choice([int(rng.integers(2, 70)), int(rng.integers(1, 600)), int(rng.integers(100, 5000))]))
        Nk = Nq if rng.random() < 0.3 else int(round(2 ** rng.uniform(4, 15)))
        c = dict(entry=str(rng.choice(["forward", "splitkv"])), B=B, H=H, H_kv=Hk, Nq=Nq, Nk=Nk,
                 d=int(rng.choice([7, 31, 32, 40, 64, 64, 72, 96, 100, 128, 128])), is_causal=int(rng.integers(0, 2)),
                 num_splits=int(rng.choice([0, 0, 1, 4, 17])))
        if rng.random() < 0.3:
            c.update(window_left=int(rng.integers(0, 2000)), window_right=int(rng.choice([-1, 0, 100])))
        if rng.random() < 0.2:
            c.update(alibi_slopes=0xA00000)
        if rng.random() < 0.2:
            c.update(dropout_p=float(rng.choice([0.1, 1e-6])), seed=3)
        if rng.random() < 0.2:
            c.update(kernel_hint=int(rng.integers(1, 3)))
        if rng.random() < 0.05:
            c.update(softmax_scale=-0.1)
        c.update(fixed)
        calls.append(c)
    return calls


def split_rows(c, r):
    """Rows of partial results that the launches write, over the split count that the combine step was given."""
    S = max(launch["split_count"] for launch in r["launches"])
    return c["B"] * c["H"] * c["Nq"] * S if S > 1 else 0


def test_workspace_does_not_depend_on_the_stage_stamps():
    """The workspace is sized before the stamp buffer is there, and the launch that sees the buffer needs no more of it."""
    calls = random_calls(1, 1500, entry="splitkv", num_splits=0, stage_stamps_out=STAMPS)
    calls.append(dict(entry="splitkv", B=14, H=64, H_kv=8, Nq=36, Nk=27335, d=128, num_splits=0, stage_stamps_out=STAMPS))
    split = 0
    for c, r in zip(calls, record(calls)):
        assert r["rc"] == 0, c
        rows = split_rows(c, r)
        split += rows > 0
        assert r["workspace"] == [rows * c["d"] * 4, rows * 4], c
    assert split > 150  # (the sample is of the kind that it is about)


def test_stage_stamp_buffer_holds_every_work_group():
    """FLASH_STAMP_WORDS words for each work-group of the tiled launch, whichever entry point and route: heads folded into the
    rows of one problem among them."""
    calls = random_calls(2, 3000, stage_stamps_out=STAMPS)
    calls.append(dict(entry="splitkv", B=4, H=32, H_kv=8, Nq=16, Nk=8192, d=128, num_splits=8, stage_stamps_out=STAMPS))
    for c, r in zip(calls, record(calls)):
        assert r["rc"] == 0, c
        first = r["launches"][0]
        groups = first["groups"] if first["variant"] is not None else 0  # (the decode stream is not stamped)
        assert r["stamp_bytes"] == groups * 9 * 8, (c, r)


def test_stage_stamps_do_not_change_the_launch():
    """A stamped call runs the instrumented twin of the instance that the call without stamps runs, on the same grid."""
    calls = random_calls(3, 3000) + [dict(entry="forward", B=32, H=32, Nq=512, Nk=512, d=64)]
    seen = set()
    for c, plain, stamped in zip(calls, record(calls), record([dict(c, stage_stamps_out=STAMPS) for c in calls])):
        assert len(plain["launches"]) == len(stamped["launches"])
        for a, b in zip(plain["launches"], stamped["launches"]):
            if a["variant"] is not None:
                assert b["variant"] == a["variant"] | STAMP, (c, a, b)
                kind = "pp" if "_pp_" in a["kernel"] else a["kernel"].split("ELi")[1]  # (the other argument: 2 = tall)
                seen.add((kind, a["variant"] & (EVERY | NARROW | FOLD | PAIR)))
            assert (b["groups"], b["threads"]) == (a["groups"], a["threads"]), (c, a, b)
    assert {("1", 0), ("2", 0), ("pp", 0), ("1", EVERY), ("1", NARROW), ("1", FOLD), ("1", PAIR), ("1", NARROW | FOLD),
            ("1", PAIR | FOLD)} <= seen


def test_workspace_helper_covers_the_calls_it_knows_nothing_of(fa):
    """workspace_bytes() of a shape is enough for the launch whatever the call's features are, and so is the size for the
    features that it is given."""
    calls = [c for c in random_calls(4, 3000, entry="splitkv", num_splits=0) if c.get("dropout_p") != 1e-6]
    for Nq in range(2, 65):  # rows whose heads are folded unless a feature keeps them apart
        for feature in (dict(), dict(alibi_slopes=0xA00000), dict(dropout_p=0.1)):
            calls.append(dict(entry="splitkv", B=14, H=64, H_kv=8, Nq=Nq, Nk=27335, d=128, num_splits=0, **feature))
    calls += [dict(c, dropout_p=1e-6) for c in calls[:300]] + [dict(c, scores_out=0xB00000) for c in calls[:300]]
    for c, r in zip(calls, record(calls)):
        assert r["rc"] == 0, c
        rows = split_rows(c, r)
        shape = [c[x] for x in ("B", "H", "Nq", "Nk", "d")]
        kw = dict(causal=c.get("is_causal", 0), window=(c.get("window_left", -1), c.get("window_right", -1)), H_kv=c["H_kv"],
                  kernel_hint=c.get("kernel_hint", 0))
        ob, lb = fa.workspace_bytes(*shape, **kw)
        assert ob >= rows * c["d"] * 4 and lb >= rows * 4, c
        alibi, p = "alibi_slopes" in c, c.get("dropout_p", 0.0)
        ob, lb = fa.workspace_bytes(*shape, alibi=alibi, dropout_p=p, **kw)
        assert ob >= rows * c["d"] * 4 and lb >= rows * 4, c
        if p != 1e-6 and c.get("softmax_scale", 1) > 0 and "scores_out" not in c:
            assert fa.resolve_splits(*shape, alibi=alibi, dropout_p=p, **kw) == r["splits"], c


def test_combine_launch_fits_a_grid_up_to_2_to_the_26_rows():
    """More than 16 splits take a work-group per row up to the 2^32 threads of a launch, and a wave per row beyond."""
    for Nq, S, waves in ((4096, 17, 4), (2 ** 24 - 1, 17, 4), (2 ** 24, 17, 1), (2 ** 24, 16, 1), (2 ** 26 - 4, 20, 1)):
        r, = record([dict(entry="splitkv", B=1, H=1, Nq=Nq, Nk=128 * S, d=8, num_splits=S)])
        assert r["rc"] == 0, (Nq, S, r)
        assert f"combine_kernelILi{waves}E" in r["launches"][1]["kernel"] and r["launches"][1]["split_count"] == S


def test_non_temporal_requests_only_where_no_other_work_group_asks_for_the_tiles():
    """One row block per K/V head: K and V pass once, whether the rows are a head's own, folded heads or a decode launch's."""
    calls = random_calls(5, 3000)
    for G, Nq in ((2, 64), (4, 32), (4, 33), (8, 16), (8, 17), (16, 64)):  # 128 rows | more
        for d in (32, 64, 96, 128):
            for S in (1, 8):
                calls.append(dict(entry="splitkv", B=3, H=8 * G, H_kv=8, Nq=Nq, Nk=9000, d=d, num_splits=S))
    seen = set()
    for c, r in zip(calls, record(calls)):
        if r["rc"] != 0 or not r["launches"] or r["launches"][0]["variant"] is None or "_pp_" in r["launches"][0]["kernel"]:
            continue
        v, G = r["launches"][0]["variant"], c["H"] // c["H_kv"]
        heads_as_rows = v & FOLD or (c["Nq"] == 1 and G >= 4 and not c.get("alibi_slopes") and not c.get("dropout_p")
                                     and c.get("window_left", -1) < 0)
        once = (c["Nq"] * G if heads_as_rows else c["Nq"] if G == 1 else 1 << 30) <= 128
        may = v & FULL_D and not v & (NARROW | ALIBI | DROPOUT)
        assert bool(v & KV_ONCE) == bool(once and may), (c, r)
        seen.add((bool(v & FOLD), bool(v & KV_ONCE), bool(v & PAIR), bool(may)))
    assert {(True, True, False, True), (True, False, False, True), (True, False, True, True), (True, True, True, True)} <= seen


def test_launch_forms_of_the_gpu_tests():
    """The shapes of the GPU tests that are about a launch form are launched in that form."""
    import test_gpu_dropout_calls as calls_
    import test_gpu_edge_cases as edge
    import test_gpu_narrow_rule as narrow
    import test_gpu_paired_halves as paired
    import test_gpu_tall_blocks as tall

    rows = [("tall", call(*s, 64)) for s in tall.SHAPES + tall.CHUNKS]
    rows += [(f, call(B, H, H, N, N, d, **kw)) for B, H, N, d, kw, f in narrow.LINES]
    rows += [("narrow", call(*shape, p, **kw)) for *shape, p, kw in narrow.ROUNDS]
    rows += [(f, call(B, H, H, Nq, Nk, d, 0.3, **kw)) for B, H, Nq, Nk, d, kw, f in calls_.WALKS]
    rows += [("paired", call(B, H, H, N, N, d, causal=True)) for B, H, N, d in paired.UNSPLIT]
    rows += [("paired", call(B, H, H, N, N, d, 0.2, **kw)) for B, H, N, d, kw in paired.UNSPLIT_DROPOUT]
    rows += [("paired", call(1, 2, 2, Nq, 1740, d, 0.2, num_splits=3, causal=True, window=(390, -1))) for Nq, d in ((33, 128), (140, 100), (128, 64))]
    rows += [("paired", call(*s, causal=True)) for s in paired.FOLLOWING]
    for *shape, S, kw, f in edge.STAMPED_FORMS:
        kw = dict(kw)
        rows.append((f, call(*shape, kw.pop("dropout_p", 0.0), num_splits=S, **kw)))
    for *shape, kw in edge.NARROW_SHAPES:
        if shape[3] > 1:  # (one row: the decode kernel)
            kw = {k: v for k, v in kw.items() if k not in ("seed", "offset")}
            rows.append(("narrow", call(*shape, kw.pop("dropout_p", 0.0), **kw)))
    for (f, c), r in zip(rows, record([c for _, c in rows])):
        launch = r["launches"][0]
        assert form(launch) == f, (f, c, launch)
        assert bool(launch["variant"] & DROPOUT) == (c["dropout_p"] > 0.0), (c, launch)


def test_launches_that_are_whole_without_their_paired_form_need_no_workspace():
    """Whether to split is not a matter of the paired work-groups' price: a caller of such a shape brings no workspace."""
    shapes = [(1, 12, 12, 425, 6429, 64, 1, 0.0), (2, 16, 2, 436, 2828, 64, 1, 0.0), (4, 48, 12, 30, 3410, 64, 0, 0.0),
              (2, 1, 1, 3543, 4219, 128, 0, 0.1), (6, 24, 12, 28, 2283, 72, 0, 0.0), (7, 2, 2, 525, 5976, 128, 1, 0.0)]
    calls = [dict(entry="splitkv", B=B, H=H, H_kv=Hk, Nq=Nq, Nk=Nk, d=d, is_causal=c, dropout_p=p, num_splits=0)
             for B, H, Hk, Nq, Nk, d, c, p in shapes]
    calls.append(dict(entry="splitkv", B=3, H=3, Nq=996, Nk=996, d=40, window_left=1470, window_right=100, num_splits=0))
    for c, r in zip(calls, record(calls)):
        assert r["rc"] == 0 and r["splits"] == 1 and r["workspace"] == [0, 0] and len(r["launches"]) == 1, (c, r)
