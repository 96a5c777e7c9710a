"""The native front end of the binding (csrc/py_binding.cpp) against binding.py's own path, which the debug outputs take:
same kernels, so bit-identical results whatever way the arguments come."""
import os
import shutil
import subprocess
import sys
import types

import pytest

from helpers import randn_f16_gpu


def _call(fa, entry, tensors, **kw):
    return (fa.flash_forward if entry == "forward" else fa.flash_forward_splitkv)(*tensors, **kw)


@pytest.mark.gpu
@pytest.mark.parametrize("entry,Nq,kw", [
    ("forward", 70, dict()),
    ("forward", 70, dict(softmax_scale=1, window=(40, 7))),
    ("forward", 70, dict(causal=1, alibi=True, dropout_p=0.25, seed=-3, offset=2 ** 40)),
    ("splitkv", 1, dict(num_splits=3)),
    ("splitkv", 1, dict()),
    ("splitkv", 33, dict(num_splits=4, causal=True, softmax_scale=0.2)),
])
@pytest.mark.parametrize("own_buffers", [False, True])
def test_matches_the_binding_s_own_path(fa, entry, Nq, kw, own_buffers):
    import torch

    # three key tiles unsplit: fewer than the narrow instances take, whose sums have another order and which a hint turns off
    Nk = 180 if entry == "forward" else 500
    q, k, v = randn_f16_gpu((2, 4, Nq, 40), 1), randn_f16_gpu((2, 2, Nk, 40), 2), randn_f16_gpu((2, 2, Nk, 40), 3)
    kw = dict(kw)
    if kw.pop("alibi", False):
        kw["alibi_slopes"] = torch.tensor([0.5, 0.25, 0.125, 0.0625], device="cuda")
    # a kernel hint keeps the call on the binding's own path
    o0, l0 = _call(fa, entry, (q, k, v), kernel_hint=fa.KERNEL_8WAVE, **kw)
    extra = {}
    if own_buffers:
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        extra = dict(out=torch.empty_like(o0), lse=torch.empty_like(l0), stream=s)
        if entry == "splitkv":
            extra["workspace"] = (torch.empty(2 * 4 * 8 * Nq * 40, device="cuda"), torch.empty(2 * 4 * 8 * Nq, device="cuda"))
    front = fa.binding._front_end()
    seen = []
    real = fa.binding._native

    class Spy:
        def __getattr__(self, name):
            def f(*a):
                r = getattr(front, name)(*a)
                seen.append(r is not NotImplemented)
                return r
            return f

    fa.binding._native = Spy()
    try:
        o1, l1 = _call(fa, entry, (q, k, v), **extra, **kw)
    finally:
        fa.binding._native = real
    torch.cuda.synchronize()
    assert seen == [True]
    if entry == "forward":  # (a hint can change the automatic split count and with it the rounding)
        assert torch.equal(o0, o1) and torch.equal(l0, l1)
    else:
        torch.testing.assert_close(o1, o0, rtol=2e-3, atol=2e-3)  # fp16 result, two roundings of at most 2^-11 each
        torch.testing.assert_close(l1, l0, rtol=0, atol=1e-5)
    if own_buffers:
        assert o1 is extra["out"] and l1 is extra["lse"]


def test_leaves_what_it_cannot_serve_to_the_binding(fa):
    import torch

    z = torch.zeros(1, 1, 2, 8)
    front = fa.binding._front_end()
    rest = (None, False, (-1, -1), None, 0.0, 0, 0, None, None, None)
    assert front.forward(z, z, z, *rest) is NotImplemented
    assert front.splitkv(z, z, z, 0, None, *rest) is NotImplemented
    assert front.forward(z) is NotImplemented
    with pytest.raises(ValueError, match="fp16"):
        fa.flash_forward(z, z, z)
    with pytest.raises(ValueError, match="fp16"):
        fa.flash_forward_splitkv(z, z, z)


CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash_attn_amd", "csrc")
DRIVER = os.path.join(os.path.dirname(os.path.abspath(__file__)), "driver")


def _dry_run(*args):
    r = subprocess.run(["make", "-n", "-C", CSRC, *args], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    return r.stdout


def test_the_library_builds_without_python():
    assert "flash_api.hip" in (out := _dry_run("-B", "PYTHON=false")) and "py_binding.cpp" not in out


@pytest.mark.parametrize("folder,target", [(CSRC, "build/fwd_d64.o"), (DRIVER, "mfma_rate")])
def test_a_failed_compilation_fails_the_build(tmp_path, folder, target):
    """Also where the result of an earlier build is there: it does not stand in for the one that was not made."""
    tree = tmp_path / "flash_attn_amd" / "csrc"
    shutil.copytree(folder, tree, ignore=shutil.ignore_patterns("*.o"))
    (tmp_path / "include").mkdir()
    (tmp_path / "include" / "flash_attn_mi355.h").touch()
    (tree / "build").mkdir(exist_ok=True)
    (tree / target).touch(0o777)
    os.utime(tree / target, (1, 1))
    r = subprocess.run(["make", "-C", str(tree), target, "HIPCC=false"], capture_output=True, text=True, timeout=120)
    assert r.returncode != 0, r.stdout


def test_the_front_end_is_rebuilt_for_another_torch():
    import torch

    version = os.path.join(os.path.dirname(torch.__file__), "version.py")
    settled = [x for f in ("../../include/flash_attn_mi355.h", "py_binding.cpp", "split_counters.h") for x in ("-o", f)]
    assert "py_binding.cpp" not in _dry_run("native", *settled, "-o", version)
    assert "py_binding.cpp" in _dry_run("native", *settled, "-W", version)


def test_counters_of_streams(tmp_path):
    exe = str(tmp_path / "split_counters_test")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-I", CSRC, os.path.join(os.path.dirname(__file__), "split_counters_test.cpp"),
                           "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("found", [None, types.SimpleNamespace(torch_version="1.0.0")])  # not built | built for another torch
def test_calls_are_served_without_the_front_end(fa, monkeypatch, found):
    import flash_attn_amd
    import torch

    monkeypatch.setitem(sys.modules, "flash_attn_amd._native", found)
    monkeypatch.delattr(flash_attn_amd, "_native", raising=False)
    if found is not None:
        monkeypatch.setattr(flash_attn_amd, "_native", found, raising=False)
    monkeypatch.setattr(fa.binding, "_native", None)
    z = torch.zeros(1, 1, 2, 8)
    with pytest.warns(RuntimeWarning, match="make -C flash_attn_amd/csrc native"), pytest.raises(ValueError, match="fp16"):
        fa.flash_forward(z, z, z)
    with pytest.raises(ValueError, match="fp16"):  # (and says so once)
        fa.flash_forward_splitkv(z, z, z)


@pytest.mark.gpu
def test_results_without_the_front_end(fa, monkeypatch):
    import torch

    q, k, v = randn_f16_gpu((2, 4, 70, 40), 1), randn_f16_gpu((2, 2, 900, 40), 2), randn_f16_gpu((2, 2, 900, 40), 3)
    with_it = fa.flash_forward(q, k, v, causal=True) + fa.flash_forward_splitkv(q, k, v)
    monkeypatch.setattr(fa.binding, "_native", fa.binding._NoFrontEnd)
    without = fa.flash_forward(q, k, v, causal=True) + fa.flash_forward_splitkv(q, k, v)
    assert all(torch.equal(a, b) for a, b in zip(with_it, without))


@pytest.mark.gpu
def test_allocations_are_seen_by_those_who_look(fa):
    """A dispatch mode sees results and workspace being allocated, and deterministic mode fills them."""
    import torch
    from torch.utils._python_dispatch import TorchDispatchMode

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            if func is torch.ops.aten.empty.memory_format:
                sizes.append(tuple(args[0]))
            return func(*args, **(kwargs or {}))

    q, k, v = randn_f16_gpu((1, 2, 3, 40), 1), randn_f16_gpu((1, 2, 500, 40), 2), randn_f16_gpu((1, 2, 500, 40), 3)
    sizes = []
    want = fa.flash_forward(q, k, v), fa.flash_forward_splitkv(q, k, v, num_splits=2)
    with Watch():
        got = fa.flash_forward(q, k, v), fa.flash_forward_splitkv(q, k, v, num_splits=2)
    assert sizes == [(1, 2, 3, 40), (1, 2, 3), (1, 2, 3, 40), (1, 2, 3), (2 * 2 * 3 * 40,), (2 * 2 * 3,)]
    assert all(torch.equal(a, b) for w, g in zip(want, got) for a, b in zip(w, g))
    before = torch.utils.deterministic.fill_uninitialized_memory
    front, rest = fa.binding._front_end(), (None, False, (-1, -1), None, 0.0, 0, 0, None, None, None)
    torch.use_deterministic_algorithms(True)
    try:
        for torch.utils.deterministic.fill_uninitialized_memory in (True, False):
            served = front.forward(q, k, v, *rest) is not NotImplemented
            assert served != torch.utils.deterministic.fill_uninitialized_memory
            assert torch.equal(fa.flash_forward(q, k, v)[0], want[0][0])
    finally:
        torch.use_deterministic_algorithms(False)
        torch.utils.deterministic.fill_uninitialized_memory = before


@pytest.mark.gpu
def test_first_call_on_a_stream_while_another_is_captured(fa):
    """Split calls on streams that have not been used yet, issued inside a capture of the current stream: they run beside it,
    and the captured graph is whole."""
    import torch

    q, k, v = randn_f16_gpu((1, 2, 1, 64), 1), randn_f16_gpu((1, 2, 3000, 64), 2), randn_f16_gpu((1, 2, 3000, 64), 3)
    want = fa.flash_forward_splitkv(q, k, v, num_splits=4)
    captured = torch.cuda.Stream()
    # (torch deals out 32 streams in turn: all of them but the captured one)
    sides = [s for s in (torch.cuda.Stream() for _ in range(32)) if s.cuda_stream != captured.cuda_stream]
    bufs = [(torch.zeros_like(want[0]), torch.zeros_like(want[1]), (torch.empty(4 * 2 * 64, device="cuda"), torch.empty(4 * 2, device="cuda")))
            for _ in sides]
    x = torch.ones(1000, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=captured):
        y = x + 1
        for s, (o, lse, ws) in zip(sides, bufs):
            fa.flash_forward_splitkv(q, k, v, num_splits=4, stream=s, out=o, lse=lse, workspace=ws)
        z = y * 2
    torch.cuda.synchronize()
    assert all(torch.equal(o, want[0]) and torch.equal(lse, want[1]) for o, lse, _ in bufs)
    for i in range(3):
        x.fill_(i)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, torch.full_like(z, 2.0 * (i + 1)))


@pytest.mark.gpu
def test_counters_on_two_streams_at_once(fa):
    """Decode calls that merge in the split launch, many of them in flight on each of two streams."""
    import torch

    shapes = [(2, 3, 2500, 64, 8), (1, 4, 9000, 128, 40)]
    sets, wants = [], []
    for i, (B, H, Nk, d, S) in enumerate(shapes):
        t = randn_f16_gpu((B, H, 1, d), 3 * i), randn_f16_gpu((B, H, Nk, d), 3 * i + 1), randn_f16_gpu((B, H, Nk, d), 3 * i + 2)
        sets.append((t, S))
        wants.append(fa.flash_forward_splitkv(*t, num_splits=S))
    streams = [torch.cuda.Stream() for _ in shapes]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(50):
        for i, ((t, S), s) in enumerate(zip(sets, streams)):
            with torch.cuda.stream(s):
                got[i].append(fa.flash_forward_splitkv(*t, num_splits=S))
    torch.cuda.synchronize()
    for want, results in zip(wants, got):
        assert all(torch.equal(o, want[0]) and torch.equal(lse, want[1]) for o, lse in results)
