"""The native front end of the binding (csrc/py_binding.cpp) against binding.py's own path, which the debug outputs take:
same kernels, so bit-identical results whatever way the arguments come."""
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
