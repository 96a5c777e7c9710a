"""flash_params::split_counters: a decode launch that merges its own partial results gives bit by bit what the separate
merge gives and leaves the counters zero, whatever the split count (one wave or four per row), row alignment and number of
query heads per work-group, call after call on the same counters."""
import ctypes as C

import pytest

from helpers import randn_f16_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 100, 31, 128])
@pytest.mark.parametrize("G", [1, 2, 3, 4, 8])
def test_merge_in_the_split_kernel(fa, G, d):
    import torch
    from flash_attn_amd import binding

    B, Hk, Nk = 2, 3, 9000
    H = Hk * G
    q, k, v = randn_f16_gpu((B, H, 1, d), 1), randn_f16_gpu((B, Hk, Nk, d), 2), randn_f16_gpu((B, Hk, Nk, d), 3)
    slopes = torch.linspace(0.001, 0.01, H, device="cuda") if G >= 4 else None  # (without a bias the heads are rows of a tile)
    counters = torch.zeros(B * H, dtype=torch.int32, device="cuda")
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for S in (2, 16, 17, 33, 70):
        res = []
        for given in (0, B * H, B * H - 1):  # none, enough, too few
            o = torch.empty_like(q)
            lse = torch.empty((B, H, 1), device="cuda")
            ws = torch.full((B * H * S * d,), float("nan"), device="cuda"), torch.full((B * H * S,), float("nan"), device="cuda")
            p = binding.make_params(q, k, v, o, lse, None, False, (-1, -1), slopes, 0.0, 0, 0, S, *ws)
            p.split_counters, p.split_counters_len = (counters.data_ptr() if given else None), given
            for _ in range(3):
                assert fa.lib().flash_forward_splitkv(C.byref(p), stream) == 0
            torch.cuda.synchronize()
            assert not counters.any()
            res.append((o, lse))
        for o, lse in res[1:]:
            assert torch.equal(o, res[0][0]) and torch.equal(lse, res[0][1]), f"S {S}"
        assert torch.isfinite(res[0][0]).all()
