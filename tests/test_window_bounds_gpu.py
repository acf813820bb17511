"""Window bounds as large as the type: they mask nothing, in every kernel form.  (Kernels add bounds to positions in 32 bits.)"""
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
FAR = 2 ** 31 - 1


def _close(a, b):
    # the same products in the same tiles; a kernel chosen for windows may sum in another order: 2^-8 of the largest entry
    return (a.float() - b.float()).abs().max() <= 4 * 2.0 ** -8 * b.float().abs().max()


@pytest.mark.parametrize("far", [(FAR, FAR), (FAR, -1), (-1, FAR), (FAR, 0)])
@pytest.mark.parametrize("b,s,h,d", [(2, 300, 4, 64), (20, 200, 8, 64), (2, 300, 4, 128), (2, 300, 2, 192), (2, 300, 2, 256), (2, 40, 4, 128)])
def test_far_bounds_mask_nothing(b, s, h, d, far):
    import flash_attn
    print("far bounds", b, s, h, d, far, flush=True)
    sys.stdout.flush()
    g = torch.Generator().manual_seed(s + d)
    q, k, v, dout = [torch.randn(b, s, h, d, generator=g).to(torch.bfloat16).to(DEV).requires_grad_() for _ in range(4)]
    near = (-1, 0) if far[1] == 0 else (-1, -1)
    res = []
    for window in (far, near):
        out = flash_attn.flash_attn_func(q, k, v, window_size=window)
        res.append((out,) + torch.autograd.grad(out, (q, k, v), dout.detach()))
    assert all(_close(x, y) for x, y in zip(*res))


@pytest.mark.parametrize("sq", [1, 4, 130])
def test_far_bounds_over_a_cache(sq):
    import flash_attn
    print("far bounds, cache", sq, flush=True)
    g = torch.Generator().manual_seed(sq)
    q, kc, vc = [torch.randn(3, n, 8, 64, generator=g).to(torch.bfloat16).to(DEV) for n in (sq, 700, 700)]
    lens = torch.tensor([200, 333, 700], dtype=torch.int32, device=DEV)
    outs = [flash_attn.flash_attn_with_kvcache(q, kc, vc, cache_seqlens=lens, window_size=w) for w in ((FAR, FAR), (-1, -1))]
    assert _close(*outs)
