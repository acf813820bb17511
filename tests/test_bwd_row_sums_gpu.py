"""softmax_d = rowsum(dout * out), which the dQ pass leaves behind: every row of it, also those that a sequence does not have."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _poison(*shape):
    """so that memory that nobody writes is likely to hold something else than zero"""
    torch.full(shape, float("nan"), dtype=torch.float32, device=DEV)


@pytest.mark.parametrize("d,dtype", [(32, torch.float16), (80, torch.bfloat16), (128, torch.bfloat16), (160, torch.bfloat16), (192, torch.float16), (256, torch.bfloat16)])
@pytest.mark.parametrize("sq", [1, 127, 128, 129, 300])
def test_dense(d, dtype, sq):
    from flash_attn import _native as nat
    gen = torch.Generator().manual_seed(sq + d)
    mk = lambda *s: torch.randn(*s, generator=gen).to(dtype).to(DEV)
    b, h, hk, sk = 2, 4, 2, 200
    q, k, v, do = mk(b, sq, h, d), mk(b, sk, hk, d), mk(b, sk, hk, d), mk(b, sq, h, d)
    r = nat.fwd(q, k, v, None, 0.0, d ** -0.5, True, -1, -1, False, None)
    _poison(b, h, (sq + 127) // 128 * 128)
    sd = nat.bwd(do, q, k, v, r[0], r[5], None, None, None, 0.0, d ** -0.5, True, -1, -1, None, None)[3]
    want = (do.double() * r[0].double()).sum(-1).permute(0, 2, 1)
    # sums of d products in 32 bits: d half-ulps of the largest partial sum, which the sum of magnitudes bounds
    bound = d * 2.0 ** -24 * (do.double() * r[0].double()).abs().sum(-1).permute(0, 2, 1)
    assert ((sd[:, :, :sq].double() - want).abs() <= bound + 1e-30).all()
    assert not sd[:, :, sq:].any()


@pytest.mark.parametrize("d", [128, 256])
def test_packed(d):
    from flash_attn import _native as nat
    gen = torch.Generator().manual_seed(d)
    lens, h, hk = [130, 0, 300, 1], 4, 2
    total, mx = sum(lens), 500
    mk = lambda *s: torch.randn(*s, generator=gen).to(torch.bfloat16).to(DEV)
    q, k, v, do = mk(total, h, d), mk(total, hk, d), mk(total, hk, d), mk(total, h, d)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(DEV)
    r = nat.varlen_fwd(q, k, v, None, cu, cu, mx, mx, 0.0, d ** -0.5, False, True, -1, -1, False, None)
    _poison(4, h, 512)
    sd = nat.varlen_bwd(do, q, k, v, r[0], r[5], None, None, None, cu, cu, mx, mx, 0.0, d ** -0.5, False, True, -1, -1, None, None)[3]
    at = 0
    for i, n in enumerate(lens):
        x, y = do[at:at + n].double(), r[0][at:at + n].double()
        at += n
        assert ((sd[i, :, :n].double() - (x * y).sum(-1).T).abs() <= d * 2.0 ** -24 * (x * y).abs().sum(-1).T + 1e-30).all()
        assert not sd[i, :, n:].any()
