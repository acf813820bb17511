"""Which of the two long forward kernels a launch takes at head dim 65..128: the fill of the last round, the window's span."""
import pytest
import torch

from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("b,h,hk,sq,sk,d,window,dropout,kernel", [
    (1, 64, 8, 1024, 1024, 128, (-1, -1), 0.0, "pingpong"),        # 256 blocks of 256 rows: one full round
    (1, 52, 4, 1030, 1001, 128, (-1, -1), 0.0, "pipelined"),       # 260
    (1, 96, 8, 1024, 800, 72, (-1, -1), 0.0, "pipelined"),         # 384: half a round
    (1, 97, 1, 1024, 800, 128, (-1, -1), 0.0, "pingpong"),         # 388: more than half
    (3, 70, 10, 513, 1025, 128, (-1, -1), 0.0, "pipelined"),       # 630: the third round
    (7, 64, 8, 290, 1024, 96, (-1, -1), 0.1, "pipelined"),         # 896: half of the fourth
    (1, 20, 5, 4096, 4096, 128, (-1, -1), 0.0, "pipelined"),       # 320, long keys: up to a quarter of a round
    (1, 24, 6, 4096, 4096, 128, (-1, -1), 0.0, "pingpong"),        # 384
    (1, 24, 6, 4096, 4096, 80, (-1, -1), 0.0, "pipelined"),
    (1, 40, 8, 2304, 2304, 128, (1000, 24), 0.0, "pipelined"),     # a span of 1024
    (1, 40, 8, 2304, 2304, 128, (1000, 25), 0.0, "pingpong"),
    (2, 41, 1, 2050, 2048, 128, (1024, 0), 0.0, "pingpong"),       # 738 blocks
    (2, 41, 1, 2050, 2048, 96, (1024, 0), 0.0, "pipelined"),
])
def test_long_kernel_of_a_launch(b, h, hk, sq, sk, d, window, dropout, kernel):
    from flash_attn import _native as nat
    from flash_attn import flash_attn_func
    gen = torch.Generator().manual_seed(h + sq)
    q, k, v = (torch.randn(b, s, n, d, generator=gen).to(torch.bfloat16) for s, n in ((sq, h), (sk, hk), (sk, hk)))
    out, lse, mask = flash_attn_func(q.to(DEV), k.to(DEV), v.to(DEV), dropout_p=dropout, window_size=window, return_attn_probs=True)
    assert nat.last_kernel()[0] == kernel
    for i, j in ((0, 0), (b - 1, h - 1)):
        cut = lambda t, n: t[i:i + 1, :, n:n + 1]
        qq, kk, vv = cut(q, j), cut(k, j // (h // hk)), cut(v, j // (h // hk))
        kw = dict(window_size=window)
        if dropout:
            kw.update(dropout_p=dropout, dropout_mask=(mask[i:i + 1, j:j + 1, :sq, :sk] >= 0).cpu())
        o_ref, l_ref, o_pt = orc.attention_reference_pair(qq, kk, vv, **kw)
        ok, err, bound = orc.tolerance_ok(cut(out.cpu(), j), o_ref, o_pt, 2.0, 1e-5)
        assert ok, (err, bound)
        assert orc.lse_ok(lse[i:i + 1, j:j + 1].cpu(), l_ref)[0]
