"""Merge of split-KV partials: rows of 16, 32 and 64 lanes, sets of up to 32, 64 and 128 splits, rows that end within a wave."""
import pytest
import torch

from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("b,sq,h,hk,d", [(1, 1, 1, 1, 16), (3, 1, 3, 1, 64), (2, 5, 3, 3, 72), (4, 1, 8, 2, 128), (2, 3, 2, 1, 136), (3, 1, 2, 2, 256)])
def test_merge(b, sq, h, hk, d):
    """every row count that leaves lanes of the last wave without a row (1, 9, 15 x 2, ...); an entry without a key in all splits;
    short entries, whose later splits hold nothing, beside full ones in one wave; the same bits twice"""
    from flash_attn import _native as nat
    gen = torch.Generator().manual_seed(d)
    mk = lambda *s: torch.randn(*s, generator=gen).to(torch.bfloat16)
    cap = 16640
    q, kc, vc = mk(b, sq, h, d), mk(b, cap, hk, d), mk(b, cap, hk, d)
    lens = torch.tensor([cap, 0, 300, 9000][:b], dtype=torch.int32)
    o_ref, l_ref, _, _ = orc.kvcache_forward(q, kc, vc, None, None, None, None, lens, causal=True)
    o_pt, _, _, _ = orc.kvcache_forward(q, kc, vc, None, None, None, None, lens, causal=True, upcast=False, reorder_ops=True)
    qd, kd, vd, ld = q.to(DEV), kc.to(DEV), vc.to(DEV), lens.to(DEV)
    for num_splits in (2, 9, 16, 17, 32, 33, 64, 65, 128):
        print(num_splits, flush=True)
        out, lse = nat.fwd_kvcache(qd, kd, vd, None, None, ld, None, None, None, None, d ** -0.5, True, -1, -1, False, num_splits)
        assert nat.last_kernel()[2]
        again = nat.fwd_kvcache(qd, kd, vd, None, None, ld, None, None, None, None, d ** -0.5, True, -1, -1, False, num_splits)
        assert torch.equal(out, again[0]) and torch.equal(lse, again[1])
        ok, err, bound = orc.tolerance_ok(out.cpu(), o_ref, o_pt, 3.0, 1e-5)
        assert ok, (num_splits, err, bound)
        assert orc.lse_ok(lse.cpu(), l_ref, 1e-3)[0], num_splits
        if b > 1:
            assert bool((out[1] == 0).all()) and bool(torch.isinf(lse[1]).all())
