"""Head dims 129-256 with split keys: equal parts of the tiles that a row block sees, on the 16-rows-per-wave kernel."""
import pytest
import torch

from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _mk(seed, dtype):
    gen = torch.Generator().manual_seed(seed)
    return lambda *s: torch.randn(*s, generator=gen).to(dtype)


@pytest.mark.parametrize("mode", ["causal", "full", "window", "window_right"])
@pytest.mark.parametrize("num_splits", [0, 2, 7, 64])
@pytest.mark.parametrize("sq,sk,h,hk,d,dtype", [
    (32, 1300, 3, 3, 136, torch.float16), (130, 961, 2, 2, 256, torch.bfloat16), (257, 2049, 4, 2, 192, torch.bfloat16),
    (300, 700, 1, 1, 200, torch.bfloat16), (128, 32, 2, 2, 256, torch.float16), (333, 95, 2, 1, 160, torch.bfloat16)])
def test_split_rows(sq, sk, h, hk, d, dtype, num_splits, mode):
    """parts of no tile at all, rows that a causal mask leaves without keys (sk < sq), a first row block of few rows, ragged last tiles, and
    the plan of the library (0)"""
    from flash_attn import _native as nat
    mk = _mk(sq + d, dtype)
    q, k, v = mk(2, sq, h, d), mk(2, sk, hk, d), mk(2, sk, hk, d)
    causal, wl, wr = mode == "causal", -1, -1
    if mode == "window":
        wl, wr = 100, 30
    if mode == "window_right":
        wr = 5
    out, lse = nat.fwd_kvcache(q.to(DEV), k.to(DEV), v.to(DEV), None, None, None, None, None, None, None, d ** -0.5, causal, wl, wr, True, num_splits)
    name, _, split, _ = nat.last_kernel()
    assert name == "pingpong_wide" and (num_splits == 0 or split == (num_splits > 1 and sk > 64))
    kw = dict(causal=causal, window_size=(wl, wr))
    ref, lse_ref, pt = orc.attention_reference_pair(q, k, v, **kw)
    ok, err, bound = orc.tolerance_ok(out.cpu(), ref, pt, 3.0, 1e-5)
    assert ok, (err, bound)
    assert orc.lse_ok(lse.cpu(), lse_ref, 1e-3)[0]


@pytest.mark.parametrize("num_splits", [0, 3])
@pytest.mark.parametrize("inter", [False, True])
@pytest.mark.parametrize("sq,h,hk,d,rot", [(40, 4, 4, 256, 256), (33, 2, 2, 160, 64), (150, 4, 2, 192, 0)])
def test_over_caches(sq, h, hk, d, rot, inter, num_splits):
    """lengths from none to all of the capacity, appended with and without rotary; q and out the same memory"""
    from flash_attn import _native as nat
    dtype, cap = torch.bfloat16, 1700
    mk = _mk(sq + d + num_splits, dtype)
    lens = torch.tensor([0, 64, 333, cap - sq], dtype=torch.int32)
    b = len(lens)
    q, kc, vc, kn, vn = mk(b, sq, h, d), mk(b, cap, hk, d), mk(b, cap, hk, d), mk(b, sq, hk, d), mk(b, sq, hk, d)
    cos, sin = orc.rotary_table(cap, rot, dtype=dtype) if rot else (None, None)
    dev = lambda t: None if t is None else t.to(DEV)
    kw = dict(causal=True, rotary_interleaved=inter)
    o_ref, l_ref, k_ref, v_ref = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, lens, **kw)
    o_pt, _, _, _ = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, lens, upcast=False, reorder_ops=True, **kw)
    for same in (False, True):
        qd, vd = q.to(DEV), vc.to(DEV)
        out, lse = nat.fwd_kvcache(qd, kc.to(DEV), vd, kn.to(DEV), vn.to(DEV), lens.to(DEV), dev(cos), dev(sin), None, qd if same else None, d ** -0.5, True, -1, -1, inter,
                                   num_splits)
        print(same, nat.last_kernel(), flush=True)
        ok, err, bound = orc.tolerance_ok(out.cpu(), o_ref, o_pt, 3.0, 1e-5)
        assert ok, (same, err, bound)
        assert orc.lse_ok(lse.cpu(), l_ref, 1e-3)[0]
        assert torch.equal(vd.cpu(), v_ref)


def test_not_a_number_passes_through_the_merge():
    from flash_attn import _native as nat
    mk = _mk(3, torch.bfloat16)
    q, k, v = mk(1, 128, 2, 256).to(DEV), mk(1, 1500, 2, 256).to(DEV), mk(1, 1500, 2, 256).to(DEV)
    q[0, 77, 1, 5] = float("nan")
    got = [nat.fwd_kvcache(q, k, v, None, None, None, None, None, None, None, 256 ** -0.5, True, -1, -1, True, n) for n in (1, 4)]
    for out, lse in got:
        bad = torch.isnan(out).any(-1)
        assert bad[0, 77, 1] and bad.sum() == 1 and torch.isinf(lse).sum() == 1 and lse[0, 1, 77] == float("inf")
    keep = ~torch.isnan(got[0][0])
    assert torch.allclose(got[0][0][keep].float(), got[1][0][keep].float(), atol=1e-2)
