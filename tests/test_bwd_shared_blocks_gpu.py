"""GPU parity of dK/dV where several workgroups share a key block (join_parts, csrc/fa_bwd.h): two to many parts of unequal
length, parts that begin inside a grouped head's tiles and at their end, uncut blocks beside cut ones, a last key block of one
key, blocks that see nothing, more than 64 key blocks (a unit finds its block 64 at a time), every width of the accumulators.
Against the CPU oracle by the rule of tests/test_bwd_gpu.py, and against the uncut pass, which the same call runs when it is
lent no scratch; scratch holds garbage before the call and keeps the words around it."""
import ctypes
import sys

import pytest
import torch

from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _gen(shape, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g, dtype=torch.float32).to(dtype)


def _lender(nat, lent):
    def lend(p, device, total_q=0, total_k=0):
        n = nat.lib.fa_bwd_lend_bytes(ctypes.byref(p), total_q, total_k)
        assert n > 0 and nat.lib.fa_bwd_scratch_bytes(ctypes.byref(p), total_q, total_k) == 0
        lent.append(torch.full((n + 2 * 4096,), 0x5A, dtype=torch.uint8, device=device))
        return lent[-1][4096:4096 + n]
    return lend


def _case(b, sq, sk, h, hk, d, dtype, mode, p_dropout=0.0):
    from flash_attn import _native as nat
    print("shared blocks", b, sq, sk, h, hk, d, dtype, mode, p_dropout, flush=True)
    sys.stdout.flush()
    q, k, v, g = [_gen(s, dtype, i) for i, s in enumerate([(b, sq, h, d), (b, sk, hk, d), (b, sk, hk, d), (b, sq, h, d)])]
    causal, (wl, wr) = mode == "causal", (300, 150) if mode == "local" else (-1, -1)
    qd, kd, vd, gd = [t.to(DEV) for t in (q, k, v, g)]
    torch.cuda.manual_seed(d)
    out, _, _, _, _, lse, S, rng = nat.fwd(qd, kd, vd, None, p_dropout, d ** -0.5, causal, wl, wr, p_dropout > 0, None)
    bwd = lambda: nat.bwd(gd, qd, kd, vd, out, lse, None, None, None, p_dropout, d ** -0.5, causal, wl, wr, None, rng)[:3]
    kw = dict(causal=causal, window_size=(wl, wr))
    if p_dropout > 0:
        kw.update(dropout_p=p_dropout, dropout_mask=~torch.signbit(S[:, :, :sq, :sk].float().cpu()))
    return bwd, (q, k, v, g), kw


def _check(got, q, k, v, g, **kw):
    ref = orc.attention_backward(q, k, v, g, **kw)
    pt = orc.attention_backward_autograd(q, k, v, g, upcast=False, reorder_ops=True, **kw)
    for name, a, r, p_ in zip(("dq", "dk", "dv"), got, ref, pt):
        err, bound = (a.float().cpu() - r).abs().max().item(), 2 * (p_.float() - r).abs().max().item() + 1e-5
        assert err <= bound, "%s error %g exceeds bound %g" % (name, err, bound)


@pytest.mark.parametrize("d,dtype", [(40, torch.float16), (64, torch.bfloat16), (96, torch.bfloat16), (128, torch.float16), (160, torch.bfloat16),
                                     (192, torch.float16), (256, torch.bfloat16)])
@pytest.mark.parametrize("mode", ["full", "causal", "local"])
@pytest.mark.parametrize("b,sq,sk,h,hk", [(1, 1025, 257, 8, 2), (2, 700, 1000, 6, 1), (1, 530, 129, 32, 4), (1, 1100, 300, 16, 1)])
def test_shared_key_blocks(monkeypatch, b, sq, sk, h, hk, d, dtype, mode):
    from flash_attn import _native as nat
    bwd, args, kw = _case(b, sq, sk, h, hk, d, dtype, mode)
    lent = []
    monkeypatch.setattr(nat, "_lend_scratch", _lender(nat, lent))
    got = bwd()
    assert (lent[0][:4096] == 0x5A).all() and (lent[0][-4096:] == 0x5A).all()
    for _ in range(3):
        assert all(torch.equal(a, c) for a, c in zip(got, bwd()))
    _check(got, *args, **kw)
    monkeypatch.setattr(nat, "_lend_scratch", lambda *a: None)
    for a, c in zip(got, bwd()):       # fp32 sums in another order, rounded to 16 bits once (and P's share of them, unchanged)
        assert (a.float() - c.float()).abs().max() <= 2 * torch.finfo(dtype).eps * c.float().abs().max()


@pytest.mark.parametrize("d,dtype", [(128, torch.float16), (192, torch.bfloat16), (256, torch.bfloat16)])
@pytest.mark.parametrize("b,sq,sk,h,hk,mode", [
    (4, 700, 700, 16, 4, "causal"), (4, 700, 700, 16, 4, "local"),        # 16 (batch, kv head) streams: two to an XCD, dealt out by turns
    (6, 600, 300, 16, 4, "causal"), (6, 600, 300, 16, 4, "local"),        # 24: three
    (9, 700, 700, 4, 1, "full"), (3, 500, 300, 24, 6, "full"),            # 9 and 18: an XCD's share begins inside a stream
])
def test_shared_key_blocks_of_many_streams(monkeypatch, b, sq, sk, h, hk, mode, d, dtype):
    """More than 8 streams: which one and which part of a key block a workgroup gets, and so where its sums meet, follows from other
    index arithmetic (xcd_stream_unit)."""
    from flash_attn import _native as nat
    bwd, args, kw = _case(b, sq, sk, h, hk, d, dtype, mode)
    lent = []
    monkeypatch.setattr(nat, "_lend_scratch", _lender(nat, lent))
    got = bwd()
    assert (lent[0][:4096] == 0x5A).all() and (lent[0][-4096:] == 0x5A).all()
    assert all(torch.equal(a, c) for a, c in zip(got, bwd()))
    for i in (0, b // 2, b - 1):
        one = slice(i, i + 1)
        _check([t[one] for t in got], *[t[one] for t in args], **kw)
    monkeypatch.setattr(nat, "_lend_scratch", lambda *a: None)
    for a, c in zip(got, bwd()):       # as above
        assert (a.float() - c.float()).abs().max() <= 2 * torch.finfo(dtype).eps * c.float().abs().max()


@pytest.mark.parametrize("d,dtype", [(64, torch.bfloat16), (128, torch.float16), (256, torch.bfloat16)])
def test_shared_key_blocks_with_dropout(monkeypatch, d, dtype):
    from flash_attn import _native as nat
    bwd, args, kw = _case(1, 600, 300, 8, 2, d, dtype, "causal", 0.17)
    monkeypatch.setattr(nat, "_lend_scratch", _lender(nat, []))
    got = bwd()
    assert all(torch.equal(a, c) for a, c in zip(got, bwd()))
    _check(got, *args, **kw)


def test_shared_key_blocks_of_a_long_sequence(monkeypatch):
    """70 key blocks of one kv head."""
    from flash_attn import _native as nat
    bwd, _, _ = _case(1, 8900, 8900, 2, 1, 128, torch.bfloat16, "causal")
    monkeypatch.setattr(nat, "_lend_scratch", _lender(nat, []))
    got = bwd()
    assert all(torch.equal(a, c) for a, c in zip(got, bwd()))
    monkeypatch.setattr(nat, "_lend_scratch", lambda *a: None)
    for a, c in zip(got, bwd()):
        assert (a.float() - c.float()).abs().max() <= 2 * 2.0 ** -7 * c.float().abs().max()


def test_shared_key_blocks_under_capture(monkeypatch):
    """Every replay counts the arrivals anew."""
    from flash_attn import _native as nat
    bwd, _, _ = _case(1, 700, 700, 8, 1, 128, torch.bfloat16, "causal")
    want = bwd()
    monkeypatch.setattr(nat, "_lend_scratch", _lender(nat, []))
    assert all((a.float() - c.float()).abs().max() <= 2 * 2.0 ** -7 * c.float().abs().max() for a, c in zip(bwd(), want))
    eager = bwd()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = bwd()
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, c) for a, c in zip(got, eager))
        bwd()
