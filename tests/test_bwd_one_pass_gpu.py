"""GPU parity of the one-pass backward kernel (csrc/fa_bwd_stream.h), which takes launches of head dim up to 64 whose
(batch, kv head) pairs fill the CUs.  Sizes sit on the edges of its tiles: 64 query rows, 32 keys of a wave, 128 keys of a
key block (up to it dQ leaves directly, beyond it through scratch), sequences that see nothing, one round of 512 pairs more or
less full, and several rounds with a last one that is partly empty (every second one in reversed order, accumulators carried
from one pair into the next).  Batch entries are independent problems, so some of them are checked against the CPU
oracle by the rule of tests/test_bwd_gpu.py, and every entry against the two-pass kernels, which the same call runs when it
is lent no scratch (more than 128 keys)."""
import sys

import pytest
import torch

from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _gen(shape, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g, dtype=torch.float32).to(dtype)


def _form():
    from flash_attn import _native as nat
    return {1: "two passes", 2: "one pass"}[nat.lib.fa_last_bwd_kernel()]


def _least_batch(h, hk, sq, sk, d):
    """the smallest batch that the kernel takes; the library's answer: past 128 keys scratch is asked for exactly where it runs"""
    import ctypes
    from flash_attn import _native as nat
    p = nat.FaBwdParams()
    p.h, p.h_k, p.d, p.seqlen_q, p.seqlen_k = h, hk, d, max(sq, sk), max(sq, sk)         # (the longer one decides)
    if max(sq, sk) <= 128:
        return 128 // hk                            # (one head per group in the cases here)
    for p.b in range(128 // hk, 512 // hk + 1):
        if nat.lib.fa_bwd_scratch_bytes(ctypes.byref(p), 0, 0) > 0:
            return p.b
    raise AssertionError("no batch of up to 512 pairs takes the kernel")


def _check(got, q, k, v, dout, **kw):
    ref = orc.attention_backward(q, k, v, dout, **kw)
    pt = orc.attention_backward_autograd(q, k, v, dout, upcast=False, reorder_ops=True, **kw)
    for name, a, r, p_ in zip(("dq", "dk", "dv"), got, ref, pt):
        assert torch.isfinite(a).all(), name
        err = (a.float().cpu() - r).abs().max().item()
        bound = 2 * (p_.float() - r).abs().max().item() + 1e-5
        _say("   %s err %.3e bound %.3e" % (name, err, bound))
        assert err <= bound, "%s error %g exceeds bound %g" % (name, err, bound)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("mode", ["full", "causal", "local"])
@pytest.mark.parametrize("sq,sk,d,h,hk", [(64, 64, 64, 8, 8), (5, 31, 32, 4, 4), (65, 128, 64, 8, 8), (63, 129, 40, 8, 4), (192, 256, 64, 8, 8), (128, 300, 64, 4, 2),
                                          (512, 512, 64, 8, 8), (257, 700, 64, 8, 2), (700, 257, 56, 2, 2), (300, 1, 64, 8, 8), (900, 1024, 64, 2, 1)])
def test_one_pass_backward(sq, sk, d, h, hk, mode, dtype, monkeypatch):
    _say("one pass", sq, sk, d, h, hk, mode, dtype)
    b = _least_batch(h, hk, sq, sk, d)
    _dense(b, sq, sk, d, h, hk, mode, dtype, (0, b // 2, b - 1), monkeypatch)


@pytest.mark.parametrize("mode", ["full", "causal", "local"])
@pytest.mark.parametrize("b,sq,sk,h,hk", [(137, 200, 200, 8, 8), (96, 500, 500, 8, 8), (180, 130, 256, 8, 4), (130, 64, 100, 8, 8), (690, 70, 140, 2, 1)])
def test_one_pass_backward_in_rounds(b, sq, sk, h, hk, mode, monkeypatch):
    """More pairs than the 512 slots, not a multiple of them: entries that the first, second and third rounds serve, and the
    last round's first and last ones."""
    _say("one pass rounds", b, sq, sk, h, hk, mode)
    entries = {i // hk for i in (0, 511, 512, 767, 1023, 1024, b * hk - 1) if i < b * hk}
    _dense(b, sq, sk, 64, h, hk, mode, torch.bfloat16, sorted(entries), monkeypatch)


def _dense(b, sq, sk, d, h, hk, mode, dtype, entries, monkeypatch):
    from flash_attn import _native as nat
    q = _gen((b, sq, h, d), dtype, 1); k = _gen((b, sk, hk, d), dtype, 2); v = _gen((b, sk, hk, d), dtype, 3)
    dout = _gen((b, sq, h, d), dtype, 4)
    causal, (wl, wr) = mode == "causal", ((70, 40) if mode == "local" else (-1, -1))
    qd, kd, vd, gd = [t.to(DEV) for t in (q, k, v, dout)]
    out, _, _, _, _, lse, _, _ = nat.fwd(qd, kd, vd, None, 0.0, d ** -0.5, causal, wl, wr, False, None)
    bwd = lambda: nat.bwd(gd, qd, kd, vd, out, lse, None, None, None, 0.0, d ** -0.5, causal, wl, wr, None, None)
    got = bwd()
    assert _form() == "one pass"
    for a, c in zip(got, bwd()):
        assert torch.equal(a[..., :sq] if a.dim() == 3 else a, c[..., :sq] if c.dim() == 3 else c)
    want_d = (gd.float() * out.float()).sum(-1).permute(0, 2, 1)
    assert torch.allclose(got[3][:, :, :sq], want_d, rtol=1e-4, atol=1e-4) and not got[3][:, :, sq:].any()
    for e in entries:
        s = slice(e, e + 1)
        _check([t[s] for t in got[:3]], q[s], k[s], v[s], dout[s], causal=causal, window_size=(wl, wr))
    if sk <= 128:
        return
    monkeypatch.setattr(nat, "_lend_scratch", lambda *a: None)
    # both forms round P, dS and the results to the tensor type; 2^-8 (bf16) or 2^-11 (fp16) of the largest entry each
    for a, c in zip(got[:3], bwd()[:3]):
        eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
        assert (a.float() - c.float()).abs().max() <= 4 * eps * c.float().abs().max() + 1e-5
    assert _form() == "two passes"


@pytest.mark.parametrize("p", [0.0, 0.17])
@pytest.mark.parametrize("mode", ["full", "causal"])
@pytest.mark.parametrize("reps", [10, 18])
def test_one_pass_backward_packed(reps, mode, p, monkeypatch):
    """Packed sequences of very different lengths (empty ones, one token, several key blocks) in launches of two and three
    rounds of 512 pairs, with and without dropout (the mask read from S_dmask)."""
    import flash_attn
    from flash_attn import _native as nat
    _say("one pass packed", reps, mode, p)
    dtype, h, d = torch.float16, 8, 64
    lens_q = [0, 1, 63, 64, 65, 300, 77, 256, 257, 513] * reps
    # (no sequence of one key: with dropout dP - D cancels there to the rounding of the 16-bit O that D is formed from)
    lens_k = [5, 40, 200, 64, 333, 0, 256, 257, 255, 513] * reps
    cu_q = torch.tensor([0] + list(torch.tensor(lens_q).cumsum(0)), dtype=torch.int32)
    cu_k = torch.tensor([0] + list(torch.tensor(lens_k).cumsum(0)), dtype=torch.int32)
    q = _gen((int(cu_q[-1]), h, d), dtype, 1); k = _gen((int(cu_k[-1]), h, d), dtype, 2)
    v = _gen((int(cu_k[-1]), h, d), dtype, 3); dout = _gen((int(cu_q[-1]), h, d), dtype, 4)
    qd, kd, vd = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out, _, S = flash_attn.flash_attn_varlen_func(qd, kd, vd, cu_q.to(DEV), cu_k.to(DEV), max(lens_q), max(lens_k), dropout_p=p,
                                                  causal=mode == "causal", return_attn_probs=True)
    launch, forms = nat._launch_bwd, []             # (autograd calls it on a thread of its own)
    monkeypatch.setattr(nat, "_launch_bwd", lambda *a: (launch(*a), forms.append(_form())))
    dq, dk, dv = torch.autograd.grad(out, (qd, kd, vd), dout.to(DEV))
    assert forms == ["one pass"]
    assert all(torch.isfinite(t).all() for t in (dq, dk, dv))
    for i in list(range(10)) + [29]:
        a, e, c, f = int(cu_q[i]), int(cu_q[i + 1]), int(cu_k[i]), int(cu_k[i + 1])
        if e == a or f == c:
            assert not dq[a:e].any() and not dk[c:f].any() and not dv[c:f].any()
            continue
        _say("  seq", i, lens_q[i], lens_k[i])
        kw = dict(causal=mode == "causal")
        if p:
            kw.update(dropout_p=p, dropout_mask=~torch.signbit(S[i:i + 1, :, :e - a, :f - c].float().cpu()))
        _check((dq[a:e][None], dk[c:f][None], dv[c:f][None]), q[a:e][None], k[c:f][None], v[c:f][None], dout[a:e][None], **kw)


def _packed(lens, h, dtype, seed):
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    q, k, v, g = [_gen((int(cu[-1]), h, 64), dtype, seed + i) for i in range(4)]
    return cu, q, k, v, g


def _packed_bwd(q, k, v, g, out, lse, cu, longest, causal=True):
    from flash_attn import _native as nat
    return nat.varlen_bwd(g, q, k, v, out, lse, None, None, None, cu, cu, longest, longest, 0.0, 64 ** -0.5, False, causal, -1, -1, None, None)


@pytest.mark.parametrize("n,lo,hi", [(63, 65, 200), (64, 1, 513), (257, 0, 130), (1100, 0, 131), (2048, 0, 131), (2100, 130, 150)])
def test_one_pass_backward_of_many_sequences(n, lo, hi, monkeypatch):
    """Batches around the chunks of 64 in which the kernel orders sequences by cost, up to the most that it orders (2048) and
    beyond, where it takes them as they come: every entry against the two passes, some against the oracle."""
    from flash_attn import _native as nat
    _say("one pass, sequences:", n, lo, hi)
    dtype, h = torch.float16, 2 if n > 256 else 8
    lens = [lo + (i * 37) % (hi - lo) for i in range(n)]
    cu, q, k, v, g = _packed(lens, h, dtype, 1)
    qd, kd, vd, gd, cud = [t.to(DEV) for t in (q, k, v, g, cu)]
    out, _, _, _, _, lse, _, _ = nat.varlen_fwd(qd, kd, vd, None, cud, cud, max(lens), max(lens), 0.0, 64 ** -0.5, False, True, -1, -1, False, None)
    got = _packed_bwd(qd, kd, vd, gd, out, lse, cud, max(lens))
    assert max(lens) > 128 and _form() == "one pass"
    for i in [i for i in (0, 1, 2, 62, 63, 64, 255, 256, 600, 1023, 1024, 1099, 2047, 2048, 2099) if i < n]:
        a, e = int(cu[i]), int(cu[i + 1])
        if e > a + 5:               # (rows of one to five keys: dP - D cancels to the rounding of the 16-bit O)
            _check([t[a:e][None] for t in got[:3]], q[a:e][None], k[a:e][None], v[a:e][None], g[a:e][None], causal=True)
    monkeypatch.setattr(nat, "_lend_scratch", lambda *a: None)
    two = _packed_bwd(qd, kd, vd, gd, out, lse, cud, max(lens))
    assert _form() == "two passes"
    for a, c in zip(got[:3], two[:3]):
        assert (a.float() - c.float()).abs().max() <= 4 * 2.0 ** -11 * c.float().abs().max() + 1e-5


def test_one_pass_backward_ends_at_the_declared_maximum(monkeypatch):
    """A sequence longer than the declared maximum: scratch, lse and softmax_d hold that many rows, so the kernel stops there.
    Its neighbours get what they get under the right maximum, bit for bit, and nothing is written around the scratch."""
    from flash_attn import _native as nat
    _say("one pass, declared maximum")
    h, lens = 8, [150, 192, 130, 250, 64, 192, 1, 180] * 8
    cu, q, k, v, g = _packed(lens, h, torch.bfloat16, 5)
    q, k, v, g, cud = [t.to(DEV) for t in (q, k, v, g, cu)]
    out, _, _, _, _, lse, _, _ = nat.varlen_fwd(q, k, v, None, cud, cud, 250, 250, 0.0, 64 ** -0.5, False, True, -1, -1, False, None)
    want = _packed_bwd(q, k, v, g, out, lse, cud, 250)
    assert _form() == "one pass"
    lent = []

    def lend(p, device, total_q, total_k):
        import ctypes
        n = nat.lib.fa_bwd_scratch_bytes(ctypes.byref(p), total_q, total_k)
        lent.append(torch.full((n + 2 * 4096,), 0x5A, dtype=torch.uint8, device=device))
        return lent[-1][4096:4096 + n]

    monkeypatch.setattr(nat, "_lend_scratch", lend)
    got = _packed_bwd(q, k, v, g, out, lse[:, :, :192].contiguous(), cud, 192)
    assert _form() == "one pass"
    assert (lent[0][:4096] == 0x5A).all() and (lent[0][-4096:] == 0x5A).all()
    for i, n in enumerate(lens):
        if n <= 192:
            a, e = int(cu[i]), int(cu[i + 1])
            assert all(torch.equal(x[a:e], y[a:e]) for x, y in zip(got[:3], want[:3])), i
            assert torch.equal(got[3][i, :, :n], want[3][i, :, :n]) and not got[3][i, :, n:].any()
