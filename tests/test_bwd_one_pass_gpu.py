"""GPU parity of the one-pass backward kernel (csrc/fa_bwd_stream.h), which takes launches of head dim up to 64 whose
(batch, kv head) pairs fill the CUs.  Sizes sit on the edges of its tiles: 64 query rows, 32 keys of a wave, 128 keys of a
key block (up to it dQ leaves directly, beyond it through scratch), sequences that see nothing, one
round of 512 pairs more or less full.  Batch entries are independent problems, so three of them are checked against the CPU
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


def _one_pass_runs(b, h, hk, sq, sk, d):
    """the library's own answer: scratch is asked for exactly where the kernel runs on several key blocks"""
    import ctypes
    from flash_attn import _native as nat
    p = nat.FaBwdParams()
    p.b, p.h, p.h_k, p.d, p.seqlen_q, p.seqlen_k = b, h, hk, d, sq, sk
    return nat.lib.fa_bwd_scratch_bytes(ctypes.byref(p)) > 0


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
    from flash_attn import _native as nat
    _say("one pass", sq, sk, d, h, hk, mode, dtype)
    b = (128 if max(sq, sk) <= 256 else 224 if max(sq, sk) <= 512 else 400) // hk      # (the least that the kernel takes)
    q = _gen((b, sq, h, d), dtype, 1); k = _gen((b, sk, hk, d), dtype, 2); v = _gen((b, sk, hk, d), dtype, 3)
    dout = _gen((b, sq, h, d), dtype, 4)
    causal, (wl, wr) = mode == "causal", ((70, 40) if mode == "local" else (-1, -1))
    qd, kd, vd, gd = [t.to(DEV) for t in (q, k, v, dout)]
    out, _, _, _, _, lse, _, _ = nat.fwd(qd, kd, vd, None, 0.0, d ** -0.5, causal, wl, wr, False, None)
    bwd = lambda: nat.bwd(gd, qd, kd, vd, out, lse, None, None, None, 0.0, d ** -0.5, causal, wl, wr, None, None)
    got = bwd()
    assert _one_pass_runs(b, h, hk, sq, sk, d) == (sk > 128)
    for a, c in zip(got, bwd()):
        assert torch.equal(a[..., :sq] if a.dim() == 3 else a, c[..., :sq] if c.dim() == 3 else c)
    want_d = (gd.float() * out.float()).sum(-1).permute(0, 2, 1)
    assert torch.allclose(got[3][:, :, :sq], want_d, rtol=1e-4, atol=1e-4) and not got[3][:, :, sq:].any()
    for e in (0, b // 2, b - 1):
        s = slice(e, e + 1)
        _check([t[s] for t in got[:3]], q[s], k[s], v[s], dout[s], causal=causal, window_size=(wl, wr))
    if sk <= 128:
        return
    monkeypatch.setattr(nat, "_lend_scratch", lambda p, device: None)
    # both forms round P, dS and the results to the tensor type; 2^-8 (bf16) or 2^-11 (fp16) of the largest entry each
    for a, c in zip(got[:3], bwd()[:3]):
        eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
        assert (a.float() - c.float()).abs().max() <= 4 * eps * c.float().abs().max() + 1e-5


@pytest.mark.parametrize("p", [0.0, 0.17])
@pytest.mark.parametrize("mode", ["full", "causal"])
def test_one_pass_backward_packed(mode, p):
    """Packed sequences of very different lengths (empty ones, one token, several key blocks) in a launch of several
    rounds, with and without dropout (the mask read from S_dmask)."""
    import flash_attn
    _say("one pass packed", mode, p)
    dtype, h, d = torch.float16, 8, 64
    lens_q = [0, 1, 63, 64, 65, 300, 77, 256, 257, 513] * 6
    # (no sequence of one key: with dropout dP - D cancels there to the rounding of the 16-bit O that D is formed from)
    lens_k = [5, 40, 200, 64, 333, 0, 256, 257, 255, 513] * 6
    cu_q = torch.tensor([0] + list(torch.tensor(lens_q).cumsum(0)), dtype=torch.int32)
    cu_k = torch.tensor([0] + list(torch.tensor(lens_k).cumsum(0)), dtype=torch.int32)
    q = _gen((int(cu_q[-1]), h, d), dtype, 1); k = _gen((int(cu_k[-1]), h, d), dtype, 2)
    v = _gen((int(cu_k[-1]), h, d), dtype, 3); dout = _gen((int(cu_q[-1]), h, d), dtype, 4)
    qd, kd, vd = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    assert _one_pass_runs(len(lens_q), h, h, max(lens_q), max(lens_k), d)
    out, _, S = flash_attn.flash_attn_varlen_func(qd, kd, vd, cu_q.to(DEV), cu_k.to(DEV), max(lens_q), max(lens_k), dropout_p=p,
                                                  causal=mode == "causal", return_attn_probs=True)
    dq, dk, dv = torch.autograd.grad(out, (qd, kd, vd), dout.to(DEV))
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
