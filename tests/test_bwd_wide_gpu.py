"""GPU parity of the dQ pass of head dims 161-256, with dropout 129-256 (bwd_dq2_kernel, csrc/fa_bwd.h), whose two waves per row block hand P and dS
over one 32-key tile later each: key lengths of one to four tiles and their edges (the pipeline fills and drains), row blocks
with nothing visible between others, both halves of the columns partly past the head dim, dropout, packed batches with empty
sequences.  Against the CPU oracle by the rule of tests/test_bwd_gpu.py."""
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


def _check(got, q, k, v, dout, **kw):
    ref = orc.attention_backward(q, k, v, dout, **kw)
    pt = orc.attention_backward_autograd(q, k, v, dout, upcast=False, reorder_ops=True, **kw)
    for name, a, r, p_ in zip(("dq", "dk", "dv"), got, ref, pt):
        assert torch.isfinite(a).all(), name
        err = (a.float().cpu() - r).abs().max().item()
        bound = 2 * (p_.float() - r).abs().max().item() + 1e-5
        assert err <= bound, "%s error %g exceeds bound %g" % (name, err, bound)


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 168), (torch.float16, 192), (torch.bfloat16, 200), (torch.float16, 256)])
@pytest.mark.parametrize("mode", ["full", "causal", "local"])
@pytest.mark.parametrize("sq,sk", [(1, 32), (33, 31), (127, 33), (129, 64), (160, 65), (96, 97), (300, 128), (257, 200), (40, 500)])
def test_wide_backward(sq, sk, mode, dtype, d):
    import flash_attn
    _say("wide", sq, sk, mode, dtype, d)
    b, h, hk = 2, 4, 2
    q, k, v = _gen((b, sq, h, d), dtype, 1), _gen((b, sk, hk, d), dtype, 2), _gen((b, sk, hk, d), dtype, 3)
    dout = _gen((b, sq, h, d), dtype, 4)
    kw = dict(causal=mode == "causal", window_size=(50, 20) if mode == "local" else (-1, -1))
    qd, kd, vd = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out = flash_attn.flash_attn_func(qd, kd, vd, **kw)
    got = torch.autograd.grad(out, (qd, kd, vd), dout.to(DEV), retain_graph=True)
    for a, c in zip(got, torch.autograd.grad(out, (qd, kd, vd), dout.to(DEV))):
        assert torch.equal(a, c)
    _check(got, q, k, v, dout, **kw)


@pytest.mark.parametrize("d", [136, 160, 192, 256])
@pytest.mark.parametrize("mode", ["full", "causal"])
def test_wide_backward_packed_dropout(mode, d):
    import flash_attn
    _say("wide packed", mode, d)
    dtype, h = torch.float16, 2
    lens_q, lens_k = [0, 1, 63, 130, 200, 257], [5, 40, 200, 33, 0, 300]
    cu_q = torch.tensor([0] + list(torch.tensor(lens_q).cumsum(0)), dtype=torch.int32)
    cu_k = torch.tensor([0] + list(torch.tensor(lens_k).cumsum(0)), dtype=torch.int32)
    q, k = _gen((int(cu_q[-1]), h, d), dtype, 1), _gen((int(cu_k[-1]), h, d), dtype, 2)
    v, dout = _gen((int(cu_k[-1]), h, d), dtype, 3), _gen((int(cu_q[-1]), h, d), dtype, 4)
    qd, kd, vd = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out, _, S = flash_attn.flash_attn_varlen_func(qd, kd, vd, cu_q.to(DEV), cu_k.to(DEV), max(lens_q), max(lens_k), dropout_p=0.17,
                                                  causal=mode == "causal", return_attn_probs=True)
    dq, dk, dv = torch.autograd.grad(out, (qd, kd, vd), dout.to(DEV))
    for i in range(len(lens_q)):
        a, e, c, f = int(cu_q[i]), int(cu_q[i + 1]), int(cu_k[i]), int(cu_k[i + 1])
        if e == a or f == c:
            assert not dq[a:e].any() and not dk[c:f].any() and not dv[c:f].any()
            continue
        kw = dict(causal=mode == "causal", dropout_p=0.17, dropout_mask=~torch.signbit(S[i:i + 1, :, :e - a, :f - c].float().cpu()))
        _check((dq[a:e][None], dk[c:f][None], dv[c:f][None]), q[a:e][None], k[c:f][None], v[c:f][None], dout[a:e][None], **kw)


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 200), (torch.float16, 256), (torch.bfloat16, 248)])
@pytest.mark.parametrize("mode", ["full", "causal", "local"])
@pytest.mark.parametrize("b,sq,sk", [(65, 33, 31), (33, 31, 129), (33, 129, 160), (17, 300, 500)])
def test_wide_backward_whole_accumulators(b, sq, sk, mode, dtype, d):
    """More than 128 key blocks: a workgroup accumulates all columns of dK and dV (the cases above: half of them)."""
    import flash_attn
    _say("wide whole", b, sq, sk, mode, dtype, d)
    h, hk = 4, 2
    assert (sk + 127) // 128 * hk * b > 128
    q, k, v = _gen((b, sq, h, d), dtype, 1), _gen((b, sk, hk, d), dtype, 2), _gen((b, sk, hk, d), dtype, 3)
    dout = _gen((b, sq, h, d), dtype, 4)
    kw = dict(causal=mode == "causal", window_size=(50, 20) if mode == "local" else (-1, -1))
    qd, kd, vd = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out = flash_attn.flash_attn_func(qd, kd, vd, **kw)
    got = torch.autograd.grad(out, (qd, kd, vd), dout.to(DEV), retain_graph=True)
    for a, c in zip(got, torch.autograd.grad(out, (qd, kd, vd), dout.to(DEV))):
        assert torch.equal(a, c)
    for i in (0, b // 2, b - 1):
        one = slice(i, i + 1)
        _check([t[one] for t in got], q[one], k[one], v[one], dout[one], **kw)


@pytest.mark.parametrize("d", [136, 160, 192, 256])
@pytest.mark.parametrize("mode", ["full", "causal"])
def test_wide_backward_packed_dropout_whole_accumulators(mode, d):
    """The packed batch above eight times over: more than 128 key blocks."""
    import flash_attn
    _say("wide packed whole", mode, d)
    dtype, h, copies = torch.float16, 2, 8
    torch.cuda.manual_seed(d)
    lens_q, lens_k = [0, 1, 63, 130, 200, 257] * copies, [5, 40, 200, 33, 0, 300] * copies
    assert len(lens_k) * h * 3 > 128
    cu_q = torch.tensor([0] + list(torch.tensor(lens_q).cumsum(0)), dtype=torch.int32)
    cu_k = torch.tensor([0] + list(torch.tensor(lens_k).cumsum(0)), dtype=torch.int32)
    q, k = _gen((int(cu_q[-1]), h, d), dtype, 1), _gen((int(cu_k[-1]), h, d), dtype, 2)
    v, dout = _gen((int(cu_k[-1]), h, d), dtype, 3), _gen((int(cu_q[-1]), h, d), dtype, 4)
    qd, kd, vd = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out, _, S = flash_attn.flash_attn_varlen_func(qd, kd, vd, cu_q.to(DEV), cu_k.to(DEV), max(lens_q), max(lens_k), dropout_p=0.17,
                                                  causal=mode == "causal", return_attn_probs=True)
    dq, dk, dv = torch.autograd.grad(out, (qd, kd, vd), dout.to(DEV))
    for i in range(len(lens_q) - 6, len(lens_q)):
        a, e, c, f = int(cu_q[i]), int(cu_q[i + 1]), int(cu_k[i]), int(cu_k[i + 1])
        if e == a or f == c:
            assert not dq[a:e].any() and not dk[c:f].any() and not dv[c:f].any()
            continue
        kw = dict(causal=mode == "causal", dropout_p=0.17, dropout_mask=~torch.signbit(S[i:i + 1, :, :e - a, :f - c].float().cpu()))
        _check((dq[a:e][None], dk[c:f][None], dv[c:f][None]), q[a:e][None], k[c:f][None], v[c:f][None], dout[a:e][None], **kw)


@pytest.mark.parametrize("copies,form", [(6, 3), (24, 2)])
@pytest.mark.parametrize("mode", ["full", "causal"])
def test_wide_backward_packed_dropout_on_both_sides_of_the_weight(mode, copies, form):
    """The packed batch above 6 and 24 times over: little enough in all for two workgroups to share a key block (FA_BWD_FORM_HALVES),
    though it is more than 128 key blocks by the declared maximum, and too much for that (FA_BWD_FORM_WHOLE)."""
    import ctypes

    import flash_attn
    from flash_attn import _native as nat
    _say("wide packed, weight", mode, copies)
    dtype, h, d = torch.float16, 2, 160
    torch.cuda.manual_seed(d)
    lens_q, lens_k = [0, 1, 63, 130, 200, 257] * copies, [5, 40, 200, 33, 0, 300] * copies
    p = nat.FaBwdParams()
    p.b, p.h, p.h_k, p.d, p.seqlen_q, p.seqlen_k, p.is_causal, p.window_left, p.window_right = len(lens_q), h, h, d, 257, 300, mode == "causal", -1, -1
    p.p_dropout, p.cu_seqlens_q, p.cu_seqlens_k = 0.17, 16, 16
    assert nat.lib.fa_bwd_plan_form(ctypes.byref(p), sum(lens_q), sum(lens_k), 0) == form
    cu_q = torch.tensor([0] + list(torch.tensor(lens_q).cumsum(0)), dtype=torch.int32)
    cu_k = torch.tensor([0] + list(torch.tensor(lens_k).cumsum(0)), dtype=torch.int32)
    q, k = _gen((int(cu_q[-1]), h, d), dtype, 1), _gen((int(cu_k[-1]), h, d), dtype, 2)
    v, dout = _gen((int(cu_k[-1]), h, d), dtype, 3), _gen((int(cu_q[-1]), h, d), dtype, 4)
    qd, kd, vd = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out, _, S = flash_attn.flash_attn_varlen_func(qd, kd, vd, cu_q.to(DEV), cu_k.to(DEV), 257, 300, dropout_p=0.17,
                                                  causal=mode == "causal", return_attn_probs=True)
    dq, dk, dv = torch.autograd.grad(out, (qd, kd, vd), dout.to(DEV))
    for i in list(range(6)) + list(range(len(lens_q) - 6, len(lens_q))):
        a, e, c, f = int(cu_q[i]), int(cu_q[i + 1]), int(cu_k[i]), int(cu_k[i + 1])
        if e == a or f == c:
            assert not dq[a:e].any() and not dk[c:f].any() and not dv[c:f].any()
            continue
        kw = dict(causal=mode == "causal", dropout_p=0.17, dropout_mask=~torch.signbit(S[i:i + 1, :, :e - a, :f - c].float().cpu()))
        _check((dq[a:e][None], dk[c:f][None], dv[c:f][None]), q[a:e][None], k[c:f][None], v[c:f][None], dout[a:e][None], **kw)
