"""The native host path (flash_attn._host) against the Python one: the same library calls, so the same bits; and which calls it leaves
to the Python layer."""
import pytest
import torch

import flash_attn
from flash_attn import _native as nat
from flash_attn import flash_attn_interface as fi

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _gen(*shape, seed=0, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed), dtype=torch.float32).to(dtype).to(DEV)


CLASSES = {"func": fi.FlashAttnFunc, "qkvpacked": fi.FlashAttnQKVPackedFunc, "kvpacked": fi.FlashAttnKVPackedFunc,
           "varlen": fi.FlashAttnVarlenFunc, "varlen_qkvpacked": fi.FlashAttnVarlenQKVPackedFunc, "varlen_kvpacked": fi.FlashAttnVarlenKVPackedFunc}


def _call(kind, d=64, dtype=torch.bfloat16, **kw):
    """(function of the inputs, inputs)"""
    b, s, h, hk = 3, 130, 4, 2
    lens = [130, 1, 77]
    cu = torch.tensor([0, 130, 131, 208], dtype=torch.int32, device=DEV)
    total = sum(lens)
    if kind == "func":
        return (lambda q, k, v: flash_attn.flash_attn_func(q, k, v, **kw)), [_gen(b, s, h, d, seed=1, dtype=dtype), _gen(b, s + 9, hk, d, seed=2, dtype=dtype), _gen(b, s + 9, hk, d, seed=3, dtype=dtype)]
    if kind == "qkvpacked":
        return (lambda x: flash_attn.flash_attn_qkvpacked_func(x, **kw)), [_gen(b, s, 3, h, d, seed=1, dtype=dtype)]
    if kind == "kvpacked":
        return (lambda q, x: flash_attn.flash_attn_kvpacked_func(q, x, **kw)), [_gen(b, s, h, d, seed=1, dtype=dtype), _gen(b, s - 60, 2, hk, d, seed=2, dtype=dtype)]
    if kind == "varlen":
        return (lambda q, k, v: flash_attn.flash_attn_varlen_func(q, k, v, cu, cu, 130, 130, **kw)), [_gen(total, h, d, seed=1, dtype=dtype), _gen(total, hk, d, seed=2, dtype=dtype), _gen(total, hk, d, seed=3, dtype=dtype)]
    if kind == "varlen_qkvpacked":
        return (lambda x: flash_attn.flash_attn_varlen_qkvpacked_func(x, cu, 130, **kw)), [_gen(total, 3, h, d, seed=1, dtype=dtype)]
    return (lambda q, x: flash_attn.flash_attn_varlen_kvpacked_func(q, x, cu, cu, 130, 130, **kw)), [_gen(total, h, d, seed=1, dtype=dtype), _gen(total, 2, hk, d, seed=2, dtype=dtype)]


def _both(monkeypatch, kind, run):
    """run() on the native path, which must have taken it, and on the Python one"""
    cls = CLASSES[kind]
    native, taken = cls.native, []

    def watch(*a):
        taken.append(native(*a))
        return taken[-1]

    monkeypatch.setattr(cls, "native", watch)
    got = run()
    assert taken and all(t is not None for t in taken), kind
    monkeypatch.setattr(cls, "native", None)
    want = run()
    monkeypatch.setattr(cls, "native", native)
    return got, want


@pytest.mark.parametrize("dropout", [0.0, 0.2])
@pytest.mark.parametrize("kw", [dict(causal=True), dict(window_size=(17, 5)), dict(softmax_scale=0.3)], ids=["causal", "window", "scale"])
@pytest.mark.parametrize("d,dtype", [(64, torch.float16), (128, torch.bfloat16), (192, torch.bfloat16)])
@pytest.mark.parametrize("kind", list(CLASSES))
def test_same_bits_as_the_python_path(monkeypatch, kind, d, dtype, kw, dropout):
    f, xs = _call(kind, d, dtype, dropout_p=dropout, **kw)

    def run():
        torch.cuda.manual_seed(5)
        outs = [f(*xs)]                                             # no gradient
        leaves = [x.clone().requires_grad_() for x in xs]
        out = f(*leaves)
        assert out.requires_grad
        g = _gen(*out.shape, seed=9, dtype=dtype)
        outs += [out.detach(), *torch.autograd.grad(out, leaves, g, retain_graph=True)]
        outs += torch.autograd.grad(out, leaves[-1], g.transpose(0, 1).contiguous().transpose(0, 1))     # another layout, one input
        outs += torch.autograd.grad(f(*leaves).float().sum(), leaves)                                    # an expanded gradient
        leaves[0].requires_grad_(False)
        if len(leaves) > 1:
            outs += torch.autograd.grad(f(*leaves), leaves[1:], g)
        outs.append(torch.tensor(torch.cuda.default_generators[torch.cuda.current_device()].get_offset()))
        return outs

    got, want = _both(monkeypatch, kind, run)
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)


def test_views_parameters_and_streams(monkeypatch):
    """q, k, v as views of one projection, an nn.Parameter, a side stream, a captured graph replayed between eager calls"""
    proj = torch.nn.Parameter(_gen(2, 100, 12, 64, seed=3))

    def run():
        q, k, v = proj[:, :, :8], proj[:, :, 8:10], proj[:, :, 10:]
        out = flash_attn.flash_attn_func(q, k, v, causal=True)
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            out2 = flash_attn.flash_attn_func(q, k, v, causal=True)
        torch.cuda.current_stream().wait_stream(s)
        return [out.detach(), out2.detach(), *torch.autograd.grad(out.float().square().sum() + out2.float().sum(), proj)]

    got, want = _both(monkeypatch, "func", run)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    q, k, v = (t.detach().contiguous() for t in (proj[:, :, :8], proj[:, :, 8:10], proj[:, :, 10:]))
    ref = flash_attn.flash_attn_func(q, k, v, causal=True)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        flash_attn.flash_attn_func(q, k, v, causal=True)
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out = flash_attn.flash_attn_func(q, k, v, causal=True)
    for _ in range(3):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref) and torch.equal(flash_attn.flash_attn_func(q, k, v, causal=True), ref)


def _declined(cls, f):
    """f() must run (or fail) without the native path, which was asked, having done it"""
    native, taken = cls.native, []
    cls.native = lambda *a: (taken.append(native(*a)), taken[-1])[1]
    try:
        return f()
    finally:
        cls.native = native
        assert taken and taken == [None] * len(taken)


def test_calls_that_the_python_layer_keeps():
    q = _gen(2, 64, 4, 64, seed=1)
    f = lambda *a, **kw: flash_attn.flash_attn_func(*a, **kw)
    for run in (lambda: f(q, q, q, return_attn_probs=True),                      # more than one result
                lambda: f(q[..., :60], q[..., :60], q[..., :60]),                # a head dim that is padded
                lambda: f(*([q.transpose(1, 3).contiguous().transpose(1, 3)] * 3)),    # head dim not contiguous
                lambda: f(q[:, :0], q, q),                                       # nothing to do
                lambda: f(q, q, q, causal=1)):
        _declined(fi.FlashAttnFunc, run)
    packed, saved = [], []
    x = q.clone().requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t), t)[1], lambda t: (saved.append(t), t)[1]):
        out = _declined(fi.FlashAttnFunc, lambda: f(x, x, x))
    out.sum().backward()
    assert len(packed) == len(saved) == 6                                        # q, k, v, out, log-sum-exp, rng state
    with torch.autograd.set_detect_anomaly(True, check_nan=False):
        _declined(fi.FlashAttnFunc, lambda: f(x, x, x))

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        _declined(fi.FlashAttnFunc, lambda: f(q, q, q))

    class Sub(torch.Tensor):
        pass

    _declined(fi.FlashAttnFunc, lambda: f(q.as_subclass(Sub), q, q))
    for module, name in ((nat, "_lend_scratch"), (fi, "_flash_attn_forward"), (fi, "_flash_attn_backward")):      # a function of the Python layer replaced
        own, calls = getattr(module, name), []
        with pytest.MonkeyPatch.context() as m:
            m.setattr(module, name, lambda *a, **kw: (calls.append(name), own(*a, **kw))[1])
            _declined(fi.FlashAttnFunc, lambda: f(x, x, x)).sum().backward()
        assert calls == [name]
    with pytest.raises(RuntimeError, match="query and key must have the same dtype"):
        f(q, q.to(torch.float16), q)
    with pytest.raises(RuntimeError, match="Number of heads in key/value must divide"):
        f(q, q[:, :, :3], q[:, :, :3])
    with pytest.raises(RuntimeError, match="p_dropout must be in"):
        f(q, q, q, dropout_p=1.0)
    with pytest.raises(RuntimeError, match="CUDA device"):
        f(q.cpu(), q.cpu(), q.cpu())
    with pytest.raises(RuntimeError, match="16-byte aligned"):
        w = torch.empty(q.numel() + 4, dtype=q.dtype, device=DEV)[4:].view(q.shape)
        f(w, q, q)


@pytest.mark.parametrize("path", ["native", "python"])
def test_autograd_rules(monkeypatch, path):
    """an input changed in place before the backward, gradients of gradients, in-place use of the result, a functorch transform"""
    if path == "python":
        monkeypatch.setattr(fi.FlashAttnFunc, "native", None)
        monkeypatch.setattr(fi.FlashAttnQKVPackedFunc, "native", None)
    base = _gen(2, 64, 3, 4, 64, seed=1).requires_grad_()
    x = base * 1
    out = flash_attn.flash_attn_qkvpacked_func(x, causal=True)
    x.add_(1)
    with pytest.raises(RuntimeError, match="inplace"):
        out.sum().backward()
    q = _gen(2, 64, 4, 64, seed=1).requires_grad_()
    out = flash_attn.flash_attn_func(q, q, q)
    out.mul_(2)                       # out is saved
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()
    out = flash_attn.flash_attn_func(q, q, q)
    (g,) = torch.autograd.grad(out.float().square().sum(), q, create_graph=True)
    assert not g.requires_grad        # the backward pass has no derivative of its own
    out = flash_attn.flash_attn_func(q, q, q)
    torch.autograd.grad(out.sum(), q)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out.sum(), q)
    with pytest.raises(RuntimeError):
        torch.vmap(lambda t: flash_attn.flash_attn_func(t, t, t))(_gen(2, 2, 64, 4, 64))


@pytest.mark.parametrize("sq,h,hk,d,cap,rot", [(1, 8, 2, 128, 600, 64), (4, 16, 2, 64, 3000, 0), (130, 8, 8, 128, 700, 128), (1, 32, 8, 128, 20000, 128)])
def test_kvcache_same_bits_as_the_python_path(sq, h, hk, d, cap, rot):
    from oracle import attention_oracle as orc
    b = 3
    q, kn, vn = _gen(b, sq, h, d, seed=1), _gen(b, sq, hk, d, seed=2), _gen(b, sq, hk, d, seed=3)
    kc, vc = _gen(b, cap, hk, d, seed=4), _gen(b, cap, hk, d, seed=5)
    lens = torch.tensor([0, 333, cap - sq], dtype=torch.int32, device=DEV)
    idx = torch.tensor([1, 0, 2], dtype=torch.int32, device=DEV)
    cos = sin = None
    if rot:
        cos, sin = (t.to(DEV) for t in orc.rotary_table(cap, rot, dtype=torch.bfloat16))
    for kw in (dict(k=kn, v=vn, rotary_cos=cos, rotary_sin=sin, cache_seqlens=lens, causal=True), dict(cache_seqlens=lens, window_size=(100, 0)),
               dict(k=kn, v=vn, cache_seqlens=lens, cache_batch_idx=idx, causal=True, rotary_cos=cos, rotary_sin=sin, rotary_interleaved=False),
               dict(cache_seqlens=lens, num_splits=3, softmax_scale=0.2), dict(), dict(cache_seqlens=50)):
        results = []
        for native in (True, False):
            k2, v2 = kc.clone(), vc.clone()
            host = nat.host
            taken = []

            class Watch:
                @staticmethod
                def with_kvcache(*a):
                    taken.append(host.with_kvcache(*a) if native else None)
                    return taken[-1]

            nat.host = Watch
            try:
                results.append((flash_attn.flash_attn_with_kvcache(q, k2, v2, **kw), k2, v2))
            finally:
                nat.host = host
            assert (taken[0] is not None) == (native and not isinstance(kw.get("cache_seqlens"), int)), kw.keys()
        for a, c in zip(*results):
            assert torch.equal(a, c), kw.keys()


@pytest.mark.parametrize("inter", [False, True])
@pytest.mark.parametrize("d,rot,cs", [(64, 64, torch.bfloat16), (128, 64, torch.float32), (80, 24, torch.bfloat16)])
def test_rotary_same_bits_as_the_python_path(monkeypatch, d, rot, cs, inter):
    from flash_attn.layers.rotary import apply_rotary_emb_qkv_
    qkv = _gen(2, 70, 3, 4, d, seed=1)
    cos, sin = _gen(100, rot // 2, seed=2, dtype=cs), _gen(100, rot // 2, seed=3, dtype=cs)
    native = nat.host.rotary_emb_qkv_
    results = []
    for on in (True, False):
        taken = []
        host = type("Host", (), {"rotary_emb_qkv_": staticmethod(lambda *a: (taken.append(native(*a) if on else None), taken[-1])[1])})
        with monkeypatch.context() as m:
            m.setattr(nat, "host", host)
            x = qkv.clone()
            y = apply_rotary_emb_qkv_(x, cos, sin, interleaved=inter, seqlen_offsets=7)
            assert (taken[0] is not None) == on
            assert y is not x and y._base is x and y.data_ptr() == x.data_ptr() and not y.requires_grad
            w = qkv.clone()
            with torch.no_grad():
                z = apply_rotary_emb_qkv_(w, cos, sin)
            results.append((x, z, y))
            # what the Python layer keeps: gradients, strided projections, a table of each, offsets on the device
            taken.clear()
            g = qkv.clone().requires_grad_()
            leaf = apply_rotary_emb_qkv_(g * 1, cos, sin)
            assert leaf.requires_grad
            apply_rotary_emb_qkv_(qkv.clone().transpose(0, 1).contiguous().transpose(0, 1), cos, sin)
            apply_rotary_emb_qkv_(qkv.clone(), cos, sin, seqlen_offsets=torch.tensor([0, 5], device=DEV))
            assert taken == [None] * 3
            apply_rotary_emb_qkv_(qkv.clone(), cos, sin, cos, sin)
            assert len(taken) == 3
            with pytest.raises(AssertionError):
                apply_rotary_emb_qkv_(qkv.clone(), cos, sin, seqlen_offsets=40)
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_rotary_asks_what_stands_in_the_python_layer(monkeypatch):
    """a program's own apply_rotary is called, not passed by"""
    from flash_attn.layers import rotary
    qkv, cos, sin = _gen(2, 20, 3, 4, 64, seed=1), _gen(30, 32, seed=2), _gen(30, 32, seed=3)
    want = rotary.apply_rotary_emb_qkv_(qkv.clone(), cos, sin)
    own, calls = rotary.apply_rotary, []
    monkeypatch.setattr(rotary, "apply_rotary", lambda *a, **kw: (calls.append(1), own(*a, **kw))[1])
    assert torch.equal(rotary.apply_rotary_emb_qkv_(qkv.clone(), cos, sin), want) and calls


@pytest.mark.parametrize("grad", [False, True])
def test_errors_of_the_library(monkeypatch, grad):
    """the library's message and a reset of the counter words, on either path (the library looks at alignment before any launch)"""
    cu = torch.tensor([0, 33, 64], dtype=torch.int32, device=DEV)
    k = _gen(64, 4, 64, seed=2)
    q = _gen(64 * 4 * 64 + 1, seed=1)[1:].view(64, 4, 64)
    own, reset = nat._reset_counters, []
    monkeypatch.setattr(nat, "_reset_counters", lambda device: (reset.append(device), own(device))[1])
    with torch.inference_mode(), torch.cuda.stream(torch.cuda.Stream()):      # words that a call in inference mode made are cleared like any others
        nat._counters(q.device, nat.WORK_COUNTER_WORDS).fill_(7)
        torch.cuda.synchronize()

    def run(call, *args):
        with pytest.raises(RuntimeError) as e:
            call(q.detach().requires_grad_(grad), k, k, cu, cu, 33, 33, *args)
        return str(e.value)

    want = "q, k, v, o, k_new and v_new must be 16-byte aligned"
    assert run(fi.FlashAttnVarlenFunc.native, 0.0, None, False, (-1, -1), False) == want and reset == [q.device]
    monkeypatch.setattr(fi.FlashAttnVarlenFunc, "native", None)
    assert run(flash_attn.flash_attn_varlen_func) == want and reset == [q.device] * 2
    assert all(not t[:nat.WORK_COUNTER_WORDS].any() for t in nat._COUNTERS.values())


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="two devices")
def test_capture_state_of_the_tensors_device():
    """a capture on the second device while the first is the current one: dropout is left to the Python layer, which takes the seed for
    each replay, and the words of a work list belong to the graph"""
    q = _gen(2, 64, 4, 64, seed=1).to("cuda:1")
    cu = torch.tensor([0, 64, 128], dtype=torch.int32, device="cuda:1")
    dropped, packed = (fi.FlashAttnFunc.native, (q, q, q, 0.1, None, True, (-1, -1), False)), (fi.FlashAttnVarlenFunc.native, (*[q.flatten(0, 1)] * 3, cu, cu, 64, 64, 0.0, None, True, (-1, -1), False))
    want = packed[0](*packed[1])
    with torch.cuda.device(1):
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            with torch.cuda.device(0):
                assert dropped[0](*dropped[1]) is None
                before = {k: t.numel() for k, t in nat._COUNTERS.items()}
                got = packed[0](*packed[1])
                assert all(t.numel() == before.get(k, 16) for k, t in nat._COUNTERS.items())
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want)
