"""Which calls skip autograd's node (flash_attn_interface._apply): only those in which autograd, a functorch transform, forward
mode, tracing or compilation has no part."""
import torch

from flash_attn import flash_attn_interface as fi


class _Fn:
    @staticmethod
    def apply(*a):
        return ("apply",) + a

    @staticmethod
    def forward(ctx, *a):
        ctx.save_for_backward(*a)
        ctx.anything = a
        return ("forward",) + a


def _route(*ts):
    got = fi._apply(_Fn, ts, *ts, 7)
    assert got[1:] == (*ts, 7)
    return got[0]


def test_no_gradient_asked_for():
    x, w = torch.zeros(2), torch.zeros(2, requires_grad=True)
    assert _route(x, x, x) == "forward"
    assert _route(x, w, x) == "apply"
    assert _route((w * 2)) == "apply"
    with torch.no_grad():
        assert _route(x, w, x) == "forward"
        assert _route(w * 2) == "forward"
    with torch.inference_mode():
        assert _route(torch.zeros(2)) == "forward"


def test_transforms_keep_the_function():
    seen = []

    def f(t):
        seen.append(_route(t))
        return t * 1

    torch.vmap(f)(torch.zeros(3, 2))
    torch.func.grad(lambda t: f(t).sum())(torch.zeros(2))
    torch.func.jvp(f, (torch.zeros(2),), (torch.ones(2),))
    with torch.autograd.forward_ad.dual_level():
        f(torch.zeros(2))                     # a plain tensor inside a level: its own values may carry tangents elsewhere
        f(torch.autograd.forward_ad.make_dual(torch.zeros(2), torch.ones(2)))
    # a transform is active, though this tensor is not part of it
    plain = torch.zeros(2)
    torch.vmap(lambda t: (f(plain), t)[1])(torch.zeros(3, 2))
    # a tensor that outlived its transform
    leak = []
    torch.vmap(lambda t: (leak.append(t), t)[1])(torch.zeros(3, 2))
    assert fi._functorch_wrapped(leak[0])
    assert fi._apply(_Fn, (leak[0],), 1) == ("apply", 1)
    torch.jit.trace(f, torch.zeros(2), check_trace=False)
    assert seen == ["apply"] * len(seen) and len(seen) == 7, seen


def test_entry_points_go_through_it(monkeypatch):
    calls = []
    monkeypatch.setattr(fi, "_apply", lambda fn, tensors, *a: calls.append((fn, tensors, a)))
    q = torch.zeros(1)
    fi.flash_attn_func(q, q, q, 0.1, 0.5, True, (1, 2), True)
    fi.flash_attn_qkvpacked_func(q, 0.1, 0.5, True, (1, 2), True)
    fi.flash_attn_kvpacked_func(q, q, 0.1, 0.5, True, (1, 2), True)
    fi.flash_attn_varlen_func(q, q, q, q, q, 3, 4, 0.1, 0.5, True, (1, 2), True)
    fi.flash_attn_varlen_qkvpacked_func(q, q, 3, 0.1, 0.5, True, (1, 2), True)
    fi.flash_attn_varlen_kvpacked_func(q, q, q, q, 3, 4, 0.1, 0.5, True, (1, 2), True)
    assert [(c[0].__name__, len(c[1]), len(c[2])) for c in calls] == [
        ("FlashAttnFunc", 3, 8), ("FlashAttnQKVPackedFunc", 1, 6), ("FlashAttnKVPackedFunc", 2, 7),
        ("FlashAttnVarlenFunc", 3, 12), ("FlashAttnVarlenQKVPackedFunc", 1, 8), ("FlashAttnVarlenKVPackedFunc", 2, 11)]
    assert all(c[2][-1] is True and c[2][-2] == (1, 2) for c in calls)
