"""What a decoding call with new rows promises about memory: every new row is in the cache before any batch entry attends.
Decode launches append in the attention kernel where no entry can see another one's rows; the cases here are those in
which it can, so that the append has to be a launch of its own."""
import sys

import pytest
import torch

from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _say(*a):
    print("[append order]", *a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("cap,first,num_splits", [(640, 10, 1), (640, 253, 0), (640, 300, 5), (16384, 9000, 0)])    # the last: tickets
@pytest.mark.parametrize("shared", ["cache_batch_idx", "expanded"])
@pytest.mark.parametrize("sq,rotary", [(1, 0), (2, 64)])
def test_entries_that_share_a_cache_row(sq, rotary, shared, cap, first, num_splits):
    """Entries of successive lengths on one cache row: each sees the rows that the shorter ones append in the same call."""
    _say(shared, cap, first, num_splits, sq, rotary)
    from flash_attn import _native as nat
    dtype, h, hk, d, n_rows, per_row = torch.bfloat16, 8, 2, 64, 3, 4
    if shared == "expanded":
        n_rows, per_row = 1, 12
    b = n_rows * per_row
    gen = torch.Generator().manual_seed(cap + first + sq)
    mk = lambda *s: torch.randn(*s, generator=gen).to(dtype)
    q, kn, vn = mk(b, sq, h, d), 4 * mk(b, sq, hk, d), mk(b, sq, hk, d)      # (large keys: a missing one shows)
    kc, vc = mk(n_rows, cap, hk, d), mk(n_rows, cap, hk, d)
    idx = torch.tensor([i % n_rows for i in range(b)], dtype=torch.int32)
    lens = torch.tensor([first + sq * (i // n_rows) for i in range(b)], dtype=torch.int32)
    cos, sin = orc.rotary_table(cap, rotary, dtype=dtype) if rotary else (None, None)
    dev = lambda t: None if t is None else t.to(DEV)
    kd, vd = kc.to(DEV), vc.to(DEV)
    k_arg, v_arg = (kd, vd) if shared == "cache_batch_idx" else (kd.expand(b, -1, -1, -1), vd.expand(b, -1, -1, -1))
    out, lse = nat.fwd_kvcache(q.to(DEV), k_arg, v_arg, kn.to(DEV), vn.to(DEV), lens.to(DEV), dev(cos), dev(sin),
                               idx.to(DEV) if shared == "cache_batch_idx" else None, None, d ** -0.5, True, -1, -1, False, num_splits)
    kw = dict(cache_seqlens=lens, cache_batch_idx=idx, causal=True, rotary_interleaved=False)
    ref, lse_ref, k_ref, v_ref = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, **kw)
    pt, _, _, _ = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, upcast=False, reorder_ops=True, **kw)
    assert torch.equal(vd.cpu(), v_ref)
    assert torch.allclose(kd.cpu().float(), k_ref.float(), rtol=1e-2, atol=1e-2)       # (bf16 rounding of the rotation)
    ok, err, bound = orc.tolerance_ok(out.cpu(), ref, pt, 3.0, 1e-5)
    assert ok, (err, bound)
    assert orc.lse_ok(lse.cpu(), lse_ref, 1e-3)[0]


@pytest.mark.parametrize("n_new", [1, 4])
@pytest.mark.parametrize("which", ["k", "v"])
def test_results_over_the_memory_of_the_new_rows(which, n_new):
    """o laid over k_new or v_new, with other heads and strides: an unsplit decode launch writes o while it runs, and every
    new row must have reached the cache before."""
    _say("o over", which, n_new)
    from flash_attn import _native as nat
    dtype, b, sq, h, hk, d, cap = torch.bfloat16, 48, 1, 8, 2, 64, 256
    gen = torch.Generator().manual_seed(n_new)
    mk = lambda *s: torch.randn(*s, generator=gen).to(dtype)
    q, kn, vn, kc, vc = mk(b, sq, h, d), mk(b, n_new, hk, d), mk(b, n_new, hk, d), mk(b, cap, hk, d), mk(b, cap, hk, d)
    lens = torch.tensor([(i * 37) % (cap - n_new) for i in range(b)], dtype=torch.int32)
    store = torch.zeros(b * max(sq * h, n_new * hk) * d, dtype=dtype, device=DEV)
    over = store[:b * n_new * hk * d].view(b, n_new, hk, d)
    over.copy_(kn if which == "k" else vn)
    out = store[:b * sq * h * d].view(b, sq, h, d)
    kd, vd = kc.to(DEV), vc.to(DEV)
    k_arg, v_arg = (over, vn.to(DEV)) if which == "k" else (kn.to(DEV), over)
    nat.fwd_kvcache(q.to(DEV), kd, vd, k_arg, v_arg, lens.to(DEV), None, None, None, out, d ** -0.5, True, -1, -1, False, 1)
    assert nat.last_kernel()[0] == "decode"
    kw = dict(cache_seqlens=lens, causal=True)
    ref, _, k_ref, v_ref = orc.kvcache_forward(q, kc, vc, kn, vn, **kw)
    pt, _, _, _ = orc.kvcache_forward(q, kc, vc, kn, vn, upcast=False, reorder_ops=True, **kw)
    assert torch.equal(kd.cpu(), k_ref) and torch.equal(vd.cpu(), v_ref)
    ok, err, bound = orc.tolerance_ok(out.cpu(), ref, pt, 3.0, 1e-5)
    assert ok, (err, bound)
