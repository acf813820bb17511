"""Decode kernels with 17 to 32 packed (position, grouped head) rows: two sets of matrix columns per wave."""
import pytest
import torch

from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(out, lse, q, kc, vc, kn, vn, cos, sin, lens, idx, **kw):
    """the rules of the other kv-cache tests: three times the error of a 16-bit reference, 1e-3 on the log-sum-exp"""
    for i in idx:
        sl = slice(i, i + 1)
        cut = lambda t: None if t is None else t[sl]
        o_ref, l_ref, _, _ = orc.kvcache_forward(q[sl], kc[sl], vc[sl], cut(kn), cut(vn), cos, sin, lens[sl], **kw)
        o_pt, _, _, _ = orc.kvcache_forward(q[sl], kc[sl], vc[sl], cut(kn), cut(vn), cos, sin, lens[sl], upcast=False, reorder_ops=True, **kw)
        ok, err, bound = orc.tolerance_ok(out[sl], o_ref, o_pt, 3.0, 1e-5)
        assert ok, (i, int(lens[i]), err, bound)
        assert orc.lse_ok(lse[sl], l_ref, 1e-3)[0], (i, int(lens[i]))


@pytest.mark.parametrize("window", [(-1, -1), (40, 3)], ids=["whole", "window"])
@pytest.mark.parametrize("num_splits", [1, 0, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("sq,h,hk,d", [(4, 16, 2, 128), (17, 3, 3, 64), (1, 32, 1, 96), (3, 18, 3, 128), (2, 20, 2, 40), (31, 2, 2, 128), (1, 17, 1, 64)])
def test_up_to_32_rows_take_the_decode_kernel(sq, h, hk, d, dtype, num_splits, window):
    """17, 18, 20, 24, 31 and 32 rows; cache lengths on the edges of a wave's 32-key step, of its range and of a chunk, an empty
    and a full cache; new rows appended with rotary, with a window (the append is a launch of its own) and without."""
    from flash_attn import _native as nat
    gen = torch.Generator().manual_seed(100 * sq + d + num_splits)
    mk = lambda *s: torch.randn(*s, generator=gen).to(dtype)
    cap, rot = 640, 32
    lens = torch.tensor([0, 1, 31, 32, 127, 255, 256, 511, cap - sq], dtype=torch.int32)
    b = len(lens)
    q, kc, vc, kn, vn = mk(b, sq, h, d), mk(b, cap, hk, d), mk(b, cap, hk, d), mk(b, sq, hk, d), mk(b, sq, hk, d)
    cos, sin = orc.rotary_table(cap, rot, dtype=dtype)
    kd, vd = kc.to(DEV), vc.to(DEV)
    out, lse = nat.fwd_kvcache(q.to(DEV), kd, vd, kn.to(DEV), vn.to(DEV), lens.to(DEV), cos.to(DEV), sin.to(DEV), None, None, d ** -0.5,
                               True, window[0], window[1], False, num_splits)
    assert nat.last_kernel()[0] == "decode"
    _check(out.cpu(), lse.cpu(), q, kc, vc, kn, vn, cos, sin, lens, range(b), causal=True, window_size=window, rotary_interleaved=False)
    for i, n in enumerate(lens.tolist()):
        assert torch.equal(vd[i, n:n + sq].cpu(), vn[i]) and torch.equal(vd[i, :n].cpu(), vc[i, :n])


@pytest.mark.parametrize("b,sq,h,hk,cap,append,left,decode", [
    (4, 33, 8, 8, 8192, False, -1, False),                                                                                              # 33 rows
    (8, 3, 64, 8, 573, True, -1, True), (2, 4, 64, 8, 40, True, -1, True), (32, 4, 64, 8, 300, True, -1, True),                                 # grouped heads, appended
    (2, 4, 64, 8, 513, False, -1, True), (2, 4, 64, 8, 512, False, -1, False), (8, 4, 64, 8, 1024, False, -1, False), (32, 4, 64, 8, 1025, False, -1, True),
    (16, 4, 64, 8, 8192, False, -1, True), (8, 4, 64, 8, 16500, False, -1, True),
    (3, 20, 8, 8, 256, True, -1, True), (3, 20, 8, 8, 257, True, -1, False), (3, 20, 8, 8, 513, True, -1, True), (8, 20, 8, 8, 1024, True, -1, False),   # ungrouped
    (8, 20, 8, 8, 1025, True, -1, True), (16, 20, 8, 8, 4096, False, -1, False), (16, 20, 8, 8, 4097, False, -1, True),
    (33, 4, 64, 8, 512, True, -1, True), (33, 4, 64, 8, 512, False, -1, False), (33, 4, 64, 8, 513, True, -1, False), (33, 4, 64, 8, 2048, True, -1, False),  # 264 streams
    (33, 4, 64, 8, 2049, False, -1, True), (64, 4, 64, 8, 512, True, -1, True), (64, 4, 64, 8, 512, False, -1, False), (64, 4, 64, 8, 513, False, -1, True),  # 512
    (17, 4, 64, 8, 1025, False, 100, True), (17, 4, 64, 8, 1024, True, 100, False), (17, 20, 8, 8, 2048, False, 100, False), (17, 20, 8, 8, 2049, True, 100, True)])
def test_lines_of_17_to_32_rows(b, sq, h, hk, cap, append, left, decode):
    """both sides of the lines between the decode kernel and the tiled one or the key waves"""
    from flash_attn import _native as nat
    gen = torch.Generator().manual_seed(sq)
    mk = lambda *s: torch.randn(*s, generator=gen).to(torch.bfloat16)
    d = 32
    q, kc, vc = mk(b, sq, h, d), mk(b, cap, hk, d), mk(b, cap, hk, d)
    kn, vn = (mk(b, sq, hk, d), mk(b, sq, hk, d)) if append else (None, None)
    top = cap - sq if append else cap
    lens = torch.randint(1 if append else sq, top + 1, (b,), generator=gen, dtype=torch.int32)
    lens[:2] = torch.tensor([0 if append else sq, top])
    cos, sin = orc.rotary_table(cap, 32, dtype=torch.bfloat16) if append else (None, None)
    dev = lambda t: None if t is None else t.to(DEV)
    kd, vd = dev(kc), dev(vc)
    out, lse = nat.fwd_kvcache(dev(q), kd, vd, dev(kn), dev(vn), dev(lens), dev(cos), dev(sin), None, None, d ** -0.5, True, left, -1, False, 0)
    assert nat.last_kernel()[0].startswith("decode") == decode
    _check(out.cpu(), lse.cpu(), q, kc, vc, kn, vn, cos, sin, lens, (0, 1, b - 1), causal=True, window_size=(left, -1), rotary_interleaved=False)
    if append:
        for i in (0, 1, b - 1):
            n = int(lens[i])
            assert torch.equal(vd[i, n:n + sq].cpu(), vn[i])


@pytest.mark.parametrize("b,sq,h,hk,d,cap,kernels", [
    (2, 1, 8, 2, 128, 1500, {"decode"}), (2, 4, 16, 2, 64, 1500, {"decode"}), (64, 1, 32, 8, 64, 8192, {"decode", "decode_tickets"}),
    (64, 4, 64, 8, 32, 8192, {"decode", "decode_tickets"}), (40, 4, 64, 8, 32, 2048, {"tiled", "tiled_tickets"}), (2, 40, 4, 2, 128, 1500, {"tiled", "tiled_tickets"}),
    (3, 33, 6, 2, 256, 9000, {"tiled", "tiled_tickets"})])
def test_not_a_number_passes_through_the_merge(b, sq, h, hk, d, cap, kernels):
    """A row one of whose chunks holds a score that is not a number is NaN with a log-sum-exp of +inf whether its keys are split or not; rows
    of other kv heads and sequences are as without it."""
    from flash_attn import _native as nat
    gen = torch.Generator(device=DEV).manual_seed(cap + sq)
    mk = lambda *s: torch.randn(*s, generator=gen, device=DEV, dtype=torch.bfloat16)
    q, kc, vc = mk(b, sq, h, d), mk(b, cap, hk, d), mk(b, cap, hk, d)
    lens = torch.full((b,), cap - 7, dtype=torch.int32, device=DEV)
    used = set()
    run = lambda n: (nat.fwd_kvcache(q, kc, vc, None, None, lens, None, None, None, None, d ** -0.5, True, -1, -1, False, n), used.add(nat.last_kernel()[0]))[0]
    splits = (1, 0, 3)
    want = [run(n) for n in splits]
    kc[1, 700, 1, 3] = float("nan")
    got = [run(n) for n in splits]
    assert used <= kernels, used
    hit = slice(h // hk, 2 * (h // hk))
    for (out, lse), (out0, lse0) in zip(got, want):
        assert torch.isnan(out[1, :, hit]).all() and (lse[1, hit] == float("inf")).all()
        out[1, :, hit], lse[1, hit] = out0[1, :, hit], lse0[1, hit]
        assert torch.equal(out, out0) and torch.equal(lse, lse0)


@pytest.mark.parametrize("cache", [True, False])
def test_one_position_on_many_heads_behind_a_window(cache):
    """17 to 32 heads of a kv head and a left bound: the decode kernel at any number of streams, for the heads are not laid out as rows"""
    from flash_attn import _native as nat
    gen = torch.Generator().manual_seed(5)
    mk = lambda *s: torch.randn(*s, generator=gen).to(torch.bfloat16)
    b, h, hk, cap, d = 20, 160, 8, 300, 64
    q, kc, vc = mk(b, 1, h, d), mk(b, cap, hk, d), mk(b, cap, hk, d)
    lens = torch.tensor([cap - 7 * i for i in range(b)], dtype=torch.int32) if cache else torch.full((b,), cap, dtype=torch.int32)
    out, lse = nat.fwd_kvcache(q.to(DEV), kc.to(DEV), vc.to(DEV), None, None, lens.to(DEV) if cache else None, None, None, None, None, d ** -0.5, True, 100, -1, False, 0)
    assert nat.last_kernel()[0] == "decode"
    _check(out.cpu(), lse.cpu(), q, kc, vc, None, None, None, None, lens, (0, 1, b - 1), causal=True, window_size=(100, -1))
