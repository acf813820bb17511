"""The pipelined kernel with split keys (equal parts of the tiles that a row block sees), with (position, grouped head) rows, and with
waves that split the keys of a launch of few rows."""
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
    (96, 1300, 3, 3, 64, torch.float16), (130, 961, 2, 2, 128, torch.bfloat16), (257, 2049, 4, 2, 96, torch.bfloat16),
    (300, 700, 1, 1, 32, torch.bfloat16), (128, 64, 2, 2, 128, torch.bfloat16)])
def test_split_rows(sq, sk, h, hk, d, dtype, num_splits, mode):
    """parts of no tile at all (64 parts of few tiles, rows of a window, rows that a causal mask leaves without keys: sk < sq), ragged
    last tiles, and the plan of the library (0)"""
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
    assert name == "pipelined" and (num_splits == 0 or split == (num_splits > 1 and sk > 64))
    kw = dict(causal=causal, window_size=(wl, wr))
    ref, lse_ref, pt = orc.attention_reference_pair(q, k, v, **kw)
    ok, err, bound = orc.tolerance_ok(out.cpu(), ref, pt, 3.0, 1e-5)
    assert ok, (err, bound)
    assert orc.lse_ok(lse.cpu(), lse_ref, 1e-3)[0]


@pytest.mark.parametrize("mode", ["causal", "full", "window"])
@pytest.mark.parametrize("num_splits", [0, 1, 3])
@pytest.mark.parametrize("inter", [False, True])
@pytest.mark.parametrize("sq,h,hk,d,rot", [(33, 6, 2, 128, 64), (12, 16, 2, 64, 64), (127, 10, 2, 96, 96), (50, 64, 8, 128, 0)])
def test_packed_rows(sq, h, hk, d, rot, inter, num_splits, mode):
    """96 rows (12 x 8, 33 x 3 = 99) and more of few positions and grouped heads: blocks that begin and end inside a position's group,
    lengths that leave a causal row without keys, appended with and without rotary"""
    from flash_attn import _native as nat
    dtype, cap = torch.bfloat16, 900
    mk = _mk(sq + d + num_splits, dtype)
    lens = torch.tensor([0, 64, 333, cap - sq, 1, 63, 500, 127], dtype=torch.int32)        # (16 row blocks or more)
    b = len(lens)
    q, kc, vc, kn, vn = mk(b, sq, h, d), mk(b, cap, hk, d), mk(b, cap, hk, d), mk(b, sq, hk, d), mk(b, sq, hk, d)
    cos, sin = orc.rotary_table(cap, rot, dtype=dtype) if rot else (None, None)
    dev = lambda t: None if t is None else t.to(DEV)
    causal, wl, wr = mode == "causal", -1, -1
    if mode == "window":
        wl, wr = 70, 2
    kd, vd = kc.to(DEV), vc.to(DEV)
    out, lse = nat.fwd_kvcache(q.to(DEV), kd, vd, kn.to(DEV), vn.to(DEV), lens.to(DEV), dev(cos), dev(sin), None, None, d ** -0.5, causal, wl, wr, inter, num_splits)
    assert nat.last_kernel()[0] in ("pipelined", "tiled_tickets")
    if num_splits:
        assert nat.last_kernel()[0] == "pipelined"
    kw = dict(causal=causal, window_size=(wl, wr), rotary_interleaved=inter)
    o_ref, l_ref, k_ref, v_ref = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, lens, **kw)
    o_pt, _, _, _ = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, lens, upcast=False, reorder_ops=True, **kw)
    ok, err, bound = orc.tolerance_ok(out.cpu(), o_ref, o_pt, 3.0, 1e-5)
    assert ok, (err, bound)
    assert orc.lse_ok(lse.cpu(), l_ref, 1e-3)[0]
    assert torch.equal(vd.cpu(), v_ref)


def test_not_a_number_passes_through_the_merge():
    """A row whose scores are not numbers is NaN with a log-sum-exp of +inf whether its keys are split or not; its neighbours are not."""
    from flash_attn import _native as nat
    mk = _mk(3, torch.bfloat16)
    q, k, v = mk(1, 128, 2, 128).to(DEV), mk(1, 1500, 2, 128).to(DEV), mk(1, 1500, 2, 128).to(DEV)
    q[0, 77, 1, 5] = float("nan")
    got = [nat.fwd_kvcache(q, k, v, None, None, None, None, None, None, None, 128 ** -0.5, True, -1, -1, True, n) for n in (1, 4)]
    for out, lse in got:
        bad = torch.isnan(out).any(-1)
        assert bad[0, 77, 1] and bad.sum() == 1 and torch.isinf(lse).sum() == 1 and lse[0, 1, 77] == float("inf")
    keep = ~torch.isnan(got[0][0])
    assert torch.allclose(got[0][0][keep].float(), got[1][0][keep].float(), atol=1e-2)


@pytest.mark.parametrize("mode", ["causal", "full", "window", "window_right"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("b,sq,sk,h,hk,d", [
    (1, 40, 20, 3, 3, 64), (2, 33, 64, 2, 2, 128), (1, 96, 65, 2, 2, 96), (1, 127, 383, 2, 2, 32), (1, 512, 512, 16, 4, 64),      # four waves
    (1, 1000, 130, 8, 8, 128), (1, 513, 513, 16, 8, 128), (2, 512, 770, 16, 16, 64), (1, 1025, 1025, 9, 3, 80)])                   # two, and the last size past four
def test_key_waves(b, sq, sk, h, hk, d, dtype, mode):
    """fewer tiles than waves (20 to 65 keys), a last wave with one tile less, rows without keys (sk < sq), ragged row groups"""
    from flash_attn import _native as nat
    mk = _mk(sq + sk, dtype)
    q, k, v = mk(b, sq, h, d), mk(b, sk, hk, d), mk(b, sk, hk, d)
    causal, wl, wr = mode == "causal", -1, -1
    if mode == "window":
        wl, wr = 40, 9
    if mode == "window_right":
        wr = 3
    r = nat.fwd(q.to(DEV), k.to(DEV), v.to(DEV), None, 0.0, d ** -0.5, causal, wl, wr, False, None)
    # (one tile of 64 keys is not shared by waves)
    assert nat.last_kernel()[0] == ("tiled" if d <= 64 and sk <= 64 else "pipelined") and not nat.last_kernel()[2]
    ref, lse_ref, pt = orc.attention_reference_pair(q, k, v, causal=causal, window_size=(wl, wr))
    ok, err, bound = orc.tolerance_ok(r[0].cpu(), ref, pt, 2.0, 1e-5)
    assert ok, (err, bound)
    assert orc.lse_ok(r[5].cpu(), lse_ref, 1e-3)[0]


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("lens,h,d", [([40, 0, 1, 100], 4, 64), ([200, 33], 8, 128), ([64, 31], 2, 96)])
def test_key_waves_packed_sequences(lens, h, d, causal):
    from flash_attn import _native as nat
    mk = _mk(sum(lens), torch.bfloat16)
    total, mx = sum(lens), max(lens)
    q, k, v = mk(total, h, d), mk(total, h, d), mk(total, h, d)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    r = nat.varlen_fwd(q.to(DEV), k.to(DEV), v.to(DEV), None, cu.to(DEV), cu.to(DEV), mx, mx, 0.0, d ** -0.5, False, causal, -1, -1, False, None)
    assert nat.last_kernel()[0] == "pipelined"
    for i, n in enumerate(lens):
        if n == 0:
            continue
        sl = slice(int(cu[i]), int(cu[i + 1]))
        ref, lse_ref, pt = orc.attention_reference_pair(q[None, sl], k[None, sl], v[None, sl], causal=causal)
        ok, err, bound = orc.tolerance_ok(r[0][None, sl].cpu(), ref, pt, 2.0, 1e-5)
        assert ok, (i, err, bound)
        assert orc.lse_ok(r[5][i:i + 1, :, :n].cpu(), lse_ref, 1e-3)[0]


@pytest.mark.parametrize("rot", [0, 64])
def test_key_waves_over_caches(rot):
    """caches of which most, some and none of the capacity is filled; appended, rotated; q and out the same memory"""
    from flash_attn import _native as nat
    mk = _mk(5 + rot, torch.bfloat16)
    b, sq, h, hk, d, cap = 4, 100, 8, 8, 128, 1500
    lens = torch.tensor([0, 1, 700, cap - sq], dtype=torch.int32)
    q, kc, vc, kn, vn = mk(b, sq, h, d), mk(b, cap, hk, d), mk(b, cap, hk, d), mk(b, sq, hk, d), mk(b, sq, hk, d)
    cos, sin = orc.rotary_table(cap, rot, dtype=torch.bfloat16) if rot else (None, None)
    dev = lambda t: None if t is None else t.to(DEV)
    o_ref, l_ref, _, _ = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, lens, causal=True)
    o_pt, _, _, _ = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, lens, upcast=False, reorder_ops=True, causal=True)
    for same in (False, True):
        qd = q.to(DEV)
        out, lse = nat.fwd_kvcache(qd, kc.to(DEV), vc.to(DEV), kn.to(DEV), vn.to(DEV), lens.to(DEV), dev(cos), dev(sin), None, qd if same else None, d ** -0.5,
                                   True, -1, -1, True, 0)
        assert nat.last_kernel()[0] == "pipelined" and not nat.last_kernel()[2]
        ok, err, bound = orc.tolerance_ok(out.cpu(), o_ref, o_pt, 3.0, 1e-5)
        assert ok, (same, err, bound)
        assert orc.lse_ok(lse.cpu(), l_ref, 1e-3)[0]


def test_key_waves_pass_on_what_is_not_a_number():
    from flash_attn import _native as nat
    mk = _mk(3, torch.bfloat16)
    q, k, v = mk(1, 128, 2, 64).to(DEV), mk(1, 300, 2, 64).to(DEV), mk(1, 300, 2, 64).to(DEV)
    q[0, 77, 1, 5] = float("nan")
    k[0, :, 0] = float("-inf")                       # head 0: q . k is -inf or NaN everywhere
    r = nat.fwd(q, k, v, None, 0.0, 0.125, True, -1, -1, False, None)
    assert nat.last_kernel()[0] == "pipelined"
    bad = torch.isnan(r[0]).any(-1)
    assert bad[0, 77, 1] and bad[0, :, 1].sum() == 1 and r[5][0, 1, 77] == float("inf") and torch.isfinite(r[5][0, 1]).sum() == 127


@pytest.mark.parametrize("form", ["dense", "packed", "cache", "cache_rotary_in_place"])
@pytest.mark.parametrize("b,sq,sk,h,d", [(5, 33, 800, 32, 128), (9, 64, 1030, 16, 80), (3, 48, 2100, 64, 96)])
def test_key_waves_of_many_heads(b, sq, sk, h, d, form):
    """129 to 256 (batch, head) pairs, up to 64 rows, no mask, long keys: a 256-row block would use a quarter of its rows at most"""
    from flash_attn import _native as nat
    mk = _mk(sq + sk, torch.bfloat16)
    q, k, v = mk(b, sq, h, d), mk(b, sk, h, d), mk(b, sk, h, d)
    few = [0, b - 1]
    if form == "packed":
        cu = lambda n: torch.arange(0, (b + 1) * n, n, dtype=torch.int32, device=DEV)
        r = nat.varlen_fwd(q.flatten(0, 1).to(DEV), k.flatten(0, 1).to(DEV), v.flatten(0, 1).to(DEV), None, cu(sq), cu(sk), sq, sk, 0.0, d ** -0.5, False, False, -1, -1, False, None)
        out, lse = r[0].view(b, sq, h, d), r[5]
    elif form == "dense":
        r = nat.fwd(q.to(DEV), k.to(DEV), v.to(DEV), None, 0.0, d ** -0.5, False, -1, -1, False, None)
        out, lse = r[0], r[5]
    else:
        rot = form != "cache"
        lens = torch.tensor([(sk - sq) * (i + 1) // b for i in range(b)], dtype=torch.int32)
        kn, vn = mk(b, sq, h, d), mk(b, sq, h, d)
        cos, sin = orc.rotary_table(sk, 64, dtype=torch.bfloat16) if rot else (None, None)
        dev = lambda t: None if t is None else t.to(DEV)
        qd = q.to(DEV)
        out, lse = nat.fwd_kvcache(qd, k.to(DEV), v.to(DEV), kn.to(DEV), vn.to(DEV), lens.to(DEV), dev(cos), dev(sin), None, qd if rot else None, d ** -0.5,
                                   False, -1, -1, False, 0)
    assert nat.last_kernel()[0] == "pipelined" and not nat.last_kernel()[2]
    for i in few:
        s = slice(i, i + 1)
        if form.startswith("cache"):
            a = (q[s], k[s], v[s], kn[s], vn[s], cos, sin, lens[s])
            ref, lse_ref, _, _ = orc.kvcache_forward(*a, rotary_interleaved=False)
            pt, _, _, _ = orc.kvcache_forward(*a, upcast=False, reorder_ops=True, rotary_interleaved=False)
        else:
            ref, lse_ref, pt = orc.attention_reference_pair(q[s], k[s], v[s])
        ok, err, bound = orc.tolerance_ok(out[s].cpu(), ref, pt, 3.0, 1e-5)
        assert ok, (i, err, bound)
        assert orc.lse_ok(lse[s].cpu(), lse_ref, 1e-3)[0]


def test_many_heads_past_the_memory_side_cache():
    """K and V of 256 MiB: the 256-row blocks of the ping-pong kernel"""
    from flash_attn import _native as nat
    gen = torch.Generator().manual_seed(1)
    mk = lambda *s: torch.randn(*s, generator=gen).to(torch.bfloat16)
    q, k, v = mk(8, 40, 32, 128), mk(8, 2048, 32, 128), mk(8, 2048, 32, 128)
    r = nat.fwd(q.to(DEV), k.to(DEV), v.to(DEV), None, 0.0, 128 ** -0.5, False, -1, -1, False, None)
    assert nat.last_kernel()[0] == "pingpong"
    ref, lse_ref, pt = orc.attention_reference_pair(q[7:], k[7:], v[7:])
    assert orc.tolerance_ok(r[0][7:].cpu(), ref, pt, 2.0, 1e-5)[0] and orc.lse_ok(r[5][7:].cpu(), lse_ref, 1e-3)[0]


@pytest.mark.parametrize("b,sq,h,hk,cap,kernel,split", [
    (3, 40, 16, 2, 9000, "pipelined", True), (1, 40, 16, 2, 9000, "tiled", True), (1, 40, 16, 2, 5000, "pipelined", True),      # 18 blocks, 6 of long and shorter caches
    (9, 40, 8, 1, 5000, "pipelined", True), (3, 100, 6, 2, 700, "pipelined", True),                 # streams that do not divide over the XCDs
    (42, 40, 16, 2, 4200, "pipelined", True), (42, 40, 16, 2, 4000, "pipelined", False)])           # 252 blocks of long and of short caches
def test_lines_of_packed_rows(b, sq, h, hk, cap, kernel, split):
    """both sides of the lines between the pipelined and the general kernel for packed rows; a full, an empty and a short cache"""
    from flash_attn import _native as nat
    mk = _mk(b + cap, torch.bfloat16)
    d = 64
    q, kc, vc = mk(b, sq, h, d), mk(b, cap, hk, d), mk(b, cap, hk, d)
    lens = torch.tensor([(cap, 0, 300, 4000)[i % 4] for i in range(b)], dtype=torch.int32)
    out, lse = nat.fwd_kvcache(q.to(DEV), kc.to(DEV), vc.to(DEV), None, None, lens.to(DEV), None, None, None, None, d ** -0.5, True, -1, -1, False, 0)
    assert nat.last_kernel()[0] == kernel and nat.last_kernel()[2] == split
    for i in {0, min(1, b - 1), min(2, b - 1)}:
        a = (q[i:i + 1], kc[i:i + 1], vc[i:i + 1], None, None, None, None, lens[i:i + 1])
        ref, lse_ref, _, _ = orc.kvcache_forward(*a, causal=True)
        pt, _, _, _ = orc.kvcache_forward(*a, causal=True, upcast=False, reorder_ops=True)
        ok, err, bound = orc.tolerance_ok(out[i:i + 1].cpu(), ref, pt, 3.0, 1e-5)
        assert ok, (i, err, bound)
        assert orc.lse_ok(lse[i:i + 1].cpu(), lse_ref, 1e-3)[0]
