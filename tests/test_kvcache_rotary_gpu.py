"""Chunks appended with rotary on the kernels that rotate the q rows as matrix operands (rotate_row): which pieces of a row a lane
holds, and where their partners lie, differs from kernel to kernel and with the rotated share of the head dim."""
import sys

import pytest
import torch

from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("inter", [False, True])
@pytest.mark.parametrize("sq,h,d,rot,cap,dtype,kernel", [
    (257, 48, 128, 128, 2048, torch.bfloat16, "pingpong"),        # whole row rotated: partners in the lane
    (257, 48, 128, 48, 2048, torch.float16, "pingpong"),          # partners in other lanes
    (300, 48, 80, 80, 2050, torch.bfloat16, "pingpong"),          # odd number of pieces per lane, columns past the head dim
    (129, 64, 64, 64, 700, torch.float16, "pipelined"),
    (140, 64, 96, 16, 700, torch.bfloat16, "pipelined"),
    (300, 48, 192, 192, 512, torch.bfloat16, None),               # 32 rows per wave
    (128, 64, 200, 160, 300, torch.float16, None),                 # 16 rows per wave, head dim of no bucket
])
def test_chunk_with_rotary_rotated_as_operand(sq, h, d, rot, cap, dtype, kernel, inter):
    import flash_attn._native as nat
    print("rotary as operand", sq, h, d, rot, cap, dtype, inter, flush=True)
    sys.stdout.flush()
    b, hk = 3, 8
    g = torch.Generator().manual_seed(sq + d + rot)
    mk = lambda *s: torch.randn(*s, generator=g).to(dtype)
    q, kc, vc, kn, vn = mk(b, sq, h, d), mk(b, cap, hk, d), mk(b, cap, hk, d), mk(b, sq, hk, d), mk(b, sq, hk, d)
    lens = torch.tensor([cap - sq, 0, 3], dtype=torch.int32)
    cos, sin = orc.rotary_table(cap, rot, dtype=dtype)
    q_d, kc_d, vc_d = q.to(DEV), kc.to(DEV), vc.to(DEV)
    # tables that start at an odd element of their storage: the requests for them assume no alignment
    odd = [torch.cat([t.new_zeros(1), t.flatten()]).to(DEV)[1:].view(t.shape) for t in (cos, sin)]
    out, lse = nat.fwd_kvcache(q_d, kc_d, vc_d, kn.to(DEV), vn.to(DEV), lens.to(DEV), *odd, None, None, d ** -0.5, True, -1, -1, inter, 0)
    if kernel:
        assert nat.last_kernel()[0] == kernel
    else:
        assert nat.last_kernel()[0] != "tiled"
    assert torch.equal(q_d.cpu(), q)
    kw = dict(causal=True, rotary_interleaved=inter)
    o_ref, l_ref, k_ref, v_ref = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, lens, **kw)
    o_pt, _, _, _ = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, lens, upcast=False, reorder_ops=True, **kw)
    ok, err, bound = orc.tolerance_ok(out.cpu(), o_ref, o_pt, 3.0, 1e-5)
    assert ok, (err, bound)
    assert orc.lse_ok(lse.cpu(), l_ref, 1e-3)[0]
    assert torch.equal(vc_d.cpu(), v_ref)
    assert torch.allclose(kc_d.cpu().float(), k_ref.float(), rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("inter", [False, True])
@pytest.mark.parametrize("sq,h,hk,d,rot,cap,dtype", [
    (1, 32, 8, 128, 128, 4096, torch.bfloat16),      # split; whole row rotated: partners in the lane
    (1, 16, 8, 128, 128, 200, torch.float16),        # one chunk
    (4, 8, 2, 128, 64, 1000, torch.bfloat16),        # 16 packed rows, partners in other lanes, columns that are not rotated
    (3, 5, 1, 64, 64, 300, torch.float16),           # one pair of pieces per lane; a packed row that is not there
    (2, 4, 4, 64, 16, 2500, torch.bfloat16),
    (1, 8, 2, 96, 96, 4096, torch.bfloat16),         # odd number of pieces that are real
    (2, 8, 2, 200, 160, 700, torch.float16),
    (1, 8, 1, 256, 256, 3000, torch.bfloat16),
])
def test_decode_rows_rotated_as_operand(sq, h, hk, d, rot, cap, dtype, inter):
    """Decoding steps: q rows rotated as operands, the new key rows piece by piece by the workgroup that appends them."""
    import flash_attn._native as nat
    print("decode with rotary", sq, h, hk, d, rot, cap, dtype, inter, flush=True)
    b = 4
    g = torch.Generator().manual_seed(sq + d + rot + cap)
    mk = lambda *s: torch.randn(*s, generator=g).to(dtype)
    q, kc, vc, kn, vn = mk(b, sq, h, d), mk(b, cap, hk, d), mk(b, cap, hk, d), mk(b, sq, hk, d), mk(b, sq, hk, d)
    lens = torch.tensor([cap - sq, 0, 127, cap // 2], dtype=torch.int32)      # new rows in the last, the first and across two chunks
    cos, sin = orc.rotary_table(cap, rot, dtype=dtype)
    q_d, kc_d, vc_d = q.to(DEV), kc.to(DEV), vc.to(DEV)
    odd = [torch.cat([t.new_zeros(1), t.flatten()]).to(DEV)[1:].view(t.shape) for t in (cos, sin)]
    out, lse = nat.fwd_kvcache(q_d, kc_d, vc_d, kn.to(DEV), vn.to(DEV), lens.to(DEV), *odd, None, None, d ** -0.5, True, -1, -1, inter, 0)
    assert nat.last_kernel()[0] == "decode"
    kw = dict(causal=True, rotary_interleaved=inter)
    o_ref, l_ref, k_ref, v_ref = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, lens, **kw)
    o_pt, _, _, _ = orc.kvcache_forward(q, kc, vc, kn, vn, cos, sin, lens, upcast=False, reorder_ops=True, **kw)
    ok, err, bound = orc.tolerance_ok(out.cpu(), o_ref, o_pt, 3.0, 1e-5)
    assert ok, (err, bound)
    assert orc.lse_ok(lse.cpu(), l_ref, 1e-3)[0]
    assert torch.equal(vc_d.cpu(), v_ref)
    assert torch.allclose(kc_d.cpu().float(), k_ref.float(), rtol=1e-3, atol=1e-3)
