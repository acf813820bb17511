"""The generator's words by value (fa_fwd_rng, fa_varlen_fwd_rng): as by fa_set_rng_state and the forward after it."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("varlen", [False, True], ids=["dense", "varlen"])
@pytest.mark.parametrize("p", [0.0, 0.3])
@pytest.mark.parametrize("b,sq,sk,h,hk,d", [
    (2, 40, 70, 2, 1, 64),                                        # the general kernel
    (3, 300, 257, 4, 2, 64), (2, 400, 500, 2, 2, 128),            # pipelined
    (9, 1030, 2100, 16, 4, 96),                                   # ping-pong
    (2, 200, 300, 2, 1, 256),                                     # pairs of waves
])
def test_words_by_value(monkeypatch, b, sq, sk, h, hk, d, p, varlen):
    """same output, log-sum-exp and words for the backward, whether the launch brings the words or a launch ahead of it"""
    from flash_attn import _native as nat
    gen = torch.Generator().manual_seed(sq + d)
    mk = lambda *s: torch.randn(*s, generator=gen).to(torch.bfloat16).to(DEV)
    if varlen:
        lens_q, lens_k = torch.arange(b) % 3 * sq // 2, torch.full((b,), sk)       # the first sequence has no rows
        lens_q[-1] = sq
        cu_q, cu_k = (torch.nn.functional.pad(t.cumsum(0), (1, 0)).to(torch.int32).to(DEV) for t in (lens_q, lens_k))
        q, k, v = mk(int(lens_q.sum()), h, d), mk(b * sk, hk, d), mk(b * sk, hk, d)
        call = lambda: nat.varlen_fwd(q, k, v, None, cu_q, cu_k, sq, sk, p, d ** -0.5, False, True, -1, -1, False, None)
    else:
        q, k, v = mk(b, sq, h, d), mk(b, sk, hk, d), mk(b, sk, hk, d)
        call = lambda: nat.fwd(q, k, v, None, p, d ** -0.5, True, -1, -1, False, None)
    torch.manual_seed(77)
    want = call()
    name = "fa_varlen_fwd" if varlen else "fa_fwd"
    by_value = getattr(nat.lib, name + "_rng")
    by_value.argtypes, by_value.restype = [ctypes.POINTER(nat.FaFwdParams), ctypes.c_uint64, ctypes.c_uint64, ctypes.c_void_p], ctypes.c_int
    seen = []

    def words(ptr, seed, offset, stream):
        seen[:] = [seed.value, offset.value]
        return 0

    class Lib:
        def __getattr__(self, n):
            return getattr(real, n)

    real = nat.lib
    lib = Lib()
    lib.fa_set_rng_state = words
    setattr(lib, name, lambda params, stream: by_value(params, *(seen or (1, 2)), stream))
    monkeypatch.setattr(nat, "lib", lib)
    torch.manual_seed(77)
    got = call()
    assert len(seen) == (2 if p > 0 else 0)
    assert torch.equal(got[0], want[0])
    for i in range(b):                     # (a packed sequence's rows of the log-sum-exp end with it)
        n = int(lens_q[i]) if varlen else sq
        assert torch.equal(got[5][i, :, :n], want[5][i, :, :n])
    if p > 0:
        assert got[7].tolist() == want[7].tolist() == [77, seen[1]]


@pytest.mark.parametrize("name", ["fa_fwd_rng", "fa_varlen_fwd_rng"])
def test_words_of_a_call_without_query_rows(name):
    """nothing attends, and no attention kernel runs: the words arrive all the same"""
    from flash_attn import _native as nat
    t = torch.zeros(4, 2, 64, dtype=torch.float16, device=DEV)
    words = torch.zeros(2, dtype=torch.int64, device=DEV)
    cu = torch.tensor([0, 0], dtype=torch.int32, device=DEV)
    p = nat.FaFwdParams()
    p.q = p.k = p.v = p.o = t.data_ptr()
    p.softmax_lse = t.data_ptr()
    if "varlen" in name:
        p.cu_seqlens_q = p.cu_seqlens_k = cu.data_ptr()
    for f in ("q", "k", "v", "o"):
        for n, v in (("batch", 512), ("row", 128), ("head", 64)):
            setattr(p, "%s_%s_stride" % (f, n), v)
    p.b, p.h, p.h_k, p.d, p.seqlen_q, p.seqlen_k = 1, 2, 2, 64, 0, 4
    p.window_left = p.window_right = -1
    p.is_seqlens_k_cumulative, p.dtype, p.softmax_scale, p.p_dropout, p.rng_state = 1, 0, 0.125, 0.5, words.data_ptr()
    f = getattr(nat.lib, name)
    f.argtypes, f.restype = [ctypes.POINTER(nat.FaFwdParams), ctypes.c_uint64, ctypes.c_uint64, ctypes.c_void_p], ctypes.c_int
    assert f(p, 5, 7, torch.cuda.current_stream().cuda_stream) == 0, nat.lib.fa_last_error()
    assert words.tolist() == [5, 7]
