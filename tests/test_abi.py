"""CPU-only checks of the C ABI: the library loads, exports every symbol the header declares, the
Python mirror of the params struct has the library's size, and the pure host functions agree with
the oracle.  No kernel is launched."""
import ctypes
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "fa_mi355x.h")
LIB = os.path.join(ROOT, "flash-attention_amd", "flash_attn", "libfa_mi355x.so")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        import __graft_entry__
        __graft_entry__.build()
    return ctypes.CDLL(LIB)


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(fa_[a-z_0-9]+)\s*\(", text)))


def test_header_symbols_exported(lib):
    names = declared_symbols()
    assert {"fa_fwd", "fa_varlen_fwd", "fa_fwd_kvcache", "fa_plan_splits", "fa_last_error",
            "fa_num_splits_heuristic_reference", "fa_version", "fa_sizeof_params", "fa_bwd", "fa_varlen_bwd",
            "fa_sizeof_bwd_params", "fa_rotary", "fa_sizeof_rotary_params"} <= set(names)
    for n in names:
        assert hasattr(lib, n), "library does not export %s" % n


def test_a_library_that_lacks_functions_is_refused():
    """an ImportError that names them, not an AttributeError somewhere in the module"""
    from flash_attn import _native as nat

    class Lib:
        pass

    for name in nat._CALLS:
        setattr(Lib, name, None)
    nat._require(Lib())
    del Lib.fa_fwd_rng, Lib.fa_bwd_lent
    with pytest.raises(ImportError, match="does not have fa_fwd_rng, fa_bwd_lent; rebuild the library"):
        nat._require(Lib())


def test_another_library_is_refused(tmp_path):
    source = tmp_path / "empty.c"
    source.write_text("int fa_version(void) { return 1; }")
    other = str(tmp_path / "libother.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", other, str(source)], check=True)
    got = subprocess.run([sys.executable, "-c", "import flash_attn"], capture_output=True, text=True,
                         env={**os.environ, "FLASH_ATTN_MI355X_LIB": other, "PYTHONPATH": os.path.join(ROOT, "flash-attention_amd")})
    assert got.returncode != 0 and "ImportError: flash_attn: %s does not have fa_fwd_rng" % other in got.stderr


def test_kernel_ids_of_the_header_have_names():
    """Every FA_KERNEL_* id that fa_last_kernel() can return is decoded by flash_attn._native.last_kernel()."""
    import flash_attn._native as nat
    text = open(HEADER).read()
    ids = {name: int(val) for name, val in re.findall(r"#define\s+FA_KERNEL_((?!FLAG_)[A-Z0-9_]+)\s+(\d+)\b", text)}
    assert ids["NONE"] == 0 and len(ids) >= 10 and len(set(ids.values())) == len(ids)
    assert set(ids.values()) == set(nat.KERNEL_NAMES)
    for name, val in ids.items():
        assert nat.KERNEL_NAMES[val] == name.lower(), (name, val, nat.KERNEL_NAMES[val])


def test_struct_mirror_size(lib):
    import flash_attn._native as nat
    lib.fa_sizeof_params.restype = ctypes.c_int32
    assert lib.fa_sizeof_params() == ctypes.sizeof(nat.FaFwdParams)
    lib.fa_sizeof_bwd_params.restype = ctypes.c_int32
    assert lib.fa_sizeof_bwd_params() == ctypes.sizeof(nat.FaBwdParams)
    lib.fa_sizeof_rotary_params.restype = ctypes.c_int32
    assert lib.fa_sizeof_rotary_params() == ctypes.sizeof(nat.FaRotaryParams)


def test_backward_argument_errors_do_not_abort(lib):
    import flash_attn._native as nat
    p = nat.FaBwdParams()
    lib.fa_bwd.argtypes = [ctypes.POINTER(nat.FaBwdParams), ctypes.c_void_p]
    lib.fa_bwd.restype = ctypes.c_int
    lib.fa_varlen_bwd.argtypes = [ctypes.POINTER(nat.FaBwdParams), ctypes.c_void_p]
    lib.fa_varlen_bwd.restype = ctypes.c_int
    lib.fa_last_error.restype = ctypes.c_char_p
    assert lib.fa_bwd(ctypes.byref(p), None) != 0 and b"must be set" in lib.fa_last_error()
    for n in ("dout", "q", "k", "v", "out", "softmax_lse", "dq", "dk", "dv", "softmax_d"):
        setattr(p, n, 16)                       # never dereferenced: the checks below fail first
    p.b, p.h, p.h_k, p.d, p.seqlen_q, p.seqlen_k, p.seqlen_q_rounded, p.dtype = 1, 4, 3, 64, 8, 8, 128, 1
    assert lib.fa_bwd(ctypes.byref(p), None) != 0 and b"Number of heads" in lib.fa_last_error()
    p.h_k, p.d = 2, 260
    assert lib.fa_bwd(ctypes.byref(p), None) != 0 and b"at most 256" in lib.fa_last_error()
    p.d = 64
    assert lib.fa_varlen_bwd(ctypes.byref(p), None) != 0 and b"cu_seqlens" in lib.fa_last_error()
    p.q_row_stride = 4
    assert lib.fa_bwd(ctypes.byref(p), None) != 0 and b"strides" in lib.fa_last_error()
    p.q_row_stride, p.dk_row_stride = 0, 4     # gradients leave 16 bytes per lane as well
    assert lib.fa_bwd(ctypes.byref(p), None) != 0 and b"strides" in lib.fa_last_error()
    p.dk_row_stride, p.dv = 0, 24
    assert lib.fa_bwd(ctypes.byref(p), None) != 0 and b"16-byte aligned" in lib.fa_last_error()
    p.dv, p.p_dropout = 16, 0.1
    assert lib.fa_bwd(ctypes.byref(p), None) != 0 and b"rng_state" in lib.fa_last_error()
    p.p_dropout = 1.0
    assert lib.fa_bwd(ctypes.byref(p), None) != 0 and b"p_dropout" in lib.fa_last_error()


def test_reference_heuristic_matches_oracle(lib):
    from oracle import attention_oracle as orc
    f = lib.fa_num_splits_heuristic_reference
    f.argtypes = [ctypes.c_int32] * 4
    f.restype = ctypes.c_int
    assert f(48, 108, 64, 128) == 2       # csrc/flash_attn/flash_api.cpp:206-211
    for blocks in (1, 2, 5, 13, 48, 80, 87, 200):
        for sms in (80, 108, 132, 256):
            for nb in (1, 2, 7, 64, 257):
                assert f(blocks, sms, nb, 128) == orc.num_splits_heuristic_reference(blocks, sms, nb, 128)


def test_argument_errors_do_not_abort(lib):
    import flash_attn._native as nat
    p = nat.FaFwdParams()
    lib.fa_fwd.argtypes = [ctypes.POINTER(nat.FaFwdParams), ctypes.c_void_p]
    lib.fa_fwd.restype = ctypes.c_int
    lib.fa_last_error.restype = ctypes.c_char_p
    assert lib.fa_fwd(ctypes.byref(p), None) != 0
    assert lib.fa_last_error()
    n = ctypes.c_int32(0)
    lib.fa_plan_splits.argtypes = [ctypes.POINTER(nat.FaFwdParams), ctypes.c_int32, ctypes.POINTER(ctypes.c_int32)]
    p.q = p.k = p.v = p.o = p.softmax_lse = 16   # never dereferenced by the planner
    p.b, p.h, p.h_k, p.d, p.seqlen_q, p.seqlen_k, p.dtype = 64, 64, 8, 128, 1, 32768, 1
    assert lib.fa_plan_splits(ctypes.byref(p), 2, ctypes.byref(n)) == 0
    assert 1 < n.value <= 128
    p.num_splits = 1
    assert lib.fa_plan_splits(ctypes.byref(p), 2, ctypes.byref(n)) == 0 and n.value == 1
    p.d = 260
    assert lib.fa_plan_splits(ctypes.byref(p), 2, ctypes.byref(n)) != 0


def test_one_pass_backward_takes_bounded_out_strides():
    """The one-pass backward kernel fetches rows of `out` by 32-bit offsets; the other kernels take any stride of it."""
    from flash_attn import _native as nat
    p = nat.FaBwdParams()
    p.b, p.h, p.h_k, p.d, p.seqlen_q, p.seqlen_k, p.o_row_stride = 64, 8, 8, 64, 512, 512, 8 * 64
    assert nat.lib.fa_bwd_scratch_bytes(ctypes.byref(p), 0, 0) > 0
    for stride in (-8 * 64, 1 << 23, 1 << 40):
        p.o_row_stride = stride
        assert nat.lib.fa_bwd_scratch_bytes(ctypes.byref(p), 0, 0) == 0
    p.o_row_stride = (1 << 23) - 8
    assert nat.lib.fa_bwd_scratch_bytes(ctypes.byref(p), 0, 0) > 0


def test_bwd_params_end_where_older_callers_end(lib):
    """A caller built before scratch could be lent hands over a struct that ends with rng_state: what lies behind it in its
    memory must not be read (a pointer taken from there would be written through)."""
    from flash_attn import _native as nat
    assert nat.FaBwdParams._fields_[-1][0] == "rng_state"
    assert lib.fa_sizeof_bwd_params() == nat.FaBwdParams.rng_state.offset + 8 == 12 * 8 + 24 * 8 + 12 * 4 + 4 + 4 + 8

    class Caller(ctypes.Structure):
        _fields_ = [("p", nat.FaBwdParams), ("behind", ctypes.c_uint64 * 2)]

    c = Caller()
    for n in ("dout", "q", "k", "v", "out", "softmax_lse", "dq", "dk", "dv", "softmax_d"):
        setattr(c.p, n, 16)                       # never dereferenced: the row stride is refused
    c.p.b, c.p.h, c.p.h_k, c.p.d, c.p.seqlen_q, c.p.seqlen_k, c.p.seqlen_q_rounded, c.p.dtype = 1, 2, 2, 64, 8, 8, 128, 1
    c.p.q_row_stride = 1 << 23
    c.behind[:] = [8, 1 << 40]                    # would be refused as a misaligned pointer
    lib.fa_bwd.argtypes = [ctypes.POINTER(nat.FaBwdParams), ctypes.c_void_p]
    lib.fa_last_error.restype = ctypes.c_char_p
    assert lib.fa_bwd(ctypes.byref(c.p), None) != 0 and b"row strides must be below" in lib.fa_last_error()
    lent = nat.lib.fa_bwd_lent
    assert lent(ctypes.byref(c.p), 0, 0, 8, 1 << 40, None) != 0 and b"16-byte aligned" in nat.lib.fa_last_error()
    assert lent(None, 0, 0, None, 0, None) != 0 and b"NULL" in nat.lib.fa_last_error()
    c.p.cu_seqlens_q = 16
    assert lent(ctypes.byref(c.p), 0, 0, None, 0, None) != 0 and b"cu_seqlens" in nat.lib.fa_last_error()


def _bwd_params(b, h, h_k, s, d=64, packed=False):
    from flash_attn import _native as nat
    p = nat.FaBwdParams()
    p.b, p.h, p.h_k, p.d, p.seqlen_q, p.seqlen_k = b, h, h_k, d, s, s
    if packed:
        p.cu_seqlens_q = p.cu_seqlens_k = 16            # never dereferenced on the host
    return p


def test_backward_scratch_is_bounded():
    """Scratch grows with the grouped heads and the declared length: what it may take has an end, past which two passes run."""
    from flash_attn import _native as nat
    sizes = {(b, g, s): nat.lib.fa_bwd_scratch_bytes(ctypes.byref(_bwd_params(b, 8 * g, 8, s)), 0, 0)
             for b in (64, 512, 4096) for g in (1, 2, 8, 32, 64) for s in (256, 512, 1024)}
    assert max(sizes.values()) <= 1 << 29 and sizes[512, 1, 512] > 0
    assert sizes[512, 64, 1024] == sizes[4096, 32, 1024] == 0


def test_backward_without_room_for_scratch_runs_in_two_passes(monkeypatch):
    import torch
    from flash_attn import _native as nat
    p = _bwd_params(512, 8, 8, 512)
    assert nat.lib.fa_bwd_scratch_bytes(ctypes.byref(p), 0, 0) > 0

    def no_room(*a, **k):
        raise torch.cuda.OutOfMemoryError("no room")

    monkeypatch.setattr(torch, "empty", no_room)
    assert nat._lend_scratch(p, torch.device("cpu")) is None


def test_one_pass_backward_takes_only_launches_that_fill_the_cus():
    """Calls on both sides of the line, past 128 keys, where scratch is asked for exactly if the one-pass kernel runs; every one
    measured (times beside the rule)."""
    from flash_attn import _native as nat
    one = lambda pairs, g, s: nat.lib.fa_bwd_scratch_bytes(ctypes.byref(_bwd_params(pairs // 8, 8 * g, 8, s)), 0, 0) > 0
    for pairs, g, s in [(160, 1, 256), (1024, 1, 256), (256, 1, 512), (512, 1, 512), (1024, 1, 512), (384, 1, 1024), (1024, 1, 1024), (768, 1, 512),
                        (192, 2, 256), (384, 2, 512), (384, 4, 512), (384, 8, 256), (384, 16, 256)]:
        assert one(pairs, g, s), (pairs, g, s)
    for pairs, g, s in [(128, 1, 256), (192, 1, 512), (520, 1, 512), (320, 1, 1024), (640, 1, 1024), (1024, 1, 2048), (128, 2, 256), (520, 2, 512),
                        (256, 4, 512), (768, 4, 1024), (256, 8, 256), (520, 8, 256), (320, 8, 512), (128, 32, 256)]:
        assert not one(pairs, g, s), (pairs, g, s)


def test_one_pass_backward_of_packed_batches_weighs_the_longest_sequence():
    """The launch lasts as long as the longest sequence takes: how many such sequences the tokens would make decides."""
    from flash_attn import _native as nat
    one = lambda b, h, s, tokens, g=1: nat.lib.fa_bwd_scratch_bytes(ctypes.byref(_bwd_params(b, h * g, h, s, packed=True)), tokens, tokens) > 0
    mixed, one_of_16 = lambda b, s: int(b * s * 0.56), lambda b, s: int(b * s * (1 / 16 + 15 / 128))
    assert one(64, 16, 512, mixed(64, 512)) and one(128, 8, 1024, mixed(128, 1024)) and one(256, 8, 512, one_of_16(256, 512))
    assert not one(64, 8, 1024, one_of_16(64, 1024)) and not one(128, 8, 1024, one_of_16(128, 1024)) and not one(16, 8, 512, mixed(16, 512))
    assert not one(24, 8, 512, mixed(24, 512), 8) and one(64, 8, 512, mixed(64, 512), 8)
    assert not one(65, 8, 512, 65 * 512) and one(64, 8, 512, 64 * 512)              # of one length: rounds, the second nearly empty
    assert not one(64, 16, 512, 0)                                                  # total unknown


ONE_PASS, WHOLE, HALVES, PARTS = 1, 2, 3, 4        # FA_BWD_FORM_*


def _form(p, tokens=0, lent=0):
    from flash_attn import _native as nat
    return nat.lib.fa_bwd_plan_form(ctypes.byref(p), tokens, tokens, lent)


def test_wide_packed_backward_shares_key_blocks_by_the_tokens_there_are():
    """Head dims 193-256, and 129-256 with dropout: whether two workgroups share a key block goes by the weight of the blocks that
    the tokens fill, not by the declared maximum times the batch.  Every call measured (times beside the rule)."""
    def packed(b, h, h_k, s, d, causal, p_dropout=0.0):
        p = _bwd_params(b, h, h_k, s, d, packed=True)
        p.is_causal, p.p_dropout, p.window_left, p.window_right = causal, p_dropout, -1, -1
        return p

    one_long = lambda b, s, share: s + (b - 1) * (s // share)
    for b, h, h_k, s, d, causal, p_dropout, tokens in [
            (19, 4, 1, 1349, 256, 1, 0.0, one_long(19, 1349, 16)), (51, 4, 1, 1314, 224, 1, 0.0, one_long(51, 1314, 16)),
            (61, 4, 1, 743, 256, 1, 0.1, one_long(61, 743, 16)), (39, 4, 1, 517, 256, 0, 0.1, one_long(39, 517, 16)),
            (50, 4, 1, 1735, 256, 0, 0.1, one_long(50, 1735, 16)), (24, 4, 1, 684, 192, 1, 0.1, 24 * 684),
            (3, 1, 1, 8015, 160, 1, 0.1, 8800), (4, 4, 2, 3697, 256, 1, 0.0, 8500),
            (2, 4, 1, 3380, 256, 0, 0.1, 3600), (3, 2, 1, 1977, 256, 0, 0.1, 4300)]:
        assert _form(packed(b, h, h_k, s, d, causal, p_dropout), tokens) == HALVES, (b, s, d)
    for b, h, h_k, s, d, causal, p_dropout, tokens in [
            (16, 32, 2, 3900, 256, 1, 0.0, 4 * 3900 + 12 * 240), (4, 8, 2, 3966, 256, 0, 0.0, one_long(4, 3966, 16)), (30, 4, 1, 3404, 160, 0, 0.1, 5100),
            (20, 4, 1, 1879, 256, 1, 0.0, 20 * 1879), (7, 1, 1, 3107, 256, 0, 0.0, 9626), (64, 16, 16, 2000, 256, 1, 0.1, 80000)]:
        assert _form(packed(b, h, h_k, s, d, causal, p_dropout), tokens) == WHOLE, (b, s, d)
    # without dropout at head dims 129-192 there is no form with halves
    assert _form(packed(19, 4, 1, 1349, 192, 1), one_long(19, 1349, 16)) == WHOLE
    # tokens unknown: as many as the maximum allows
    assert _form(packed(19, 4, 1, 1349, 256, 1), 0) == WHOLE and _form(packed(2, 4, 1, 1349, 256, 1), 0) == HALVES


def test_wide_dense_backward_shares_key_blocks_that_leave_cus_idle():
    """The same for dense batches: up to 128 key blocks, or a mask that leaves as little to do."""
    def dense(b, h, h_k, sq, sk, d, causal, left=-1, p_dropout=0.0):
        p = _bwd_params(b, h, h_k, sk, d)
        p.seqlen_q, p.is_causal, p.window_left, p.window_right, p.p_dropout = sq, causal, left, -1, p_dropout
        return p
    for a in [(2, 4, 2, 2048, 2048, 256, 0), (12, 4, 1, 1377, 1377, 200, 1), (6, 4, 4, 1227, 662, 136, 1, 512, 0.1), (14, 4, 2, 3441, 625, 136, 1, -1, 0.1),
              (6, 4, 4, 672, 672, 256, 1, 512)]:
        assert _form(dense(*a)) == HALVES, a
    for a in [(9, 2, 1, 623, 1888, 256, 0), (14, 2, 1, 2095, 2095, 256, 1), (52, 1, 1, 469, 469, 256, 1), (16, 16, 4, 2039, 2039, 256, 1), (2, 4, 2, 2048, 2048, 192, 0)]:
        assert _form(dense(*a)) == WHOLE, a
    assert _form(dense(2, 4, 2, 2048, 2048, 257, 0)) == 0 and _form(dense(0, 4, 2, 2048, 2048, 256, 0)) == 0


def test_wide_dense_backward_cuts_key_blocks_only_where_that_wins():
    """Head dims 129-256: blocks of few steps stay whole or shared by two workgroups, with whatever room is lent; longer ones are cut.  Every
    call measured (times beside the rule)."""
    def dense(b, h, h_k, sq, sk, d, causal, left=-1, p_dropout=0.0):
        p = _bwd_params(b, h, h_k, sk, d)
        p.seqlen_q, p.is_causal, p.window_left, p.window_right, p.p_dropout = sq, causal, left, -1, p_dropout
        return _form(p, 0, 1 << 29)
    for a in [(6, 1, 1, 666, 666, 224, 0), (2, 16, 8, 340, 340, 224, 0), (12, 4, 2, 343, 343, 256, 1), (2, 32, 8, 150, 150, 256, 0), (1, 2, 2, 1999, 1999, 256, 1, 512),
              (9, 1, 1, 537, 537, 192, 0, -1, 0.1), (1, 4, 1, 134, 134, 200, 0)]:
        assert dense(*a) == HALVES, a
    for a in [(11, 2, 2, 552, 138, 160, 0), (8, 4, 2, 307, 307, 160, 0)]:
        assert dense(*a) == WHOLE, a
    for a in [(4, 16, 4, 2039, 2039, 256, 1), (6, 1, 1, 1000, 1000, 224, 0), (2, 8, 2, 2054, 2054, 256, 1), (6, 4, 1, 6315, 6315, 160, 1), (2, 8, 8, 852, 852, 136, 1),
              (1, 8, 1, 2048, 2048, 128, 1)]:
        assert dense(*a) == PARTS, a


def test_backward_lent_less_than_it_asks_for_runs_as_without():
    """One byte less than fa_bwd_lend_bytes is nothing lent, whichever form the room is for."""
    import random
    from flash_attn import _native as nat
    rng, asked = random.Random(0), {ONE_PASS: 0, PARTS: 0}
    for _ in range(8000):
        h_k, g = rng.choice([1, 2, 4, 8, 16]), rng.choice([1, 2, 4, 8])
        p = _bwd_params(rng.randint(1, 128), h_k * g, h_k, rng.randint(64, 2048), rng.choice([32, 64, 128, 192, 256]))
        p.seqlen_q, p.is_causal, p.window_left, p.window_right = rng.randint(64, 2048), rng.randint(0, 1), rng.choice([-1, -1, 64, 256]), -1
        n = nat.lib.fa_bwd_lend_bytes(ctypes.byref(p), 0, 0)
        assert 0 <= n <= 1 << 29
        if n:
            asked[_form(p, 0, n)] += 1
            assert _form(p, 0, n - 1) == _form(p, 0, 0) in (WHOLE, HALVES)
            assert _form(p, 0, 1 << 40) == _form(p, 0, n)
    assert min(asked.values()) > 100, asked


def test_backward_plan_of_a_shape_is_made_once_and_in_little_time():
    """The plan of one shape does not show in that of another, in one thread or several, and neither its first nor a repeated asking
    costs what a call does: least time of several, long sequences of few heads (421 and 210 us each time, before)."""
    import random
    import threading
    import time
    from flash_attn import _native as nat

    def shape(b, h, h_k, s, causal, p_dropout=0.0):
        p = _bwd_params(b, h, h_k, s, 128)
        p.is_causal, p.window_left, p.window_right, p.p_dropout = causal, -1, -1, p_dropout
        return p

    lend = lambda p: nat.lib.fa_bwd_lend_bytes(ctypes.byref(p), 0, 0)
    shapes = [shape(b, 8, h_k, s, c) for b in (1, 3) for h_k in (1, 2, 8) for s in (700, 2048, 5000) for c in (0, 1)]
    want = [lend(p) for p in shapes]
    assert len(set(want)) > 10
    failed = []

    def ask(seed):
        rng = random.Random(seed)
        for _ in range(300):
            i = rng.randrange(len(shapes))
            if lend(shapes[i]) != want[i] or (_form(shapes[i], 0, want[i]) == PARTS) != (want[i] > 0):
                failed.append(i)

    threads = [threading.Thread(target=ask, args=(seed,)) for seed in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed

    def least(p, *between):
        best = 1.0
        for _ in range(20):
            for other in between:
                lend(other)
            t = time.perf_counter()
            lend(p)
            best = min(best, time.perf_counter() - t)
        return best

    other = shapes[0]
    assert least(shape(3, 2, 1, 30140, 1), other) < 150e-6
    long = shape(1, 8, 1, 32768, 1)
    assert least(long) < least(long, other) / 5


def test_backward_plan_counts_the_parts_that_the_kernel_counts():
    """The room asked for shared key blocks is two partial sums and a counter for every join, a block of n parts having n - 1 joins, as the
    launch and each workgroup count them (bwd_block_parts) for one limit of the plan; at most 512 MiB; none for packed batches."""
    import random
    from flash_attn import _native as nat

    def tiles(n0, sq, sk, left, right, rows):
        shift, end = sk - sq, min(n0 + 128, sk)
        lo = max(0, n0 - shift - right) if right >= 0 else 0
        hi = min(sq, end - shift + left) if left >= 0 else sq
        return (hi + rows - 1) // rows - lo // rows if hi > lo else 0

    rng, cut, most_bytes = random.Random(1), 0, 0
    for _ in range(3000):
        h_k, g = rng.choice([1, 1, 2, 4, 8]), rng.choice([1, 2, 4, 8])
        b, d = rng.randint(1, 12), rng.choice([64, 80, 128, 160, 192, 256])
        sq, sk = (int(100 * 150 ** rng.random()) for _ in range(2))
        p = _bwd_params(b, h_k * g, h_k, sk, d)
        p.seqlen_q, p.is_causal, p.window_left, p.window_right = sq, rng.randint(0, 1), rng.choice([-1, -1, 256]), rng.choice([-1, 100])
        n = nat.lib.fa_bwd_lend_bytes(ctypes.byref(p), 0, 0)
        if n == 0 or nat.lib.fa_bwd_scratch_bytes(ctypes.byref(p), 0, 0):
            continue
        cut, most_bytes = cut + 1, max(most_bytes, n)
        bucket, rows = (64, 128) if d <= 64 else (128, 64) if d <= 128 else (256, 32)
        joins, rest = divmod(n, 2 * 128 * bucket * 2 * 4 + 4)
        steps = [g * tiles(n0, sq, sk, p.window_left, 0 if p.is_causal else p.window_right, rows) for n0 in range(0, sk, 128)]
        counts = [sum(min(-(-t // limit), 16) - 1 for t in steps if t > limit) * b * h_k
                  for limit in ((max(steps) * k + 15) // 16 for k in (12, 10, 8, 7, 6, 5, 4, 3, 2, 1)) if limit >= 4]
        assert rest == 0 and joins in counts, (b, sq, sk, h_k, g, d)
        p.cu_seqlens_q = p.cu_seqlens_k = 16
        assert nat.lib.fa_bwd_lend_bytes(ctypes.byref(p), b * sq, b * sk) == nat.lib.fa_bwd_scratch_bytes(ctypes.byref(p), b * sq, b * sk)
    assert cut > 300 and 1 << 28 < most_bytes <= 1 << 29


def test_plans_of_17_to_32_rows_fit_the_no_allocation_scratch():
    """fa_plan_splits of decode launches with 17-32 packed rows: their partial results, b x h x seqlen_q x (1 + d rounded up) floats a
    slot, fit the 48 MiB that fa_fwd_kvcache_noalloc has, whatever the batch, as the unsplit launches before them did."""
    from flash_attn import _native as nat
    lib = nat.lib
    p = nat.FaFwdParams()
    for name in ("q", "k", "v", "o", "softmax_lse"):
        setattr(p, name, 4096)
    words = (ctypes.c_int32 * 4096)()
    base = ctypes.addressof(words)
    p.work_counter, p.work_counter_len = (base + 63) // 64 * 64, 4000
    p.cu_seqlens_k = 4096
    p.dtype, p.window_left, p.window_right, p.is_causal = 1, -1, -1, 1
    n = ctypes.c_int32(-1)
    checked = 0
    for b in (1, 3, 16, 48, 200, 1000):
        for sq, h, hk in ((4, 64, 8), (1, 32, 1), (20, 32, 32), (17, 8, 8)):
            for d in (32, 64, 128):
                for sk in (300, 1024, 4096, 5043, 9000, 32768, 200000):
                    p.b, p.seqlen_q, p.h, p.h_k, p.d, p.seqlen_k = b, sq, h, hk, d, sk
                    streams = b * hk
                    if (d > 64 and 4 * streams * sk * d >= 3 << 27) or (256 < streams < 512 and sk <= 2048) or \
                            (streams <= 256 and sk <= (1024 if h > hk else 4096)) or (streams >= 512 and sk <= 512):
                        continue                # the tiled kernel's plan, or near it
                    assert lib.fa_plan_splits(ctypes.byref(p), 2, ctypes.byref(n)) == 0
                    assert 1 <= n.value <= 128
                    if n.value > 1:
                        assert n.value * b * h * sq * 4 * (1 + d) + (128 << 10) <= 48 << 20, (b, sq, h, hk, d, sk, n.value)
                        checked += 1
    assert checked > 60


def test_plans_of_packed_rows_fit_the_no_allocation_scratch():
    """parts of packed rows on the pipelined kernel (a part more than fill the CUs' slots from 64 row blocks on)"""
    from flash_attn import _native as nat
    p = nat.FaFwdParams()
    for name in ("q", "k", "v", "o", "softmax_lse", "cu_seqlens_k"):
        setattr(p, name, 4096)
    p.dtype, p.window_left, p.window_right, p.is_causal = 1, -1, -1, 1
    n, split = ctypes.c_int32(-1), 0
    for b in range(1, 300):
        for sq, h, hk in ((16, 8, 1), (32, 8, 1), (16, 16, 2), (24, 8, 2)):
            for d, sk in ((64, 5000), (64, 20000), (128, 4097), (128, 8192), (128, 30000), (96, 8192)):
                p.b, p.seqlen_q, p.h, p.h_k, p.d, p.seqlen_k = b, sq, h, hk, d, sk
                assert nat.lib.fa_plan_splits(ctypes.byref(p), 2, ctypes.byref(n)) == 0
                if n.value > 1:
                    assert n.value * b * h * sq * 4 * (1 + d) + (128 << 10) <= 48 << 20, (b, sq, h, hk, d, sk, n.value)
                    split += 1
    assert split > 500


@pytest.mark.parametrize("streams,sk,chunk", [(8, 8192, 256), (16, 8192, 256), (17, 8192, 512), (4, 16384, 256), (5, 16384, 512), (8, 8193, 512), (7, 9216, 256), (4, 16385, 512),
                                              (3, 9000, 256), (24, 9000, 512)])
def test_chunks_of_17_to_32_rows_follow_the_load(streams, sk, chunk):
    """256 keys while all chunks run at once (512) and a row has no more of them than the lanes of its merge (32), or while they fill half of the
    resident slots (256) and it has 64; nothing depends on a size of its own"""
    from flash_attn import _native as nat
    p = nat.FaFwdParams()
    for name in ("q", "k", "v", "o", "softmax_lse", "cu_seqlens_k"):
        setattr(p, name, 4096)
    p.dtype, p.window_left, p.window_right, p.is_causal = 1, -1, -1, 1
    p.b, p.seqlen_q, p.h, p.h_k, p.d, p.seqlen_k = streams, 4, 8, 1, 64, sk
    n = ctypes.c_int32(-1)
    assert nat.lib.fa_plan_splits(ctypes.byref(p), 2, ctypes.byref(n)) == 0
    assert n.value == -(-sk // chunk)


@pytest.mark.parametrize("b,sq,h,hk,d,sk,cache,splits", [
    (21, 54, 8, 8, 256, 16212, True, 4), (13, 38, 8, 8, 224, 32771, True, 8), (5, 88, 32, 32, 256, 5777, True, 1), (1, 54, 8, 8, 256, 32768, True, 32),      # one row block
    (2, 488, 16, 16, 224, 2049, True, 1), (3, 508, 8, 8, 256, 8192, True, 1), (3, 508, 8, 8, 256, 8200, True, 2), (7, 301, 8, 8, 256, 18424, True, 1),               # more, over caches
    (2, 488, 16, 16, 224, 2049, False, 2), (7, 301, 8, 8, 256, 18424, False, 1)])                                                                           # known lengths
def test_parts_of_wide_heads(b, sq, h, hk, d, sk, cache, splits):
    """head dims 129-256: a part of a cache is not so long that one full cache among short ones keeps a few CUs busy, and no launch that would fill
    the chip is cut by a capacity that may be mostly empty"""
    from flash_attn import _native as nat
    p = nat.FaFwdParams()
    for name in ("q", "k", "v", "o", "softmax_lse"):
        setattr(p, name, 4096)
    words = (ctypes.c_int32 * 32)()
    p.work_counter, p.work_counter_len = (ctypes.addressof(words) + 63) // 64 * 64, 4
    p.dtype, p.window_left, p.window_right, p.is_causal = 1, -1, -1, 1
    if cache:
        p.cu_seqlens_k = 4096
    p.b, p.seqlen_q, p.h, p.h_k, p.d, p.seqlen_k = b, sq, h, hk, d, sk
    n = ctypes.c_int32(-1)
    assert nat.lib.fa_plan_splits(ctypes.byref(p), 2 if cache else 0, ctypes.byref(n)) == 0
    assert n.value == splits
