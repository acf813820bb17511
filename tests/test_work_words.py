"""Which words the Python layer lends a launch for its work list: the stream's own outside capture, the call's own inside."""
import ctypes

import pytest
import torch

from flash_attn import _native as nat


def test_captured_launches_with_a_list_share_no_words(monkeypatch):
    """Graphs captured on one stream may replay side by side: a list that two of them wrote and read would be one of them's."""
    dev = torch.device("cpu", 0)
    capturing = [False]
    monkeypatch.setattr(nat, "_stream", lambda device: 77)
    monkeypatch.setattr(nat, "_COUNTERS", {})
    monkeypatch.setattr(nat, "_RETIRED", [])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    span = lambda t: (t.data_ptr(), t.data_ptr() + 4 * t.numel())
    apart = lambda a, b: span(a)[1] <= span(b)[0] or span(b)[1] <= span(a)[0]
    eager = nat._counters(dev, 100)
    assert not eager.any() and nat._counters(dev, 100) is eager and nat._counters(dev, nat.WORK_COUNTER_WORDS) is eager
    capturing[0] = True
    a, b = nat._counters(dev, 100), nat._counters(dev, 100)
    assert a.numel() >= 100 and apart(a, b) and apart(a, eager) and apart(b, eager)
    assert nat._counters(dev, 200).numel() >= 200 and not nat._RETIRED
    assert nat._counters(dev, nat.WORK_COUNTER_WORDS) is eager          # tickets: tagged per call, the stream's words
    assert list(nat._COUNTERS.values()) == [eager]


@pytest.mark.parametrize("b,sq,h,hk,d,listed", [(22, 24, 8, 1, 128, False), (4, 2048, 1, 1, 64, False), (2, 90, 64, 64, 64, False), (16, 64, 16, 16, 128, False),
                                                (16, 65, 16, 16, 128, True), (22, 130, 8, 1, 64, True), (16, 64, 16, 16, 192, True)])
def test_packed_launches_of_few_rows_ask_for_no_list(b, sq, h, hk, d, listed):
    """Up to 256 blocks of 32 or 64 rows (waves that split the keys, head dims up to 128) run all at once: the launch that would order them
    takes longer than they do.  4 sequences of one head do not spread over the XCDs."""
    p = nat.FaFwdParams()
    for name in ("q", "k", "v", "o", "softmax_lse", "cu_seqlens_q", "cu_seqlens_k"):
        setattr(p, name, 4096)
    p.b, p.seqlen_q, p.seqlen_k, p.h, p.h_k, p.d, p.dtype, p.is_seqlens_k_cumulative = b, sq, sq, h, hk, d, 1, 1
    p.window_left = p.window_right = -1
    assert (nat.lib.fa_work_list_words(ctypes.byref(p)) > nat.WORK_COUNTER_WORDS) == listed
