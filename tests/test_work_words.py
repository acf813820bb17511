"""Which words the Python layer lends a launch for its work list: the stream's own outside capture, the call's own inside."""
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
