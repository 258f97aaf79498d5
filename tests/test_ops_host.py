"""Host logic of the operator entry points, on the CPU: which calls share a
scratch buffer."""
import threading

import torch

from moe_stream_amd import ops

CPU = torch.device("cpu")


def test_scratch_is_shared_only_in_one_streams_order():
    """One buffer per purpose, stream and thread: calls on one stream from one
    thread reuse it (it grows), calls that can run beside each other never do."""
    ws = ops.Workspace()
    a = ws.get("ffn", 1000, CPU, 1)
    assert ws.get("ffn", 500, CPU, 1) is a
    b = ws.get("ffn", 1000, CPU, 2)
    assert b is not a and b.data_ptr() != a.data_ptr()
    assert ws.get("route", 1000, CPU, 1, zero=True) is not a
    other = []
    t = threading.Thread(target=lambda: other.append(ws.get("ffn", 1000, CPU, 1)))
    t.start()
    t.join()
    assert other[0] is not a and other[0].data_ptr() != a.data_ptr()
    grown = ws.get("ffn", 2000, CPU, 1)
    assert grown is not a and grown.numel() >= 2000
    assert ws.get("ffn", 1000, CPU, 1) is grown
    assert ws.get("ffn", 1000, CPU, 2) is b


def test_scratch_is_bounded_and_zeroed_when_asked():
    ws = ops.Workspace()
    keep = ws.get("ffn", 64, CPU, 0)
    for handle in range(1, 3 * ops.Workspace.KEEP):
        assert not ws.get("route", 4096, CPU, handle, zero=True).any()
        assert ws.get("ffn", 64, CPU, 0) is keep   # in use: stays
    assert len(ws._bufs) <= ops.Workspace.KEEP
