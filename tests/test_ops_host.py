"""ops.py's host side, without a GPU."""

from __future__ import annotations

import torch

from ggmlc_amd import ops


def test_calls_without_a_workspace_share_no_scratch(monkeypatch):
    """two calls in flight (streams, threads) hold buffers of their own, inside a capture too"""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda n, dtype, device: empty(n, dtype=dtype))
    a, b = ops._ws(None), ops._ws(None)
    (pa, na), (pb, nb) = a.get(4096), b.get(4096)
    assert na == nb == 4096 and abs(pa - pb) >= 4096
    assert a.get(0) == (0, 0)
    own = ops.Workspace()
    assert ops._ws(own) is own
