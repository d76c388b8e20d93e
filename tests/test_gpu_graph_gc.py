"""Cyclic garbage collection stays off while a graph is captured (a collected graph's destructor
synchronises the device, which ends the process in the middle of a capture) and comes back afterwards."""
import gc

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("enabled", [True, False])
def test_no_collection_while_capturing(enabled):
    from sdpvibe_amd.graph import Captured
    seen = []

    def fn(x):
        seen.append((torch.cuda.is_current_stream_capturing(), gc.isenabled()))
        return x + 1

    was = gc.isenabled()
    (gc.enable if enabled else gc.disable)()
    try:
        x = torch.zeros(4, device="cuda")
        c = Captured(fn, x)
        assert gc.isenabled() == enabled
        x += 2
        assert torch.equal(c.replay(), x + 1)
    finally:
        (gc.enable if was else gc.disable)()
    assert seen == [(False, enabled)] * 2 + [(True, False)]
