"""Graph captures on several threads (torch's capture replaced by a stand-in, no GPU): cyclic collection stays off until
the last of the overlapping captures has ended, and is then as it was before the first."""
import contextlib
import gc
import threading
import types

import pytest
import torch

from sdpvibe_amd import graph


@pytest.fixture
def fake_capture(monkeypatch):
    on = contextlib.nullcontext()
    monkeypatch.setattr(torch.cuda, "Stream", lambda: types.SimpleNamespace(wait_stream=lambda s: None))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(wait_stream=lambda s: None))
    monkeypatch.setattr(torch.cuda, "stream", lambda s: on)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", object)
    monkeypatch.setattr(torch.cuda, "graph", lambda g: on)


@pytest.mark.parametrize("collecting", [True, False])
def test_overlapping_captures(fake_capture, collecting):
    first_in, second_in, first_done = threading.Event(), threading.Event(), threading.Event()
    seen = {}

    def first():
        first_in.set()
        assert second_in.wait(20)

    def second():
        assert first_in.wait(20)
        second_in.set()
        assert first_done.wait(20)
        seen["second"] = gc.isenabled()

    def run_first():
        graph.Captured(first, warmup=0)
        first_done.set()

    was = gc.isenabled()
    (gc.enable if collecting else gc.disable)()
    try:
        threads = [threading.Thread(target=run_first), threading.Thread(target=lambda: graph.Captured(second, warmup=0))]
        for t in threads:
            t.start()
        for t in threads:
            t.join(30)
        assert seen == {"second": False}
        assert gc.isenabled() is collecting
    finally:
        (gc.enable if was else gc.disable)()


def test_a_failing_capture_restores_collection(fake_capture):
    def fail():
        assert not gc.isenabled()
        raise RuntimeError("x")
    was = gc.isenabled()
    gc.enable()
    try:
        with pytest.raises(RuntimeError):
            graph.Captured(fail, warmup=0)
        assert gc.isenabled()
    finally:
        if not was:
            gc.disable()
