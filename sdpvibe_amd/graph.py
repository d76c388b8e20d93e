"""HIP graph capture of a launch sequence (the reference has no counterpart; its launches go one by
one through Triton and CuPy).

Every entry point of the library launches on torch's current stream, allocates nothing inside the
C ABI and never synchronises with the host, so a whole call such as mpf.gemm can be captured once
and replayed: the replay re-runs the same kernels on the same buffers with no host work and no
launch gaps. Inputs are updated in place (copy_ into the captured tensors) between replays.
"""
import contextlib
import gc
import threading

import torch

_lock = threading.Lock()
_captures = 0                  # captures under way, on any thread
_collecting = False            # whether collection was on before the first of them


@contextlib.contextmanager
def _no_collection():
    """Cyclic garbage collection off while any thread captures: it may destroy another object's graph (a solver that
    went out of use), whose destructor synchronises the device, which a capture forbids. The last capture to end
    turns it on again."""
    global _captures, _collecting
    with _lock:
        if _captures == 0:
            _collecting = gc.isenabled()
            gc.disable()
        _captures += 1
    try:
        yield
    finally:
        with _lock:
            _captures -= 1
            if _captures == 0 and _collecting:
                gc.enable()


class Captured:
    """fn(*args) captured into a graph. args: tensors / MPF objects used as static inputs; the
    returned object (tensors inside) is static too and is overwritten by every replay."""

    def __init__(self, fn, *args, warmup=2):
        self.fn, self.args = fn, args
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            for _ in range(warmup):                 # first launches set kernel attributes, build contexts
                fn(*args)
        torch.cuda.current_stream().wait_stream(s)
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with _no_collection(), torch.cuda.graph(self.graph):
            self.out = fn(*args)

    def replay(self):
        self.graph.replay()
        return self.out
