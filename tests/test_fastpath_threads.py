"""The C++ fast path's calls run without the interpreter lock.  Declined calls (host tensors) show it
without a GPU: the lock is given up around the whole call."""

import sys
import threading
import time

import pytest
import torch

from velograd_amd import _lib


def _calls(fp):
    x, inv, q = torch.randn(4, 64), torch.rand(4, 1), torch.randn(2, 8, 4, 64)
    return {
        "forward": lambda: fp.forward(x, x, None, 1e-6, 0.0),
        "forward_quantised": lambda: fp.forward_quantised(x, x, None, 1e-6, -1),
        "backward": lambda: fp.backward(x, x, None, inv, True, None, None),
        "rope": lambda: fp.rope(q, None, 0, 1e4, False),
        "rope_interleaved": lambda: fp.rope_interleaved(x, 1e4, False),
        "norm_rope": lambda: fp.norm_rope(x, None, None, 1e-6, 1e4, 0.0),
        "norm_rope_backward": lambda: fp.norm_rope_backward(x, x, None, inv, 1e4),
    }


@pytest.mark.parametrize("name", ["forward", "forward_quantised", "backward", "rope",
                                  "rope_interleaved", "norm_rope", "norm_rope_backward"])
def test_other_threads_run_during_a_call(name):
    try:
        fp = _lib.fastpath()
    except (_lib.KernelLibraryMissing, OSError):
        fp = None
    if fp is None:
        pytest.skip("the fast path is not built (velograd_amd.build builds it)")
    call = _calls(fp)[name]
    assert call() == []
    turns, stop = [0], [False]

    def other():
        while not stop[0]:
            turns[0] += 1
            time.sleep(0)  # gives the lock back

    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other)
    sys.setswitchinterval(1000.0)  # nobody takes the lock from a thread that does not give it up
    try:
        thread.start()
        time.sleep(0.01)
        end = time.monotonic() + 10.0
        before = turns[0]
        while turns[0] == before and time.monotonic() < end:
            for _ in range(300):
                call()
        gained = turns[0] - before
    finally:
        stop[0] = True
        sys.setswitchinterval(interval)
        thread.join()
    assert gained > 0
