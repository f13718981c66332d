"""The host's wait for the hand-off's counts, with a thread in the place of the kernel that writes them to host memory."""

import os
import signal
import threading
import time
from types import SimpleNamespace

import pytest
import torch

from mi355_vit import _lib, handoff


@pytest.mark.parametrize("where", ["in front of the wait", "during the wait"])
def test_an_interrupted_wait_ends_only_when_the_counts_are_there(monkeypatch, where):
    """An exception out of a signal handler, as Ctrl-C raises it, while the kernel is still to run: the counts' memory must not go back to
    an allocator that does not know of the kernel."""
    counts, lib, calls = torch.full((2,), -1, dtype=torch.int64), _lib.load(), []

    def interrupt(*args):
        raise KeyboardInterrupt

    def wait(values, n, stream):
        calls.append(stream)
        if where == "in front of the wait" and len(calls) == 1:
            interrupt()
        return lib.mvit_wait_host_values(values, n, 10_000_000)  # like the wait on a stream, one call

    def kernel():
        time.sleep(0.05)
        if where == "during the wait":
            os.kill(os.getpid(), signal.SIGUSR1)
        time.sleep(0.2)
        counts.copy_(torch.tensor([4, 0]))

    monkeypatch.setattr(_lib, "load", lambda: SimpleNamespace(mvit_await_host_values=wait))
    before, thread = signal.signal(signal.SIGUSR1, interrupt), threading.Thread(target=kernel)
    try:
        arrival = handoff._Arrival(counts, 7)
        with pytest.raises(KeyboardInterrupt):
            thread.start()
            arrival.synchronize()
        there = counts.tolist()
    finally:
        thread.join()
        signal.signal(signal.SIGUSR1, before)
    assert there == [4, 0] and set(calls) == {7}


def test_the_wait_ends_when_the_stream_cannot_write_the_values():
    """Without a GPU every stream has failed: an error, and values that are there are taken all the same."""
    if torch.cuda.is_available():
        pytest.skip("streams work here")
    values = torch.full((2,), -1, dtype=torch.int64)
    with pytest.raises(RuntimeError, match="await_host_values"):
        handoff._Arrival(values, 0).synchronize()
    values.zero_()
    handoff._Arrival(values, 0).synchronize()
