"""What surrounds the capture of a hipGraph, on the host."""
import contextlib
import gc

import pytest
import torch

from promptcache_amd.model import llama_hip


class Cycle:
    """Unreachable once dropped, but found by the collector only."""

    def __init__(self, log):
        self.me, self.log = self, log

    def __del__(self):
        self.log.append(1)


@pytest.mark.parametrize("fails", [False, True])
def test_nothing_is_collected_during_a_capture(monkeypatch, fails):
    """Garbage that holds graphs and events must not be released in the middle of a capture: with cycles around and the collector as eager as it
    gets, it runs before and after the block, not in it, and is on again whether the block ends well or not."""
    primed, log, seen = [], [], []

    @contextlib.contextmanager
    def graph(g):
        yield
    monkeypatch.setattr(llama_hip, "prime_graph_capture", primed.append)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", object)
    monkeypatch.setattr(torch.cuda, "graph", graph)
    old = gc.get_threshold()
    gc.set_threshold(5, 1, 1)
    try:
        with contextlib.suppress(ZeroDivisionError):
            with llama_hip.graph_capture("cuda:0") as g:
                Cycle(log)
                junk = [[] for _ in range(1000)]
                seen.append(len(log))
                if fails:
                    1 / 0
        assert gc.isenabled() and seen == [0] and primed == ["cuda:0"] and type(g) is object
        del junk
        junk = [[] for _ in range(1000)]
        assert log == [1]
    finally:
        gc.set_threshold(*old)


def test_a_capture_leaves_a_collector_off_that_was_off(monkeypatch):
    monkeypatch.setattr(llama_hip, "prime_graph_capture", lambda d: None)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", object)
    monkeypatch.setattr(torch.cuda, "graph", lambda g: contextlib.nullcontext())
    gc.disable()
    try:
        with llama_hip.graph_capture("cuda:0"):
            pass
        assert not gc.isenabled()
    finally:
        gc.enable()
