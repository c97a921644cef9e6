"""Streams and unwinding of a gradient graph (no GPU).

A gradient graph needs a stream of its own per box and one to record on, joins
every branch it forked also after a failure, and drops the graph before the
contexts whose buffers it uses.
"""
from __future__ import annotations

import contextlib
from types import SimpleNamespace

import pytest

pytest.importorskip("torch")

from cosmosim import ensemble as E  # noqa: E402


class FakeCuda:
    """Streams from a pool of 32 handed out in turn, as torch's; calls go to `log`."""

    def __init__(self, log):
        self.log = log
        self.next = 5

    def Stream(self, device=None):
        handle = self.next % 32
        self.next += 1
        return SimpleNamespace(cuda_stream=handle, wait_stream=lambda o: self.log.append(("wait", handle, o.cuda_stream)))

    def synchronize(self, device=None):
        pass

    def CUDAGraph(self):
        return "graph"

    def stream(self, st):
        return contextlib.nullcontext()

    @contextlib.contextmanager
    def graph(self, graph, stream=None):
        self.log.append("begin")
        try:
            yield
        finally:
            self.log.append("end")


def faked(monkeypatch, fail_at=None):
    log = []
    monkeypatch.setattr(E.torch, "cuda", FakeCuda(log))

    def box_problem(spec, steps, device, checkpoint_every):
        prob = SimpleNamespace(coord=SimpleNamespace(set_capture_safe=lambda on: None, set_stream=lambda h: None),
                               graph_mode=False, name=spec)
        prob.close = lambda: log.append(("close", spec))
        return prob, None, None

    def sweeps(psi, target, prob):
        if prob.name == fail_at:
            raise RuntimeError("recording failed")
        return "diff", "grad"

    monkeypatch.setattr(E, "box_problem", box_problem)
    monkeypatch.setattr(E.adjoint, "loss_and_gradient", lambda psi, target, prob: None)
    monkeypatch.setattr(E.adjoint, "gradient_sweeps", sweeps)
    return log


def test_gradient_graph_refuses_more_boxes_than_streams(monkeypatch):
    log = faked(monkeypatch)
    with pytest.raises(ValueError, match="streams"):
        E.GradientGraph(list(range(32)), 1)
    assert log == []  # nothing made, nothing recorded
    gg = E.GradientGraph(list(range(31)), 1)
    handles = [gg.main.cuda_stream] + [s.cuda_stream for s in gg.streams]
    assert len(set(handles)) == 32
    assert gg.grad == ["grad"] * 31 and not any(p.graph_mode for p in gg.problems)


def test_failed_recording_joins_its_branches_and_closes(monkeypatch):
    log = faked(monkeypatch, fail_at=2)
    with pytest.raises(RuntimeError, match="recording failed"):
        E.GradientGraph(list(range(4)), 1)
    main, streams = 5, [6, 7, 8]
    forks = [("wait", s, main) for s in streams]
    joins = [("wait", main, s) for s in streams]
    assert log == ["begin"] + forks + joins + ["end"] + [("close", b) for b in range(4)]
