"""The shared decode loop's host side, with the device's part replaced."""
import contextlib
import gc

import pytest
import torch

from moondream_amd import engine


class Engine(engine.DeviceEngine):
    def __init__(self):
        self._device, self._graphs, self.use_graphs = torch.device("cpu"), {}, True

    def _h2d(self, t):
        return t


@pytest.mark.parametrize("fails", [False, True], ids=["captured", "raises"])
def test_nothing_is_collected_inside_a_capture(monkeypatch, fails):
    """An unused model with captured graphs is cyclic garbage; collected during another model's capture it ends the process."""
    capturing, collected = [], []

    @contextlib.contextmanager
    def graph(g):
        capturing.append(1)
        try:
            yield
        finally:
            capturing.clear()

    def make_step(pos):
        def step(tok_in, tok_out, u):
            for _ in range(50):
                cycle = []
                cycle.append(cycle)
            if capturing and fails:
                raise RuntimeError("launch")
            tok_out.copy_(tok_in + 1)

        return step

    class Stream:
        cuda_stream = 0

    monkeypatch.setattr(torch.cuda, "graph", graph)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: None)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda d=None: None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: Stream)
    watch = lambda phase, info: capturing and collected.append(phase)  # noqa: E731
    before = gc.get_threshold()
    gc.callbacks.append(watch)
    gc.set_threshold(1, 1, 1)
    try:
        e = Engine()
        with pytest.raises(RuntimeError) if fails else contextlib.nullcontext():
            hist = e._lockstep_loop(torch.tensor([5, 8], dtype=torch.int32), [0, 0], 4, make_step, ("k",), None)
            assert hist.tolist() == [[5 + i, 8 + i] for i in range(5)]
        assert gc.isenabled()
    finally:
        gc.set_threshold(*before)
        gc.callbacks.remove(watch)
    assert not collected


def test_a_model_with_graphs_is_no_cycle(monkeypatch):
    """A model is freed with its last reference, its captured graphs with it."""
    import weakref

    class Stream:
        cuda_stream = 0

    monkeypatch.setattr(torch.cuda, "graph", lambda g: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: None)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda d=None: None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: Stream)

    class Model(Engine):
        def generate(self):
            return self._lockstep_loop(torch.tensor([5], dtype=torch.int32), [0], 4,
                                       lambda pos: lambda tok_in, tok_out, u: tok_out.copy_(tok_in + self.one), ("k",), None)

        one = 1

    e = Model()
    assert e.generate().flatten().tolist() == [5, 6, 7, 8, 9] and e._graphs
    gone = weakref.ref(e)
    with engine.no_collection():
        del e
        assert gone() is None


def test_layers_of_a_cache_as_one_tensor():
    """What ``encode_image`` hands out is taken as one tensor, in every other form layer by layer."""
    import torch

    from moondream_amd.moondream import _layers_as_one

    whole = torch.randn(4, 1, 3, 5, 8)
    views = list(whole.unbind(0))
    assert torch.equal(_layers_as_one(views, 4), whole)
    part = [t[:, :, 1:4] for t in views]  # rows left out, strides kept
    assert torch.equal(_layers_as_one(part, 4), whole[:, :, :, 1:4])
    assert torch.equal(_layers_as_one(list(whole.transpose(0, 2).contiguous().transpose(0, 2).unbind(0)), 4), whole)
    for other in ([t.clone() for t in views], views[::-1], views[:3], [views[0]] * 4, views[:3] + [views[3][:, :, :4]], views[:3] + [views[3].clone()],
                  views[:3] + [views[3].double()], [views[k] for k in (0, 2, 1, 3)], [t[0] for t in views], [t.transpose(1, 2) if i == 2 else t for i, t in enumerate(views)]):
        assert _layers_as_one(other, 4) is None
