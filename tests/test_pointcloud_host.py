"""The host side of the point-cloud losses, with the library's entry points
replaced by stand-ins that look at what they are given."""
import weakref

import pytest
import torch

from diffskill_amd import pointcloud as pc


class Library:
    """Entry points that succeed without touching memory; seen[name] are their calls."""

    def __init__(self, **calls):
        self.calls, self.seen = calls, {}

    def __getattr__(self, name):
        def call(*args):
            self.seen.setdefault(name, []).append(args)
            f = self.calls.get(name)
            return f(*args) if callable(f) else (0 if f is None else f)
        return call


@pytest.fixture
def host(monkeypatch):
    """Clouds on the CPU pass for the device's."""
    def use(lib):
        monkeypatch.setattr(pc._lib, "load", lambda: lib)
        return lib
    monkeypatch.setattr(pc, "_cloud", lambda p, name: p.detach().to(torch.float32).contiguous())
    monkeypatch.setattr(pc, "_stream", lambda: None)
    return use


def test_sinkhorn_scratch_lives_through_the_call(host, monkeypatch):
    """The launches are issued inside the call, without the GIL: scratch that is
    back in the allocator by then could be another thread's."""
    refs, alive = [], []
    make = pc._sinkhorn_work

    def tracked(x, y):
        t = make(x, y)
        refs.append(weakref.ref(t))
        return t

    def look(*args):
        alive.append(refs[-1]() is not None)
        return 0

    monkeypatch.setattr(pc, "_sinkhorn_work", tracked)
    host(Library(pc_sinkhorn_step_work_bytes=4096, pc_sinkhorn_solve=look, pc_sinkhorn_grad=look))
    x, y = torch.rand(5, 3, requires_grad=True), torch.rand(4, 3)
    pc.sinkhorn_divergence(x, y).backward()
    assert alive == [True, True]
