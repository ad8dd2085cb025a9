"""The host side of the point-cloud losses, with the library's entry points
replaced by stand-ins that look at what they are given."""
import ctypes
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


def _zeros(p, nbytes):
    if p is not None:
        ctypes.memset(p, 0, nbytes)
    return 0


def _search(x, n, y, m, squared, work, ix, dx, iy, dy, loss, stream):
    """Every point's nearest target is target 0, at distance 0."""
    return _zeros(ix, 4 * n) or _zeros(dx, 4 * n) or _zeros(iy, 4 * m) or _zeros(dy, 4 * m)


def _chamfer_library():
    return Library(pc_nearest_pair_work_bytes=64, pc_chamfer=_search)


@pytest.mark.parametrize("both", [False, True])
def test_chamfer_batch_of_gradients(host, both):
    """Several gradients of one loss at once (vmap over the backward)."""
    lib = host(_chamfer_library())
    x, y = torch.rand(5, 3, requires_grad=True), torch.rand(4, 3, requires_grad=True)
    loss = pc.chamfer_distance(x, y, bidirectional=both)
    gx, gy = torch.autograd.grad(loss, (x, y), torch.tensor([1.0, -2.0]), is_grads_batched=True)
    ref = 2 * (x - y[0]) / 5
    add = torch.zeros(4, 3).index_add(0, torch.zeros(5, dtype=torch.long), -ref)
    if both:
        hy = 2 * (y - x[0]) / 4
        ref, add = ref.index_add(0, torch.zeros(4, dtype=torch.long), -hy), add + hy
    for k, f in enumerate((1.0, -2.0)):
        assert torch.allclose(gx[k], f * ref) and torch.allclose(gy[k], f * add)


def test_sinkhorn_batch_of_gradients(host):
    def grad(x, n, y, m, pot, eps, p, go, gx, gy, work, stream):
        f = 1.0 if go is None else ctypes.cast(go, ctypes.POINTER(ctypes.c_float))[0]
        for g, k in ((gx, n), (gy, m)):
            if g is not None:
                ctypes.memmove(g, (ctypes.c_float * (3 * k))(*([f] * (3 * k))), 12 * k)
        return 0

    host(Library(pc_sinkhorn_step_work_bytes=4096, pc_sinkhorn_grad=grad))
    x, y = torch.rand(5, 3, requires_grad=True), torch.rand(4, 3, requires_grad=True)
    loss = pc.sinkhorn_divergence(x, y)
    one = torch.autograd.grad(loss, (x, y), torch.tensor(0.5), retain_graph=True)
    got = torch.autograd.grad(loss, (x, y), torch.tensor([1.0, -2.0]), is_grads_batched=True)
    for a, b in zip(one, got):
        assert (a == 0.5).all() and (b[0] == 1.0).all() and (b[1] == -2.0).all()


@pytest.mark.parametrize("fixed", [False, True])
def test_chamfer_gradient_of_deterministic_algorithms(host, fixed):
    """The gradient kernel's sums have no fixed order: not where one is asked for."""
    lib = host(_chamfer_library())
    x, y = torch.rand(5, 3, requires_grad=True), torch.rand(4, 3, requires_grad=True)
    torch.use_deterministic_algorithms(fixed)
    try:
        gx, gy = torch.autograd.grad(pc.chamfer_distance(x, y), (x, y))
    finally:
        torch.use_deterministic_algorithms(False)
    assert ("pc_chamfer_grad" in lib.seen) != fixed
    if fixed:
        assert torch.allclose(gx, 2 * (x - y[0]) / 5) and torch.allclose(gy[0], -gx.sum(0)) and (gy[1:] == 0).all()


@pytest.mark.parametrize("squared", [False, True])
def test_chamfer_gradient_without_a_nearest_target(host, squared):
    """A point at infinity: NaN for itself, nothing for the targets, in torch's
    operations as in the kernel (where an index of -1 stopped the program)."""
    def search(x, n, y, m, squared, work, ix, dx, iy, dy, loss, stream):
        idx = (ctypes.c_int * n)(*[-1 if k == 2 else 0 for k in range(n)])
        d2 = (ctypes.c_float * n)(*[float("inf") if k == 2 else 4.0 for k in range(n)])
        ctypes.memmove(ix, idx, 4 * n)
        ctypes.memmove(dx, d2, 4 * n)
        return 0

    host(Library(pc_nearest_pair_work_bytes=64, pc_chamfer=search))
    x, y = torch.rand(5, 3), torch.rand(4, 3, requires_grad=True)
    x[2] = float("inf")
    x.requires_grad_(True)
    gx, gy = torch.autograd.grad(pc.chamfer_distance(x, y, squared=squared), (x, y), create_graph=True)
    keep = [0, 1, 3, 4]
    ref = ((2.0 if squared else 0.5) * (x - y[0]) / 5)[keep]
    assert torch.isnan(gx[2]).all() and torch.allclose(gx[keep], ref)
    assert torch.allclose(gy[0], -ref.sum(0)) and (gy[1:] == 0).all()


def test_chamfer_saved_tensor_hooks(host):
    """Hooks that keep floats at half precision: the gradient kernel still gets
    float32 clouds and the search's own indices."""
    seen = {}

    def search(x, n, y, m, squared, work, ix, dx, iy, dy, loss, stream):
        ctypes.memmove(ix, (ctypes.c_int * n)(*range(100000, 100000 + n)), 4 * n)
        return _zeros(dx, 4 * n)

    def grad(x, n, y, m, ix, dx, iy, dy, squared, go, gx, gy, stream):
        seen["idx"] = list((ctypes.c_int * n).from_address(ix))
        seen["x"] = list((ctypes.c_float * (3 * n)).from_address(x))
        return _zeros(gx, 12 * n) or _zeros(gy, 12 * m)

    host(Library(pc_nearest_pair_work_bytes=64, pc_chamfer=search, pc_chamfer_grad=grad))
    x, y = torch.rand(5, 3, requires_grad=True), torch.rand(4, 3, requires_grad=True)
    half = lambda t: t.half() if t.is_floating_point() else t   # noqa: E731
    with torch.autograd.graph.saved_tensors_hooks(half, lambda t: t):
        loss = pc.chamfer_distance(x, y)
    loss.backward()
    assert seen["idx"] == list(range(100000, 100005))
    assert seen["x"] == x.detach().half().float().flatten().tolist()
