"""Point-cloud losses on the GPU: nearest neighbours by the HIP kernel
``pc_nearest`` and the Chamfer losses built on it, differentiable in both
clouds through ``torch.autograd``.

- ``plb_chamfer_loss``: compute_chamfer_loss_kernel of the reference's loss
  module (plb/engine/losses/loss.py:183-204): the mean Euclidean distance from
  every particle to its nearest target plus the mean from every target to its
  nearest particle; the targets are the grid nodes whose target mass exceeds
  1e-4, at node positions I * dx (loss.py:71-75, ``grid_target_points``).
  The reference's subsampling stride ``min(n // 1000, 1)`` is 1 for every
  cloud of at least 1000 particles, the only case it runs.
- ``sinkhorn_divergence`` / ``plb_emd_loss``: the debiased Sinkhorn
  divergence of ``geomloss.SamplesLoss(loss='sinkhorn', p=1, blur=0.001)``,
  the reference's EMD loss (plb/engine/taichi_env.py:23-26, used at :269-270
  and :303).  geomloss is a third-party dependency absent here (the
  reference pins only its companion pykeops 1.5; geomloss 0.2.4 is that
  generation); its published algorithm is restated: uniform weights, cost
  |x - y|^p / p, epsilon annealing from the clouds' bounding-box diagonal
  down to blur^p by ``scaling``, symmetric (averaged) soft-min updates of the
  x-y problem and of the two debiasing problems, a last extrapolation step,
  S = <a, b_x - a_x> + <b, a_y - b_y>.  Its gradient is the library's: the
  last step differentiated with its input potentials held fixed and only the
  first argument of each cost (C(x, y.detach())), i.e. the transport plans'
  barycentric displacements.  The annealing loop is ``pc_sinkhorn_solve``
  (one launch per epsilon), the gradient ``pc_sinkhorn_grad``.
- ``chamfer_distance``: nearest squared (or Euclidean) distances averaged over
  the source, one-way or both ways -- the quantity of the chamferdist loss the
  reference builds in create_chamfer_loss (plb/engine/taichi_env.py:28-32; that
  package is a third-party dependency absent here, its exact reductions are
  not reproduced).

The adjoint of a nearest distance d_i = |x_i - y_k(i)| (k(i) fixed, as the
reference's branch-wise Taichi adjoint and chamferdist's saved indices both
hold it) is (x_i - y_k) / d_i for x_i and its negative for y_k, scattered to
k(i); squared distances give 2 (x_i - y_k).
"""
import ctypes

import numpy as np
import torch

from . import _lib


def _stream():
    # (torch.cuda.current_stream() takes 16 us in a loss's forward and backward
    # passes, this 3; their library calls take 19 and 10)
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _has_memory(t):
    """Whether a kernel can read t: a gradient batched by vmap has no memory of its own."""
    try:
        t.data_ptr()
        return True
    except RuntimeError:
        return False


def _check(name, rc):
    if rc != 0:
        raise RuntimeError("%s failed: %s" % (name, _lib.load().pc_last_error().decode(errors="replace")))


def _cloud(p, name):
    if not (isinstance(p, torch.Tensor) and p.is_cuda):
        raise TypeError("%s must be a CUDA (HIP) tensor" % name)
    p = p.detach().to(torch.float32).contiguous()
    if p.dim() != 2 or p.shape[1] != 3:
        raise ValueError("%s must be (n, 3), got %s" % (name, tuple(p.shape)))
    return p


def nearest(q, t):
    """For each row of q (n, 3) the nearest row of t (m, 3): (indices (n,)
    int64, squared distances (n,) float32); ties go to the smaller index."""
    q = _cloud(q, "q")
    t = _cloud(t, "t")
    idx, d2 = _nearest_pair(q, t, (True, False))[0]
    return idx.long(), d2


def _nearest_pair(x, y, want):
    """(int32 indices, squared distances) of x in y and of y in x, None for a
    direction not wanted."""
    L = _lib.load()
    n, m = x.shape[0], y.shape[0]
    out = [(torch.empty(k, dtype=torch.int32, device=x.device), torch.empty(k, dtype=torch.float32, device=x.device)) if w else None
           for k, w in zip((n, m), want)]
    work = torch.empty((L.pc_nearest_pair_work_bytes(n, m) + 15) // 16 * 4, dtype=torch.float32, device=x.device)
    ptrs = [p for o in out for p in ((_p(o[0]), _p(o[1])) if o else (None, None))]
    _check("pc_nearest_pair", L.pc_nearest_pair(_p(x), n, _p(y), m, _p(work), *ptrs, _stream()))
    return out


def _distance_grad(x, y, idx, d, squared, g, want_y, none=None):
    """Gradients in x and y of d_i = |x_i - y_idx(i)| (or its square) times g; NaN
    for the points of x in ``none``, which have no nearest y."""
    if none is not None:
        idx = idx.clamp_min(0)
    diff = x - y.index_select(0, idx)
    if none is not None:
        diff = diff.masked_fill(none[:, None], 0.0)
    if squared:
        gx = 2.0 * diff * g[:, None]
    else:
        inv = torch.where(d > 0, 1.0 / d.clamp_min(1e-30), torch.zeros_like(d))
        gx = diff * (g * inv.to(g.dtype))[:, None]
    gy = torch.zeros_like(y).index_add(0, idx, -gx) if want_y else None
    return gx if none is None else gx.masked_fill(none[:, None], float("nan")), gy


class _NearestDistance(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, y, squared):
        idx, d2 = nearest(x, y)
        d = d2 if squared else torch.sqrt(d2)
        ctx.save_for_backward(x, y, idx, d)
        ctx.squared = squared
        return d.to(x.dtype)

    @staticmethod
    def backward(ctx, g):
        x, y, idx, d = ctx.saved_tensors
        gx, gy = _distance_grad(x, y, idx, d, ctx.squared, g, ctx.needs_input_grad[1])
        return gx if ctx.needs_input_grad[0] else None, gy, None


class _PairDistance(torch.autograd.Function):
    """Both directions of _NearestDistance from one search."""

    @staticmethod
    def forward(ctx, x, y, squared):
        (ix, dx), (iy, dy) = _nearest_pair(_cloud(x, "q"), _cloud(y, "t"), (True, True))
        if not squared:
            dx, dy = torch.sqrt(dx), torch.sqrt(dy)
        ctx.save_for_backward(x, y, ix.long(), dx, iy.long(), dy)
        ctx.squared = squared
        return dx.to(x.dtype), dy.to(y.dtype)

    @staticmethod
    def backward(ctx, gdx, gdy):
        x, y, ix, dx, iy, dy = ctx.saved_tensors
        want = ctx.needs_input_grad
        gx, gy = _distance_grad(x, y, ix, dx, ctx.squared, gdx, want[1])
        hy, hx = _distance_grad(y, x, iy, dy, ctx.squared, gdy, want[0])
        return gx + hx if want[0] else None, gy + hy if want[1] else None, None


class _Chamfer(torch.autograd.Function):
    """chamfer_distance of non-empty float32 clouds, loss and gradients in
    kernels of their own."""

    @staticmethod
    def forward(ctx, x, y, bidirectional, squared):
        L = _lib.load()
        xd, yd = _cloud(x, "q"), _cloud(y, "t")
        n, m = xd.shape[0], yd.shape[0]
        # indices, then squared distances (their bits), of x's points; the same of y's.
        # (integers: what a saved-tensor hook may do to floats would be other indices)
        near = torch.empty(2 * (n + m) if bidirectional else 2 * n, dtype=torch.int32, device=xd.device)
        loss = torch.empty((), dtype=torch.float32, device=xd.device)
        work = torch.empty((L.pc_nearest_pair_work_bytes(n, m) + 15) // 16 * 4, dtype=torch.float32, device=xd.device)
        _check("pc_chamfer", L.pc_chamfer(xd.data_ptr(), n, yd.data_ptr(), m, squared, work.data_ptr(),
                                          *_Chamfer.ptrs(near, n, m, bidirectional), loss.data_ptr(), _stream()))
        ctx.save_for_backward(x, y, near)
        ctx.bidirectional, ctx.squared = bidirectional, squared
        return loss

    @staticmethod
    def ptrs(near, n, m, both):
        at = near.data_ptr()
        return (at, at + 4 * n) + ((at + 8 * n, at + 8 * n + 4 * m) if both else (None, None))

    @staticmethod
    def backward(ctx, go):
        x, y, near = ctx.saved_tensors
        want_x, want_y = ctx.needs_input_grad[:2]
        n, m = x.shape[0], y.shape[0]
        if torch.is_grad_enabled() or not _has_memory(go) or torch.are_deterministic_algorithms_enabled():
            # a gradient that is to be differentiated again, a batch of them, or one
            # summed in a fixed order (pc_chamfer_grad's sums over the points that
            # share a target have none): in operations that take those
            def one(p, t, at, w):
                k = len(p)
                idx, d2 = near[at:at + k].long(), near[at + k:at + 2 * k].view(torch.float32)
                return _distance_grad(p, t, idx, d2 if ctx.squared else torch.sqrt(d2), ctx.squared, (go / k).expand(k), w, idx < 0)
            gx, gy = one(x, y, 0, want_y)
            if ctx.bidirectional:
                hy, hx = one(y, x, 2 * n, want_x)
                gx, gy = (gx + hx if want_x else None), (gy + hy if want_y else None)
            return gx if want_x else None, gy, None, None
        # (as the kernel reads them, whatever came back from the hooks)
        xd, yd = _cloud(x, "q"), _cloud(y, "t")
        near = near.to(xd.device, torch.int32).contiguous()
        gx, gy = (torch.empty_like(c) if w else None for c, w in ((xd, want_x), (yd, want_y)))
        _check("pc_chamfer_grad", _lib.load().pc_chamfer_grad(
            xd.data_ptr(), n, yd.data_ptr(), m, *_Chamfer.ptrs(near, n, m, ctx.bidirectional), ctx.squared, go.data_ptr(),
            gx.data_ptr() if want_x else None, gy.data_ptr() if want_y else None, _stream()))
        return gx, gy, None, None


def nearest_distance(x, y, squared=True):
    """Distance from every row of x to its nearest row of y, (n,), differentiable
    in x and y."""
    return _NearestDistance.apply(x, y, squared)


def chamfer_distance(x, y, bidirectional=False, squared=True):
    """mean_i min_j d(x_i, y_j) (+ mean_j min_i d(x_i, y_j) when bidirectional),
    d the squared (default) or Euclidean distance."""
    if all(torch.is_tensor(c) and c.dtype == torch.float32 and c.dim() and len(c) for c in (x, y)):
        return _Chamfer.apply(x, y, bool(bidirectional), bool(squared))
    if bidirectional:
        dx, dy = _PairDistance.apply(x, y, squared)
        return dx.mean() + dy.mean()
    return nearest_distance(x, y, squared).mean()


def grid_target_points(grid, dx, threshold=1e-4):
    """Target points of the reference's Chamfer loss: the positions I * dx of
    the nodes with mass above the threshold, in numpy's C order (loss.py:71-72)."""
    g = grid.detach().cpu().numpy() if isinstance(grid, torch.Tensor) else np.asarray(grid)
    return (np.array(np.where(g > threshold)).transpose() * dx).astype(np.float64)


def plb_chamfer_loss(x, target_points):
    """compute_chamfer_loss_kernel (loss.py:183-204): Euclidean Chamfer both
    ways, each direction averaged over its own points."""
    t = torch.as_tensor(target_points, dtype=x.dtype, device=x.device)
    return chamfer_distance(x, t, bidirectional=True, squared=False)


def epsilon_schedule(x, y, p, blur, scaling):
    """geomloss's annealing: the bounding-box diagonal d of both clouds, then
    exp(arange(p log d, p log blur, p log scaling)), then blur^p.  A diagonal
    below blur (all points within blur of each other) is taken as blur, so the
    schedule is just blur^p twice instead of starting at eps = 0."""
    if (x.is_cuda and x.device == y.device and x.dtype == y.dtype == torch.float32 and x.is_contiguous() and y.is_contiguous()
            and x.dim() == y.dim() == 2 and x.shape[1] == y.shape[1] == 3):   # (rows of three are what the kernel reads)
        ext = torch.empty(3, dtype=torch.float32, device=x.device)
        _check("pc_extent", _lib.load().pc_extent(_p(x), x.shape[0], _p(y), y.shape[0], _p(ext), _stream()))
    else:
        pts = torch.cat([x, y])
        ext = pts.max(0).values - pts.min(0).values
    d = max(float(ext.norm()), blur)
    return [d ** p] + [float(np.exp(e)) for e in np.arange(p * np.log(d), p * np.log(blur), p * np.log(scaling))] + [blur ** p]


def _sinkhorn_work(x, y):
    """Scratch of one call on the current stream.  The caller holds it until the
    call has returned: its launches are issued without the GIL, and a tensor let
    go before them could be handed to another thread's launches in between."""
    nb = _lib.load().pc_sinkhorn_step_work_bytes(x.shape[0], y.shape[0])
    return torch.empty((nb + 15) // 16 * 4, dtype=torch.float32, device=x.device)


class _SinkhornDivergence(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, y, p, blur, scaling):
        xd, yd = _cloud(x, "x"), _cloud(y, "y")
        N, M = xd.shape[0], yd.shape[0]
        if N == 0 or M == 0:
            raise ValueError("sinkhorn_divergence needs two non-empty clouds")
        eps_s = epsilon_schedule(xd, yd, p, blur, scaling)
        pot = torch.empty(4 * (N + M), dtype=torch.float32, device=xd.device)
        loss = torch.empty((), dtype=torch.float32, device=xd.device)
        eps = (ctypes.c_float * len(eps_s))(*eps_s)
        work = _sinkhorn_work(xd, yd)
        _check("pc_sinkhorn_solve", _lib.load().pc_sinkhorn_solve(_p(xd), N, _p(yd), M, eps, len(eps_s), p, _p(pot), _p(loss),
                                                                  _p(work), _stream()))
        ctx.clouds, ctx.pot, ctx.eps, ctx.p = (xd, yd), pot, eps_s[-1], p
        return loss.to(x.dtype)

    @staticmethod
    def backward(ctx, go):
        xd, yd = ctx.clouds
        want = ctx.needs_input_grad[:2]
        gx, gy = (torch.empty_like(c) if w else None for c, w in zip((xd, yd), want))
        # a gradient that is to be differentiated again (in go), or a batch of them,
        # takes the factor outside the kernel
        inside = go.to(torch.float32) if not go.requires_grad and _has_memory(go) else None
        work = _sinkhorn_work(xd, yd)
        _check("pc_sinkhorn_grad", _lib.load().pc_sinkhorn_grad(
            _p(xd), xd.shape[0], _p(yd), yd.shape[0], _p(ctx.pot), ctx.eps, ctx.p, None if inside is None else _p(inside),
            *(None if g is None else _p(g) for g in (gx, gy)), _p(work), _stream()))
        if inside is None:
            gx, gy = (None if g is None else g * go for g in (gx, gy))
        return (*(None if g is None else g.to(go.dtype) for g in (gx, gy)), None, None, None)


def sinkhorn_divergence(x, y, p=1, blur=0.001, scaling=0.5):
    """Debiased Sinkhorn divergence S(x, y) of two uniformly weighted clouds
    ((n, 3) and (m, 3) CUDA tensors), differentiable in both (p = 1 or 2)."""
    if p not in (1, 2):
        raise ValueError("p must be 1 or 2")
    return _SinkhornDivergence.apply(x, y, int(p), float(blur), float(scaling))


def plb_emd_loss(x, target):
    """create_emd_loss()(x, target) of the reference (taichi_env.py:23-26):
    SamplesLoss(loss='sinkhorn', p=1, blur=0.001)."""
    return sinkhorn_divergence(x, target, p=1, blur=0.001, scaling=0.5)
