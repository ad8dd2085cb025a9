"""The sorted nearest search with points far outside the others, at infinity and
NaN: results equal to the search over every pair bit for bit, and the other
points still spread over the sort's cells."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _cloud(n, kind, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.rand((n, 3), generator=g)
    if kind == "ordered":          # along an axis, as a lattice or a scan comes
        x = x[x[:, 0].argsort()]
    elif kind == "lattice":        # rows of 64 points along one axis
        k = torch.arange(n)
        x = torch.stack([k // 64 // 16, k // 64 % 16, k % 64], 1) / 64.0 + 0.001 * x
    elif kind == "one":
        x[n // 2] = 500.0 * (1 if seed % 2 else -1)
    elif kind == "few":
        x[torch.randperm(n, generator=g)[:5]] = torch.randn((5, 3), generator=g)[:len(x)] * 1e4
    elif kind == "huge":
        x[n // 3] = 1e30
    elif kind == "infinite":
        x[n // 2], x[n // 3, 1], x[0, 2] = float("inf"), float("-inf"), float("nan")
    elif kind == "special":
        x[:] = float("nan")
        x[::2, 1] = float("inf")
    return x.cuda()


@pytest.mark.parametrize("n,m", [(6, 9), (40, 31), (700, 600), (3000, 2999), (20000, 5001)])
@pytest.mark.parametrize("kind", ["ordered", "lattice", "one", "few", "huge", "infinite", "special"])
def test_outliers(n, m, kind):
    from diffskill_amd import _lib
    L = _lib.load()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    print("case nearest outliers %d x %d %s" % (n, m, kind), flush=True)
    x, y = _cloud(n, kind, 2 * n + 1), _cloud(m, kind, 2 * m)
    out = [[(torch.empty(k, dtype=torch.int32, device="cuda"), torch.empty(k, device="cuda")) for k in (n, m)] for _ in range(2)]
    for (q, t), o in zip(((x, y), (y, x)), out[0]):
        w = torch.empty(len(q), dtype=torch.int64, device="cuda")
        assert L.pc_nearest(_p(q), len(q), _p(t), len(t), _p(w), _p(o[0]), _p(o[1]), s) == 0
    work = torch.zeros(L.pc_nearest_pair_work_bytes(n, m), dtype=torch.uint8, device="cuda")
    assert L.pc_nearest_pair(_p(x), n, _p(y), m, _p(work), *[_p(t) for o in out[1] for t in o], s) == 0
    for r, o in zip(*out):
        assert torch.equal(o[0], r[0]) and torch.equal(o[1], r[1])
    if kind != "special" and n >= 3000:
        # the workspace's cells of x, behind its sorted points and boxes: 16^3 of them,
        # a few of which take 3000 or more points' outliers
        at = (n + 31) // 32 * (32 * 16 + 32)
        cells = work[at:at + 8 * n].view(torch.int32)[::2]
        rows = -(-n // (64 * 16)) if kind == "lattice" else 16
        assert 1500 * min(16, rows) // 16 < len(cells.unique()) <= 4096
