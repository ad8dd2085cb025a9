"""pc_chamfer_grad where many points share a target (summed in LDS up to 5120
targets of 32 points or more each, added point by point otherwise) against fp64."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("n,m", [(1, 1), (31, 1), (32, 1), (1023, 7), (40000, 300), (50001, 1250), (163840, 5120), (163872, 5121),
                                 (300000, 1)])
@pytest.mark.parametrize("both", [False, True])
@pytest.mark.parametrize("squared", [0, 1])
def test_many_points_to_a_target(n, m, both, squared):
    from diffskill_amd import _lib
    L = _lib.load()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    print("case chamfer gradient %d to %d, both=%s squared=%d" % (n, m, both, squared), flush=True)
    g = torch.Generator().manual_seed(n + m)
    x, y = torch.rand((n, 3), generator=g) + 1.0, torch.rand((m, 3), generator=g) - 1.0
    ix, iy = (torch.randint(0, k, (j,), generator=g, dtype=torch.int32) for j, k in ((n, m), (m, n)))
    d2x, d2y = ((p - t[k.long()]).square().sum(1) for p, t, k in ((x, y, ix), (y, x, iy)))
    go = torch.tensor(0.7)
    dev = [t.cuda() for t in (x, y, ix, d2x, iy, d2y, go)]
    gx, gy = torch.empty_like(dev[0]), torch.empty_like(dev[1])
    args = (_p(dev[0]), n, _p(dev[1]), m, _p(dev[2]), _p(dev[3]), _p(dev[4]) if both else None, _p(dev[5]) if both else None, squared, _p(dev[6]))
    rx, ry, size = torch.zeros((n, 3), dtype=torch.float64), torch.zeros((m, 3), dtype=torch.float64), {}
    mx, my = torch.zeros((n, 3), dtype=torch.float64), torch.zeros((m, 3), dtype=torch.float64)   # the terms' magnitudes
    for p, t, k, d2, rp, rt, mp, mt in ((x, y, ix, d2x, rx, ry, mx, my), (y, x, iy, d2y, ry, rx, my, mx))[:2 if both else 1]:
        term = 0.7 / len(p) * (2.0 if squared else 1.0 / d2.double().sqrt()[:, None]) * (p.double() - t[k.long()].double())
        rp += term
        mp += term.abs()
        rt.index_add_(0, k.long(), -term)
        mt.index_add_(0, k.long(), term.abs())
    # a term is off by 8 roundings of its size (weight, root, reciprocal, difference),
    # a sum by one of its magnitude for each of its k additions: at most
    # sqrt(k) of them when their signs are random; 4 standard deviations
    for want in ((True, True), (True, False), (False, True)):
        gx.fill_(7.0), gy.fill_(7.0)
        assert L.pc_chamfer_grad(*args, _p(gx) if want[0] else None, _p(gy) if want[1] else None, s) == 0
        for w, got, ref, mag, k in ((want[0], gx, rx, mx, m / n), (want[1], gy, ry, my, n / m)):
            if w:
                bound = (8 + 4 * (k + 16) ** 0.5) * 2.0 ** -24 * mag.max()
                assert (got.double().cpu() - ref).abs().max() <= bound
