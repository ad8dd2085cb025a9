"""epsilon_schedule of device clouds of any width, layout and type against the
same clouds on the CPU."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(1, 1), (7, 300), (2000, 33)])
@pytest.mark.parametrize("width", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("kind", ["float", "double", "strided"])
def test_schedule(n, m, width, kind):
    from diffskill_amd.pointcloud import epsilon_schedule
    print("case schedule %d x %d, %d wide, %s" % (n, m, width, kind), flush=True)
    g = torch.Generator().manual_seed(n + width)
    x, y = (torch.rand((k, width), generator=g) * torch.arange(1, width + 1) for k in (n, m))
    if kind == "double":
        x, y = x.double(), y.double()
    xd, yd = x.cuda(), y.cuda()
    if kind == "strided":
        xd, yd = xd.t().contiguous().t(), yd.t().contiguous().t()
    ref, got = epsilon_schedule(x, y, 2, 0.01, 0.5), epsilon_schedule(xd, yd, 2, 0.01, 0.5)
    # the diagonal's few fp32 roundings
    assert len(got) == len(ref) and all(abs(a - b) <= 8 * 2.0 ** -24 * b for a, b in zip(got, ref))
