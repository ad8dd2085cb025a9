"""pc_chamfer's loss by one workgroup and by several, against the fp64 mean of the
distances that it returns, and those against pc_nearest_pair's."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("n,m", [(1, 1), (8193, 5), (49151, 1), (49152, 1), (24577, 24600), (65600, 65500), (200003, 90001), (1000001, 10), (4194500, 3)])
@pytest.mark.parametrize("both", [False, True])
@pytest.mark.parametrize("squared", [0, 1])
def test_loss(n, m, both, squared):
    from diffskill_amd import _lib
    L = _lib.load()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    print("case chamfer loss %d x %d both=%s squared=%d" % (n, m, both, squared), flush=True)
    g = torch.Generator().manual_seed(n + m)
    x, y = (torch.rand((k, 3), generator=g).cuda() for k in (n, m))
    out, ref = ([(torch.empty(k, dtype=torch.int32, device="cuda"), torch.empty(k, device="cuda")) if w else (None, None)
                 for k, w in ((n, True), (m, both))] for _ in range(2))
    work = torch.empty(L.pc_nearest_pair_work_bytes(n, m), dtype=torch.uint8, device="cuda")
    loss = torch.empty((), device="cuda")
    assert L.pc_nearest_pair(_p(x), n, _p(y), m, _p(work), *[_p(t) for o in ref for t in o], s) == 0
    assert L.pc_chamfer(_p(x), n, _p(y), m, squared, _p(work), *[_p(t) for o in out for t in o], _p(loss), s) == 0
    want = 0.0
    for o, r in list(zip(out, ref))[:2 if both else 1]:
        assert torch.equal(o[0], r[0]) and torch.equal(o[1], r[1])
        d = r[1].double()
        want += float((d if squared else d.sqrt()).mean())
    # fp32 roots of values of a sign, summed in fp64, each mean and their sum rounded
    assert abs(float(loss) - want) <= 4 * 2.0 ** -24 * want
