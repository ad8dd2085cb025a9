"""Which search pc_nearest_pair takes, over equal and unequal clouds, on the side
that measured the faster; the results are the same bit for bit either way."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


# queries, targets, both ways, whether every pair is looked at
CASES = [(300, 300, False, True), (300, 1000, False, False), (40000, 300, False, True), (40000, 2000, False, False),
         (1000, 20000, False, False), (100, 200000, False, True), (100, 1000000, False, True), (10000, 100000, False, False),
         (1000000, 1000, False, True), (200000, 10000, False, False), (15312, 15508, False, False), (300, 100, True, False),
         (100, 1000000, True, True), (1000000, 100, True, True), (30000, 25001, True, False), (200000, 5000, True, False)]


@pytest.mark.parametrize("n,m,both,every", CASES)
def test_route(n, m, both, every):
    from diffskill_amd import _lib
    L = _lib.load()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    print("case nearest route %d x %d both=%s" % (n, m, both), flush=True)
    g = torch.Generator().manual_seed(n + 3 * m)
    x, y = (torch.rand((k, 3), generator=g).cuda() for k in (n, m))
    got, ref = ([(torch.empty(k, dtype=torch.int32, device="cuda"), torch.empty(k, device="cuda")) for k in (n, m)] for _ in range(2))
    work = torch.full((L.pc_nearest_pair_work_bytes(n, m),), 0xcc, dtype=torch.uint8, device="cuda")
    outs = [_p(t) if both or not k else None for k, o in enumerate(got) for t in o]
    assert L.pc_nearest_pair(_p(x), n, _p(y), m, _p(work), *outs, s) == 0
    # every pair: a word for each query alone
    assert bool((work[8 * (max(n, m) if both else n):] == 0xcc).all()) == every
    for k, (q, t) in enumerate(((x, y), (y, x)) if both else ((x, y),)):
        w = torch.empty(len(q), dtype=torch.int64, device="cuda")
        assert L.pc_nearest(_p(q), len(q), _p(t), len(t), _p(w), _p(ref[k][0]), _p(ref[k][1]), s) == 0
        assert torch.equal(got[k][0], ref[k][0]) and torch.equal(got[k][1], ref[k][1])
