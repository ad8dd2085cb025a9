"""Device actions set on one stream and read back on another."""
import numpy as np
import pytest
import torch

from scenes import capsule_scene
from test_gpu_parity import build

pytestmark = pytest.mark.gpu


def test_table_waits_for_the_stream_that_fills_it():
    print("case action table, two streams", flush=True)
    sim, P = build(*capsule_scene(n=100))
    a = torch.tensor([0.25, -2.0, 0.5], device="cuda")
    P.set_action(0, 5, torch.zeros(3, device="cuda"))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(200_000_000)   # (a fraction of a second)
        P.set_action(1, 5, a)
    assert not side.query()
    got = np.array(P._table(1))
    torch.cuda.synchronize()
    assert np.array_equal(got[0, :3], np.float32([0.25, -1.0, 0.5]))
    assert np.array_equal(got, P._table(1))
