"""mpm_update_prims after a refused call: the device gets the constants of the
call that succeeds, though the refused one had the same."""
import numpy as np
import pytest

from scenes import capsule_scene
from test_gpu_parity import build, flat

pytestmark = pytest.mark.gpu


def _scene(friction):
    sim_cfg, prims, st = capsule_scene(n=800)
    prims = [dict(prims[0], friction=friction), dict(prims[0], init_pos=(0.45, 0.16, 0.5))]
    return build(sim_cfg, prims, st)


def _frame(sim, P):
    P.set_action(0, 5, np.array([0.3, -1.0, 0.2] * 2))
    sim.engine.substep_fwd(0, 5)
    return flat(sim.get_state(5))


def test_update_after_a_refused_one():
    print("case update prims", flush=True)
    ref, other = _frame(*_scene(0.1)), _frame(*_scene(5.0))
    assert not np.array_equal(ref, other)   # (the friction shows)
    sim, P = _scene(5.0)
    P[0].friction = 0.1
    descs = sim._prim_descs()
    assert np.float32(descs[0].friction) == np.float32(0.1)
    kind = descs[1].type
    descs[1].type = kind + 1
    with pytest.raises(RuntimeError):
        sim.engine.update_prims(descs)
    descs[1].type = kind
    sim.engine.update_prims(descs)
    assert np.array_equal(_frame(sim, P), ref)
