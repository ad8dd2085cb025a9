"""A particle at an infinite, a huge or a NaN position beside finite ones of the
same cell block: in the particle-to-grid scatter and its adjoint counterpart it
reaches no other cell's sums.  The finite particles' substep and adjoint are
those of a context without it."""
import numpy as np
import pytest
import torch

from scenes import capsule_scene, particles_box
from test_gpu_parity import build, flat

pytestmark = pytest.mark.gpu


def _run(st, adj1):
    sim_cfg, prims, _ = capsule_scene(n=len(st))
    sim, P = build(sim_cfg, prims, st)
    P.set_action(0, sim_cfg["substeps"], np.zeros(3))
    sim.substep(0)
    out = flat(sim.get_state(1))
    sim.clear_grads()
    sim.add_obs_grad(1, torch.as_tensor(adj1[:, 0:6], dtype=torch.float32), None)
    a = sim.engine.adjoint(1)
    a[6:24, sim.engine.scene_cols(0)] = sim._to_slots(torch.as_tensor(adj1[:, 6:24], dtype=torch.float32, device="cuda")).t()
    sim.substep_grad(0)
    gx, gv, gF, gC = [t.detach().cpu().double().numpy() for t in sim.get_adjoint(0)]
    return out, np.concatenate([gx, gv, gC.reshape(-1, 9), gF.reshape(-1, 9)], 1)


@pytest.mark.parametrize("where", [float("-inf"), -1e30, float("inf"), 1e30, float("nan")])
@pytest.mark.parametrize("n", [15, 200, 1500])
def test_special_position(n, where):
    print("case special position n=%d at %s" % (n, where), flush=True)
    # a block at the corner of the 32^3 grid that the position is binned into
    lo, hi = (0.9, 0.99) if where > 0 else (0.02, 0.14)
    st = particles_box(n, [lo] * 3, [hi] * 3, seed=n, v_sigma=0.5, F_jitter=0.05)
    rng = np.random.default_rng(n)
    st[:, 6:15] = rng.normal(0, 5.0, (n, 9))
    st = st.astype(np.float32).astype(np.float64)
    adj1 = rng.normal(size=(n, 24)).astype(np.float32).astype(np.float64)
    ref, gref = _run(st, adj1)
    odd = st[:1].copy()
    odd[:, 0:3] = where
    got, g = _run(np.concatenate([st, odd]), np.concatenate([adj1, adj1[:1]]))
    # a NaN particle's own cell is cell 0, nodes 0 to 2: particles with a base of 3
    # in some axis read none of them
    keep = np.ones(n, bool)
    if np.isnan(where):
        base = np.trunc(st[:, 0:3] * 32 - 0.5)
        keep = (base >= 3).any(1)
        assert keep.any()
        # nodes of NaN mass count as empty
        assert (got[:n][base.max(1) == 0, 3:6] == 0.0).all()
    # the same kernels with one slot more: sums in another order
    for a, b, rel in ((got[:n], ref, 1e-4), (g[:n], gref, 1e-3)):
        for sl in (slice(0, 3), slice(3, 6), slice(6, 15), slice(15, 24)):
            assert np.isfinite(a[keep, sl]).all()
            assert np.abs(a[keep, sl] - b[keep, sl]).max() <= rel * np.abs(b[:, sl]).max()
