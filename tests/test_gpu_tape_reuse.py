"""A differentiable run of the shape of the one before reuses its tape's buffers: the same gauges and gradients as on
buffers allocated for the run, whatever ran in between (other coefficients, another shape, a failed call)."""
import numpy as np
import pytest

from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd.adjoint import DifferentiableRun

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,precision", [(2, H.FP64), (3, H.FP64), (3, H.FP32)])
def test_runs_on_a_kept_tape_equal_a_fresh_context(dim, precision):
    lay = G.adjoint_tank(delta=0.02, length=2.0) if dim == 2 else G.piston_basin_3d(delta=0.05, length=1.0, width=0.8)
    prm = lay.params
    zs = None if dim == 2 else [0.3, 0.5]
    spec = H.gauge_spec([0.1, 0.2], radius=3 * prm.delta, tau=prm.delta / 4, y_ref=prm.depth, zs=zs)
    a, b = np.array(prm.piston_a), np.array(prm.piston_b)

    def once(run, scale, steps=12, every=5):
        run.nsteps, run.every = steps, every
        eta = run.forward(scale * a, scale * b)
        return eta, run.backward(2 * (eta - prm.depth), len(a))

    def fresh():
        return DifferentiableRun(H.HipStep(prm, precision=precision), dict(lay.state), 12, 5, spec, prm.piston_omega)

    kept = fresh()
    once(kept, 1.0)
    once(kept, 0.3)
    once(kept, 1.0, steps=7, every=3)
    with pytest.raises(H.RrsphError):
        kept.sim.adjoint_forward(12, 0, spec)
    once(kept, 0.5)
    eta, g = once(kept, 1.0)
    ref = fresh()
    once(ref, 1.0, steps=11)  # another shape: its tape is freed; 3D list builds start from the same measured interval
    eta_r, g_r = once(ref, 1.0)
    assert np.array_equal(eta, eta_r)
    for f in ("r", "v", "rho"):
        assert np.array_equal(g[f], g_r[f]), f
    # the coefficients' sums over blocks are atomic adds: equal to rounding
    for f in ("a", "b"):
        assert np.max(np.abs(g[f] - g_r[f])) <= 1e-12 * np.max(np.abs(g_r[f]))
    part = kept.sim.adjoint_backward(2 * (eta - prm.depth), len(a), state=False)
    assert set(part) == {"a", "b"} and np.max(np.abs(part["a"] - g["a"])) <= 1e-12 * np.max(np.abs(g["a"]))
