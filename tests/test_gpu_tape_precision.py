"""3D FP32 tapes that keep every state give bit for bit the gradients of the segments' replays (but for the coefficients',
whose sums over blocks are atomic adds): a segment's last step that builds lists is reversed with FP64 separations on
both, also where every step is a segment of its own."""
import numpy as np
import pytest

from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd.adjoint import DifferentiableRun

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [1, 3, 5])
def test_kept_3d_fp32_tapes_equal_their_replays(monkeypatch, every):
    lay = G.piston_basin_3d(delta=0.05, length=1.0, width=0.8)
    prm = lay.params
    spec = H.gauge_spec([0.1, 0.2], radius=3 * prm.delta, tau=prm.delta / 4, y_ref=prm.depth, zs=[0.3, 0.5])
    a, b = np.array(prm.piston_a), np.array(prm.piston_b)
    c = np.random.default_rng(5).normal(0.0, 1.0, (12, 2))
    monkeypatch.setenv("RRSPH_HIP_LIST_SKIN", "0.0005")  # many builds
    out = {}
    for store in ("all", "segments"):
        monkeypatch.setenv("RRSPH_HIP_ADJ_STORE", store)
        run = DifferentiableRun(H.HipStep(prm, precision=H.FP32), dict(lay.state), 12, every, spec, prm.piston_omega)
        out[store] = (run.forward(a, b), run.backward(c, len(a)))
        print("tapes", every, store, run.sim.list_stats(), flush=True)
        run.sim.close()
    (e1, g1), (e0, g0) = out["all"], out["segments"]
    assert np.array_equal(e1, e0)
    for f in ("r", "v", "rho"):
        assert np.array_equal(g1[f], g0[f]), f
