"""Tapes of list steps that keep every step's state give what the replays of their segments give: the
same schedule of builds, the same states, records and gauges; also where lists go stale and steps halt and resume."""
import numpy as np
import pytest

from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd.adjoint import DifferentiableRun

pytestmark = pytest.mark.gpu


def _run(dim, precision, delta=0.0075, change=None):
    if dim == 2:
        lay = G.adjoint_tank(delta=delta, length=1.5, sigma=0.01, seed=5)
        xs, zs = [0.03, 0.06, 0.1], None
    else:
        lay = G.piston_basin_3d(delta=0.05, length=1.0, width=0.8)
        xs, zs = [0.1, 0.2, 0.2], [0.3, 0.5, 0.7]
    prm = lay.params
    if change:
        change(lay)
    spec = H.gauge_spec(xs, radius=3 * prm.delta, tau=prm.delta / 4, y_ref=prm.depth, zs=zs)
    sim = H.HipStep(prm, precision=precision)
    return DifferentiableRun(sim, dict(lay.state), 30, 8, spec, prm.piston_omega), prm


def _gradients(run, prm, scale=1.0):
    a, b = scale * np.array(prm.piston_a), scale * np.array(prm.piston_b)
    eta = run.forward(a, b)
    c = np.random.default_rng(5).normal(0.0, 1.0, eta.shape)
    return eta, run.backward(c, len(a)), run.sim.download()


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("precision", [H.FP64, H.FP32])
@pytest.mark.parametrize("skin", [None, "0.004"])
def test_kept_list_tapes_equal_their_replays(monkeypatch, dim, precision, skin):
    if skin:
        monkeypatch.setenv("RRSPH_HIP_LIST_SKIN", skin)
    res = {}
    for store in ("all", "segments"):
        monkeypatch.setenv("RRSPH_HIP_ADJ_STORE", store)
        run, prm = _run(dim, precision)
        first = _gradients(run, prm)
        _gradients(run, prm, 0.3)  # another run on the same tape
        res[store] = (first, run.sim.list_stats())
        run.sim.close()
    ((e1, g1, s1), q1), ((e0, g0, s0), q0) = res["all"], res["segments"]
    print("list stats", q1, q0, flush=True)
    assert q1["list_steps"] > 0
    assert q0["list_steps"] + q0["builds"] > q1["list_steps"] + q1["builds"]  # the replays ran
    if skin:
        assert q1["stale_halts"] > 0
    assert np.array_equal(e1, e0)
    for f in ("r", "v", "rho"):
        assert np.array_equal(s1[f], s0[f]), f
        # A replay does not launch a segment's last step; where that one builds, its reverse walks the cells: in 2D in
        # another order of FP64 sums (30 terms in 30 steps), in 3D with FP64 differences of positions instead of the
        # FP32 near records', which are rounded to 2^-24 of up to 2.1 cells, about 3e-7 of a particle spacing, a step.
        if dim == 2 or precision == H.FP32:
            tol = 1e-12 if dim == 2 else 1e-5
            assert np.max(np.abs(g1[f] - g0[f])) <= tol * np.max(np.abs(g0[f])), f
        else:
            assert np.array_equal(g1[f], g0[f]), f
    for f in ("a", "b"):  # sums over blocks are atomic adds
        tol = 1e-5 if dim == 3 and precision == H.FP32 else 1e-12
        assert np.max(np.abs(g1[f] - g0[f])) <= tol * np.max(np.abs(g0[f]))


@pytest.mark.parametrize("dim", [2, 3])
def test_a_kept_tape_without_memory_for_lists_starts_over(monkeypatch, dim):
    """In 2D on sorted steps, whose states all fit, in 3D with one segment's states: the results of such runs."""
    res = {}
    other = ("RRSPH_HIP_LIST", "0") if dim == 2 else ("RRSPH_HIP_ADJ_STORE", "segments")
    for name, var, value in (("short", "RRSPH_HIP_TAPE_LISTS", "2"), ("other", *other)):
        with monkeypatch.context() as m:
            m.setenv(var, value)
            run, prm = _run(dim, H.FP64)
            res[name] = _gradients(run, prm)
            run.sim.close()
    for k in (0, 1, 2):
        a, b = res["short"][k], res["other"][k]
        for f in ("r", "v", "rho") if k else (None,):
            x, y = (a, b) if f is None else (a[f], b[f])
            assert np.array_equal(x, y), (k, f)


def _smooth_viscosity(lay):  # without the switch between approaching and parting pairs, as a kink
    lay.params.artificial_shear_visc, lay.params.artificial_bulk_visc = 0.0, 0.5
    lay.state["itype"][7:4000:531] = 0  # and a few particles that no longer exist


# 4,237 particles: just above the smallest list tape; 8 lanes a particle below 25,000 and 2 above, ragged last blocks
@pytest.mark.parametrize("delta", [0.01294, 0.0075, 0.0051, 0.0047])
def test_2d_list_tapes_equal_sorted_ones(monkeypatch, delta):
    out = {}
    for lists in ("1", "0"):
        monkeypatch.setenv("RRSPH_HIP_LIST", lists)
        run, prm = _run(2, H.FP64, delta, _smooth_viscosity)
        out[lists] = (_gradients(run, prm), run.sim.list_stats(), prm.ntotal)
        run.sim.close()
    ((e1, g1, s1), q1, n), ((e0, g0, s0), q0, _) = out["1"], out["0"]
    print(n, q1, flush=True)
    assert q1["list_steps"] > 0 and q0["interval"] == 0
    # the neighbour sets are the same, only summation orders differ (the bounds of the 3D tapes' test)
    assert np.max(np.abs(e1 - e0)) <= 1e-12 * np.max(np.abs(e0))
    for f in ("a", "b", "r", "v", "rho"):
        assert np.max(np.abs(g1[f] - g0[f])) <= 1e-9 * np.max(np.abs(g0[f])), f
    for f in ("r", "v", "rho"):
        assert np.max(np.abs(s1[f] - s0[f])) <= 1e-12 * np.max(np.abs(s0[f])), f


def test_2d_tape_without_room_for_lists_starts_over_on_sorted_steps(monkeypatch):
    """A particle outside the cell grid has no list: the run starts over as a sorted one, with the same results as a
    context without lists."""
    out = {}

    def outside(lay):
        lay.params.consistency_check = False
        lay.state["r"][lay.params.nfluid - 1, 1] = lay.params.y_maxgeom + 3 * lay.params.cell_scale_k * lay.params.hsml

    for lists in ("1", "0"):
        monkeypatch.setenv("RRSPH_HIP_LIST", lists)
        run, prm = _run(2, H.FP64, change=outside)
        out[lists] = (_gradients(run, prm), run.sim.list_stats())
        run.sim.close()
    ((e1, g1, s1), q1), ((e0, g0, s0), _) = out["1"], out["0"]
    print(q1, flush=True)
    assert q1["builds"] > 0 and q1["interval"] == 0  # it tried, and keeps to sorted steps
    assert np.array_equal(e1, e0)
    for f in ("r", "v", "rho"):
        assert np.array_equal(g1[f], g0[f]) and np.array_equal(s1[f], s0[f]), f
