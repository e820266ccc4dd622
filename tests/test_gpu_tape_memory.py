"""A tape that keeps every state admits its lists by a likely number of builds; where a run builds more often, the lists
stay within the same bound (here set by RRSPH_HIP_TAPE_MEMORY, by default half the free memory), and the run starts over
as one whose tape fits."""
import ctypes

import numpy as np
import pytest

from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd.adjoint import DifferentiableRun

pytestmark = pytest.mark.gpu
STEPS, MIB = 40, 1 << 20


def _layout(dim):
    if dim == 2:
        return G.adjoint_tank(delta=0.0035, length=1.5), [0.03, 0.1], None
    return G.piston_basin_3d(delta=0.03, length=1.0, width=0.8), [0.1, 0.2], [0.3, 0.5]


def _free_memory(sim):
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert sim.L.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0  # of the HIP runtime the library links
    return free.value


def _gradients(dim):
    lay, xs, zs = _layout(dim)
    prm = lay.params
    spec = H.gauge_spec(xs, radius=3 * prm.delta, tau=prm.delta / 4, y_ref=prm.depth, zs=zs)
    run = DifferentiableRun(H.HipStep(prm, precision=H.FP64), dict(lay.state), STEPS, 8, spec, prm.piston_omega)
    run.sim.upload(*(lay.state[f] for f in ("r", "v", "rho", "itype")))
    a, b = np.array(prm.piston_a), np.array(prm.piston_b)
    free = _free_memory(run.sim)
    eta = run.forward(a, b)
    used = free - _free_memory(run.sim)
    g = run.backward(2 * (eta - prm.depth), len(a))
    stats = run.sim.list_stats()
    run.sim.close()
    return eta, g, used, stats


@pytest.mark.parametrize("dim", [2, 3])
def test_lists_of_a_kept_tape_stay_within_its_bound(monkeypatch, dim):
    n = _layout(dim)[0].params.ntotal
    monkeypatch.setenv("RRSPH_HIP_LIST_SKIN", "0.0002")  # every step builds
    # bytes of the kept states and sorts of FP64 steps, of a build's lists (their capacity: max_neighbours with the
    # skin, 8 more and 8 rows of padding), and of the rest of the tape (checkpoints, adjoints, records)
    states = STEPS * n * (124 if dim == 2 else 140)
    lists = 4 * n * (_layout(dim)[0].params.max_neighbours + 19)
    rest = 6 * n * 120 + n * 400 + 16 * MIB
    bound = states + (STEPS // 4 + STEPS // 8 + 2) * lists  # builds in every fourth step and at the checkpoints, and one
    monkeypatch.setenv("RRSPH_HIP_TAPE_MEMORY", str(bound))
    eta, g, used, stats = _gradients(dim)
    print("tape memory", dim, "n", n, "bound MiB", bound / MIB, "used", used / MIB, stats, flush=True)
    assert stats["builds"] > STEPS // 4 + STEPS // 8 + 2  # it ran out
    assert used <= bound + rest
    monkeypatch.setenv(*(("RRSPH_HIP_LIST", "0") if dim == 2 else ("RRSPH_HIP_ADJ_STORE", "segments")))
    eta0, g0, *_ = _gradients(dim)
    assert np.array_equal(eta, eta0)
    for f in ("r", "v", "rho"):
        assert np.array_equal(g[f], g0[f]), f


@pytest.mark.parametrize("dim", [2, 3])
def test_a_run_that_fits_keeps_its_lists_after_one_that_did_not(monkeypatch, dim):
    """What ran out of room is a run of one shape; a shorter one on the same context keeps its states and lists."""
    monkeypatch.setenv("RRSPH_HIP_LIST_SKIN", "0.0002")  # every step builds
    lay, xs, zs = _layout(dim)
    prm = lay.params
    spec = H.gauge_spec(xs, radius=3 * prm.delta, tau=prm.delta / 4, y_ref=prm.depth, zs=zs)
    a, b = np.array(prm.piston_a), np.array(prm.piston_b)
    c = np.random.default_rng(7).normal(0.0, 1.0, (16, 2))
    out = []
    for long_run_first in (True, False):
        monkeypatch.setenv("RRSPH_HIP_TAPE_LISTS", "20")
        run = DifferentiableRun(H.HipStep(prm, precision=H.FP64), dict(lay.state), STEPS, 8, spec, prm.piston_omega)
        if long_run_first:
            run.forward(a, b)
            assert run.sim.list_stats()["builds"] > 20  # it ran out
        run.nsteps = 16
        for _ in range(2):  # by the second run the schedule is a build in every step
            before = run.sim.list_stats()
            eta = run.forward(a, b)
            g = run.backward(c, len(a))
            after = run.sim.list_stats()
        # the forward's steps built their lists, and the reverse pass replayed none
        assert after["builds"] - before["builds"] == 16 and after["list_steps"] == before["list_steps"]
        out.append((eta, g))
        run.sim.close()
    assert np.array_equal(out[0][0], out[1][0])
    for f in ("r", "v", "rho"):
        assert np.array_equal(out[0][1][f], out[1][1][f]), f
