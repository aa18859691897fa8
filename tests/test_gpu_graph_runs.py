"""Step graphs on the device: what captures, replays and refuses them."""
import ctypes

import numpy as np
import pytest

import test_gpu_graph_lengths as G
from multigpu_advectiondiffusion_amd import _capi, solvers

pytestmark = pytest.mark.gpu


def test_short_graph_call_is_refused_during_a_capture(hipdev):
    """The caller's capture stays empty and valid, and the solver usable."""
    s = solvers.PeriodicBurgers(16)
    u0 = solvers.ic_fourier(16, seed=4)
    s.set_initial(u0)
    s.stream.synchronize()
    L = hipdev.lib()
    g, n = ctypes.c_void_p(), ctypes.c_size_t(99)
    assert L.hipStreamBeginCapture(s.stream.handle, 1) == 0
    with pytest.raises(_capi.MgadError):
        s.steps(2, graph=True)
    assert L.hipStreamEndCapture(s.stream.handle, ctypes.byref(g)) == 0
    assert L.hipGraphGetNodes(g, None, ctypes.byref(n)) == 0 and n.value == 0
    assert L.hipGraphDestroy(g) == 0
    _capi.last_error()
    assert np.array_equal(s.solution(), u0)
    s.steps(2, graph=True)
    assert s.state().steps == 2


# steps of a call that is captured and replayed, with a remainder: graphs of 16
# steps (WENO7 9, heat13 48, heat7 192), the first 50 of them launched directly
@pytest.mark.parametrize("make,n", [(G.periodic, 835), (G.slab, 835), (G.weno7, 475), (G.reference, 835),
                                    (G.heat13, 2503), (G.heat7, 9803), (G.batch, 835),
                                    (lambda: G.batch(True), 419)],
                         ids=["periodic", "slab", "weno7", "reference", "heat13", "heat7", "batch", "serial"])
def test_long_runs_equal_direct_launches(hipdev, make, n):
    """The call that captures, a short one, and one of replays from its start,
    with the program's own work and synchronisation in between."""
    a, run_a = make()
    b, run_b = make()
    for k in (n, 2, n // 3):
        run_a(k, True)
        run_b(k, False)
        for x, y in zip(G.result(a), G.result(b)):
            assert np.isfinite(x).all() and np.array_equal(x, y)


# 32x16x12: 4 steps a launch, graphs of 192; 128^3: 5 and 240
@pytest.mark.parametrize("shape,counts", [((32, 16, 12), (9800, 191, 192, 193, 199, 200, 201, 1001)),
                                          ((128, 128, 128), (12250, 239, 240, 241, 249, 250, 251, 1205))],
                         ids=["low", "tall"])
def test_heat7_calls_around_the_graph_length(hipdev, shape, counts):
    """Every call equals the same steps without a graph; the first one is
    captured, the others replay its graph."""
    u0 = np.random.default_rng(6).random(shape[::-1])
    a, b = solvers.Heat7(shape, r=0.1), solvers.Heat7(shape, r=0.1)
    for n in counts:
        a.set_initial(u0)
        b.set_initial(u0)
        a.steps(n, graph=True)
        b.steps(n, graph=False)
        x = a.solution()
        assert np.isfinite(x).all() and np.array_equal(x, b.solution()), n


def test_threads_capture_and_replay_at_the_same_time(hipdev):
    """Four host threads, each with its own stream and grid, in runs long enough
    to be captured and replayed, with a remainder: every result equals the same
    steps launched directly.  The threads issue only work ordered on their own
    streams, since a device-wide wait would invalidate a capture."""
    import threading

    sizes = (16, 32, 24, 48)
    u0s = [solvers.ic_fourier(n, seed=40 + i) for i, n in enumerate(sizes)]
    direct = []
    for n, u0 in zip(sizes, u0s):
        s = solvers.PeriodicBurgers(n)
        s.set_initial(u0)
        s.steps(4 * 300, graph=False)
        direct.append(s.solution())
    solver = [solvers.PeriodicBurgers(n) for n in sizes]
    hipdev.synchronize()
    got, errors = [None] * len(sizes), []

    def work(i):
        try:
            solver[i].set_initial(u0s[i])
            for _ in range(4):
                solver[i].steps(300, graph=True)
            got[i] = solver[i].solution()
        except Exception as e:  # reported below
            errors.append(repr(e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not errors, errors
    for x, y in zip(got, direct):
        assert x is not None and np.array_equal(x, y)


def _status(s):
    st = _capi.BurgersState()
    rc = _capi.lib().mgad_burgers_read_ctrl(s.stream.handle, s.ctrl.ptr, ctypes.byref(st))
    _capi.last_error()
    return rc, st


def _time(s):
    if isinstance(s, solvers.Weno7Burgers):
        t, _, steps = s.state()
        return t, steps
    st = _status(s)[1]
    return st.t, st.steps


@pytest.mark.parametrize("bad", [np.nan, np.inf, 1e200], ids=["nan", "inf", "overflow"])
def test_a_replayed_graph_stops_at_a_non_finite_value(hipdev, bad):
    """The graph of a finite run replayed on a field that is not, or stops
    being so inside the first step: u, t and the step count stay."""
    n = 32
    s = solvers.PeriodicBurgers(n)
    u0 = solvers.ic_fourier(n, seed=8)
    s.set_initial(u0)
    s.steps(820)
    assert s.state().steps == 820
    u0[10, 3, 4] = bad
    s.set_initial(u0, tend=10.0)
    s.steps(35)
    rc, st = _status(s)
    assert rc == _capi.MGAD_ERR_NONFINITE and (st.dt, st.t, st.steps) == (0.0, 0.0, 0)
    assert np.array_equal(s.solution(), u0, equal_nan=True)


@pytest.mark.parametrize("make", [lambda: solvers.PeriodicBurgers((32, 16, 12)),
                                  lambda: solvers.SlabBurgers((32, 16, 12), 3),
                                  lambda: solvers.Weno7Burgers((32, 16, 12))],
                         ids=["periodic", "slab", "weno7"])
def test_a_run_that_ends_inside_a_graph(hipdev, make):
    """tend falls inside a replay: the steps after it do nothing."""
    u0 = 0.5 + 0.4 * np.random.default_rng(9).random((12, 16, 32))
    a, b = make(), make()
    a.set_initial(u0)
    a.steps(820)  # captures
    b.set_initial(u0)
    b.steps(25, graph=False)
    tend = _time(b)[0] - 1e-4
    for s, calls, graph in ((a, (20, 20, 20), True), (b, (60,), False)):
        s.set_initial(u0, tend=tend)
        for n in calls:
            s.steps(n, graph=graph)
    assert _time(a) == _time(b) == (tend, 25)
    assert np.array_equal(a.solution(), b.solution())
