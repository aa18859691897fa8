"""Step graphs on the device: what captures, replays and refuses them."""
import ctypes

import numpy as np
import pytest

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


# 32x16x12: 4 steps a launch, graphs of 192; 128^3: 5 and 240
@pytest.mark.parametrize("shape,counts", [((32, 16, 12), (191, 192, 193, 199, 200, 201, 1001)),
                                          ((128, 128, 128), (239, 240, 241, 249, 250, 251, 1205))],
                         ids=["low", "tall"])
def test_heat7_calls_around_the_graph_length(hipdev, shape, counts):
    """Every call equals the same steps without a graph; later calls replay the
    first one's graph."""
    u0 = np.random.default_rng(6).random(shape[::-1])
    a, b = solvers.Heat7(shape, r=0.1), solvers.Heat7(shape, r=0.1)
    a.set_initial(u0)
    b.set_initial(u0)
    for n in counts:
        a.steps(n, graph=True)
        b.steps(n, graph=False)
        x = a.solution()
        assert np.isfinite(x).all() and np.array_equal(x, b.solution()), n
