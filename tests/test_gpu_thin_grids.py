"""Periodic grids of few columns and many planes, at the edges of the rule that
picks their bands (more than 128 bands of 1, 2, 3 and 4 planes, and beyond),
against the CPU oracle, bit for bit."""
import numpy as np
import pytest

import oracle as O
from multigpu_advectiondiffusion_amd import solvers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(16, 16, 128), (16, 16, 129), (16, 16, 200), (27, 11, 257), (27, 11, 441),
                                   (32, 32, 512), (16, 16, 513), (5, 4, 1100)])
@pytest.mark.parametrize("scheme,kw", [("Z2", O.Z2_GLOBAL), ("JS", O.JS_GLOBAL)])
def test_default_launch_of_thin_grids(hipdev, shape, scheme, kw):
    cfl = 0.3 * shape[0] / max(shape)
    s = solvers.PeriodicBurgers(shape, scheme=scheme, cfl=cfl)
    u = solvers.ic_fourier(shape, seed=33)
    s.set_initial(u)
    s.steps(1)
    O.burgers_run(u, (s.dx, s.dy, s.dz), cfl, 0.0, 10.0, nsteps=1, **kw)
    got = s.solution()
    assert np.array_equal(got, u), np.argwhere(got != u)[:5]
