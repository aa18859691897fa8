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


# the set-up pass takes eight row segments at a time: groups across rows and
# planes, two and three segments a row, a last group of 1, 3 and 7 segments
@pytest.mark.parametrize("shape", [(7, 7, 7), (7, 41, 11), (26, 13, 15), (64, 9, 7), (65, 9, 11), (130, 7, 9)])
def test_reference_set_up_of_narrow_grids(hipdev, shape):
    nx, ny, nz = shape
    u = np.random.default_rng(5).uniform(-1.0, 1.0, size=(nz, ny, nx))
    s = solvers.ReferenceBurgers(shape, 0.1, 0.1, 0.1, scheme="Z1", viscous=False)
    for w in (s.w1, s.w2):
        w.upload(np.full((nz, ny, nx), 1e300), s.stream)
    s.set_initial(u)
    s.steps(1, 1e-3)
    for w in (s.w1, s.w2):  # the ghost layers are u's, nothing else was copied
        g = w.download(s.stream)
        inner = (slice(3, -3),) * 3
        assert not np.isin(g[inner], u[inner]).any()
        g[inner] = u[inner]
        assert np.array_equal(g, u)
    Lu, uo = np.zeros_like(u), u.copy()
    for rk in (1, 2, 3):
        for axis in range(3):
            O.adv(axis, u, Lu, 0.1, **O.REFERENCE)
        O.ssprk_b5(u, uo, Lu, rk, 1e-3)
    assert np.array_equal(s.solution(), u)
