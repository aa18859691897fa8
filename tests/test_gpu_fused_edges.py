"""Values and schemes that the other tests of the fused kernels leave out:
infinite and NaN nodes in several 7-point steps a launch, and the reference step's
16x16 tiles with every scheme."""
import numpy as np
import pytest

import oracle as O
from multigpu_advectiondiffusion_amd import reference_api as R
from multigpu_advectiondiffusion_amd import solvers

pytestmark = pytest.mark.gpu


# whole columns a block, 16-row and 36-row tiles; nodes inside a tile, in the
# columns and rows that two tiles share, next to the boundary and on it
@pytest.mark.parametrize("shape", [(64, 40, 20), (70, 60, 60), (180, 200, 44)], ids=["cube", "low", "tall"])
@pytest.mark.parametrize("nsteps", [4, 8, 10])
def test_heat7_infinite_and_nan_nodes_spread_as_in_single_steps(hipdev, shape, nsteps):
    nx, ny, nz = shape
    u = np.random.default_rng(24).uniform(-1.0, 2.0, size=(nz, ny, nx))
    u[nz // 2, ny // 2, nx // 2] = np.nan
    u[3, 14, 57] = np.inf
    u[nz - 2, ny - 2, 1] = -np.inf
    u[0, 5, 5] = np.nan
    h = solvers.Heat7(shape, r=0.1)
    h.set_initial(u)
    h.steps(nsteps, graph=False)
    with np.errstate(all="ignore"):
        O.heat7_fe(u, h.kx, h.ky, h.kz, h.dt, nsteps)
    assert np.array_equal(h.solution(), u, equal_nan=True)


LOCAL = {"Z1": O.REFERENCE, "JS": O.MB3, "Z2": dict(weno=O.WENO_Z, p=2, eps=1e-40, lf=O.LF_LOCAL)}


@pytest.mark.parametrize("shape", [(9, 8, 8), (24, 24, 24), (64, 64, 30), (39, 23, 20)])
@pytest.mark.parametrize("scheme", list(LOCAL))
@pytest.mark.parametrize("viscous", [False, True])
def test_reference_step_small_tiles(hipdev, shape, scheme, viscous):
    nx, ny, nz = shape
    u = np.random.default_rng(25).uniform(-1.0, 1.0, size=(nz, ny, nx))
    kx, ky, kz, dt = 2e-3, 3e-3, 1e-3, 1e-3
    R.CopyToConstantMemory(kx, ky, kz)
    s = solvers.ReferenceBurgers(shape, 0.1, 0.1, 0.1, scheme=scheme, viscous=viscous)
    s.set_initial(u)
    s.steps(1, dt)
    Lu, uo = np.zeros_like(u), u.copy()
    for rk in (1, 2, 3):
        for axis in range(3):
            O.adv(axis, u, Lu, 0.1, **LOCAL[scheme])
        if viscous:
            O.diff13_b5(u, Lu, kx, ky, kz)
        O.ssprk_b5(u, uo, Lu, rk, dt)
    assert np.array_equal(s.solution(), u)
