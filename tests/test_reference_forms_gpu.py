"""The powlib build (RHY_FP64_POW_FAST=0) promises the reference's expressions in
the walks too: a solve and a step equal, bit for bit, the same composed from the
unit-level entry points (limiter, half step, Riemann solve, flux), which
evaluate them operation for operation, and the sum done here in IEEE doubles."""
import numpy as np
import pytest

from rhyme_amd import _lib, build, hydro, ics

pytestmark = pytest.mark.gpu


def params(ndim, limiter, omega):
    return hydro.make_params(
        ndim, rp=hydro.RiemannProblem(irs=hydro.Irs(n_iteration=100, tolerance=1e-8)),
        sl=hydro.SlopeLimiter(type=limiter, w=omega), cfl=hydro.Cfl(0.3),
        bc=hydro.SamrBc(types=[hydro.PERIODIC] * 6))


def composed(p, cells, n, dx, dt):
    """One 1D solve of the ghosted cells (6 planes of n + 4) from the unit level."""
    u = np.ascontiguousarray(cells[:3].T)  # (n + 4, 3)
    mid = u[1:-1]
    delta = hydro.limiter_batch(p, u[:-2], mid, u[2:])
    one = np.ones(len(mid), dtype=np.int32)
    l, r = hydro.half_step_batch(p, mid, delta, one, dx, dt)
    face = hydro.riemann_batch(p, r[:-1], l[1:], one[:-1])
    f = hydro.flux_batch(p, face, one[:-1])
    return (u[2:-2] + (dt / dx) * (f[:-1] - f[1:])).T


@pytest.mark.parametrize("omega", [0.0, 0.3])
@pytest.mark.parametrize("limiter", [1, 2, 3, 4])
def test_solve_is_the_unit_level_composed(limiter, omega):
    n, dx, dt = 200, 1.0 / 64, 1e-3
    with _lib.using(build.variant_path("powlib")):
        p = params(1, limiter, omega)
        cells = ics.random_smooth(1, [n], seed=limiter)
        box = hydro.SamrBox(1, [n], cells=cells.copy())
        box.upload()
        hydro.rhyme_samr_bc_set_boundaries(p, box)
        before = box.download().copy()
        hydro.rhyme_muscl_hancock_solve(p, box, [dx], dt)
        got = box.download()[:3, 2:-2].copy()
        box.close()
        want = composed(p, before, n, dx, dt)
    assert np.array_equal(got, want), np.abs(got - want).max()


@pytest.mark.parametrize("ndim,dims", [(1, [150]), (2, [40, 33]), (3, [20, 17, 15])])
def test_steps_are_the_solves(ndim, dims):
    with _lib.using(build.variant_path("powlib")):
        p = params(ndim, hydro.VAN_ALBADA, 0.0)
        cells = ics.random_smooth(ndim, dims, seed=3)
        dx = [1.0 / 32] * ndim
        a = hydro.SamrBox(ndim, dims, cells=cells.copy())
        b = hydro.SamrBox(ndim, dims, cells=cells.copy())
        a.upload()
        b.upload()
        dts = hydro.run(p, a, dx, 4)
        for dt in dts:
            assert hydro.rhyme_cfl_time_step(p, b, dx) == dt
            hydro.rhyme_samr_bc_set_boundaries(p, b)
            hydro.rhyme_muscl_hancock_solve(p, b, dx, dt)
        inner = (slice(0, ndim + 2),) + (slice(2, -2),) * ndim
        assert np.array_equal(a.download()[inner], b.download()[inner])
        a.close()
        b.close()
