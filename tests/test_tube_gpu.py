"""Small 1D boxes, whose steps run in one launch (tube_run_kernel), against
the module procedures called one by one, which take the kernels of a step:
bit for bit the same time steps and state, at sizes around a wave, a workgroup,
a second and third round and the kernel's limit, for every limiter and kind
of face, with and without faces that take the Riemann solver's slow paths."""
import numpy as np
import pytest

from rhyme_amd import _lib, hydro

pytestmark = pytest.mark.gpu

SIZES = [2, 3, 61, 62, 63, 64, 127, 765, 766, 767, 1024, 1534, 1535, 2040, 2041]


def params(limiter, faces, solver=2):
    return hydro.make_params(
        1, rp=hydro.RiemannProblem(irs=hydro.Irs(n_iteration=100, tolerance=1e-6)),
        sl=hydro.SlopeLimiter(type=limiter), mh=hydro.MusclHancock(solver_type=solver),
        cfl=hydro.Cfl(0.5), bc=hydro.SamrBc(types=faces))


def state(n, seed, vacuum):
    g = np.random.default_rng(seed)
    cells = np.zeros(hydro.box_shape(1, [n], hydro.ncmp_for(1)))
    rho = g.uniform(0.5, 2.0, n)
    v = g.uniform(-0.5, 0.5, n)
    p = g.uniform(0.5, 2.0, n)
    if vacuum:  # a receding pair: the solver's vacuum paths
        v[: n // 2] -= 8.0
        v[n // 2:] += 8.0
    cells[0, 2:-2] = rho
    cells[1, 2:-2] = rho * v
    cells[2, 2:-2] = 0.5 * rho * v * v + p / (5.0 / 3.0 - 1.0)
    return cells


def check(n, limiter, faces, precision, vacuum=False, steps=12, solver=2):
    p = params(limiter, faces, solver)
    cells = state(n, n + limiter, vacuum)
    a = hydro.SamrBox(1, [n], precision=precision, cells=cells.copy())
    b = hydro.SamrBox(1, [n], precision=precision, cells=cells.copy())
    a.upload()
    b.upload()
    dx = [1.0 / n]
    dts = hydro.run(p, a, dx, steps)
    want = []
    for _ in range(steps):
        dt = hydro.rhyme_cfl_time_step(p, b, dx)
        hydro.rhyme_samr_bc_set_boundaries(p, b)
        hydro.rhyme_muscl_hancock_solve(p, b, dx, dt)
        want.append(dt)
    assert np.array_equal(dts, np.array(want)), (n, limiter, faces)
    assert a.last_deferred() == b.last_deferred()
    hydro.rhyme_samr_bc_set_boundaries(p, b)  # a run leaves the ghosts filled
    x, y = a.download().copy(), b.download().copy()
    # (the receding states leave the gas law in a half step: NaN on both sides)
    assert vacuum or np.isfinite(y).all()
    assert np.array_equal(x, y, equal_nan=True), (n, limiter, faces)
    a.close()
    b.close()


@pytest.mark.parametrize("precision", [hydro.FP64, hydro.MIXED])
@pytest.mark.parametrize("n", SIZES)
def test_sizes(n, precision):
    check(n, 1 + n % 4, [1, 2, 1, 1, 1, 1], precision)


@pytest.mark.parametrize("faces", [(1, 1), (2, 1), (3, 3)])
@pytest.mark.parametrize("limiter", [1, 2, 3, 4])
def test_forms(limiter, faces):
    check(200, limiter, list(faces) * 3, hydro.FP64, solver=1 + limiter % 2)


@pytest.mark.parametrize("precision", [hydro.FP64, hydro.MIXED])
def test_slow_paths(precision):
    check(130, 2, [2, 2, 1, 1, 1, 1], precision, vacuum=True, steps=3)
    try:
        assert _lib.load().rhy_debug_defer(3, -1) == 0
        check(130, 4, [2, 2, 1, 1, 1, 1], precision)
    finally:
        _lib.load().rhy_debug_defer(0, -1)
