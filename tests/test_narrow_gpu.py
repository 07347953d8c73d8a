"""2D boxes on both sides of the width, and just over the size, where rhy_run's
route changes between the walk and the flux planes: N steps equal N rounds of the
module procedures bit for bit, with the ghost faces of the final state filled."""
import numpy as np
import pytest

import oracle
from rhyme_amd import hydro, ics

pytestmark = pytest.mark.gpu

# (precision, dims): 2^17 cells and a little more, even and odd
CASES = [(hydro.FP64, [2, 65536]), (hydro.FP64, [31, 4229]), (hydro.FP64, [32, 4097]),
         (hydro.MIXED, [5, 26215]), (hydro.MIXED, [64, 2049]), (hydro.MIXED, [65, 2017])]


@pytest.mark.parametrize("bc", [[1, 2, 3, 3, 0, 0], [3, 3, 4, 1, 0, 0]])
@pytest.mark.parametrize("solver", [hydro.MEMORY_INTENSIVE, hydro.CPU_INTENSIVE])
@pytest.mark.parametrize("precision,dims", CASES)
def test_run_equals_procedures(precision, dims, solver, bc):
    inflows = np.zeros((6, hydro.ncmp_for(2)))
    inflows[:, 0], inflows[:, 3] = 1.1, 2.0
    p = hydro.make_params(
        2, rp=hydro.RiemannProblem(irs=hydro.Irs(n_iteration=100, tolerance=1e-6)),
        sl=hydro.SlopeLimiter(type=1 + dims[0] % 4), mh=hydro.MusclHancock(solver_type=solver),
        cfl=hydro.Cfl(0.3), bc=hydro.SamrBc(types=bc, cons_inflows=inflows))
    cells = ics.random_smooth(2, dims, seed=dims[0])
    dx = [1.0 / 32, 1.0 / 30]
    boxes = []
    for _ in range(2):
        boxes.append(hydro.SamrBox(2, dims, cells=cells.copy(), precision=precision))
        boxes[-1].upload()
    a, b = boxes
    dts = hydro.run(p, a, dx, 3)
    want = []
    for _ in range(3):
        want.append(hydro.rhyme_cfl_time_step(p, b, dx))
        hydro.rhyme_samr_bc_set_boundaries(p, b)
        hydro.rhyme_muscl_hancock_solve(p, b, dx, want[-1])
    x, y = a.download().copy(), b.download().copy()
    assert np.array_equal(dts, np.array(want))
    assert np.isfinite(y).all()
    inner = (slice(0, 4), slice(2, -2), slice(2, -2))
    assert np.array_equal(x[inner], y[inner])
    filled = x.copy()
    oracle.bc_set_boundaries(oracle.params_from(p), dims, filled)
    if precision == hydro.MIXED:
        filled = filled.astype(np.float32).astype(np.float64)
    assert np.array_equal(x[:4, 2:-2, :], filled[:4, 2:-2, :])
    assert np.array_equal(x[:4, :, 2:-2], filled[:4, :, 2:-2])
    a.close()
    b.close()
