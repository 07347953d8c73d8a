"""A cell holding an infinite value: the slopes of its neighbours are the
reference's (0 towards an infinite difference, no number past one), so that one
solve leaves exactly the cells without a number that the oracle does, and the
others its values (1e-12 of the largest: one step of a converged Riemann solve)."""
import numpy as np
import pytest

import oracle
from rhyme_amd import hydro, ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("what", [0, 1, -1])
@pytest.mark.parametrize("value", [np.inf, -np.inf])
@pytest.mark.parametrize("limiter", [1, 2, 3, 4])
@pytest.mark.parametrize("ndim,dims", [(1, [41]), (2, [21, 19]), (3, [12, 11, 10])])
def test_one_infinite_cell(ndim, dims, limiter, value, what):
    p = hydro.make_params(
        ndim, rp=hydro.RiemannProblem(irs=hydro.Irs(n_iteration=200, tolerance=1e-13)),
        sl=hydro.SlopeLimiter(type=limiter), bc=hydro.SamrBc(types=[hydro.PERIODIC] * 6))
    cells = ics.random_smooth(ndim, dims, seed=5 + limiter)
    cells[(what % (ndim + 2),) + (9,) * ndim] = value
    ref = cells.copy()
    oracle.bc_set_boundaries(oracle.params_from(p), dims, ref)
    dx = [1.0 / 32] * ndim
    box = hydro.SamrBox(ndim, dims, cells=cells.copy())
    box.upload()
    hydro.rhyme_samr_bc_set_boundaries(p, box)
    hydro.rhyme_muscl_hancock_solve(p, box, dx, 1e-3)
    out = box.download().copy()
    box.close()
    oracle.mh_solve(oracle.params_from(p), dims, ref, dx, 1e-3)
    inner = (slice(0, ndim + 2),) + (slice(2, -2),) * ndim
    a, b = out[inner], ref[inner]
    fine = np.isfinite(b)
    assert not fine.all() and fine.sum() > 0.5 * fine.size
    print(limiter, value, what, "cells without a number", int((~fine[0]).sum()),
          int((~np.isfinite(a[0])).sum()), flush=True)
    assert np.array_equal(np.isfinite(a), fine)
    assert np.abs(a - b)[fine].max() <= 1e-12 * np.abs(b[fine]).max()
