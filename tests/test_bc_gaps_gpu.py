"""The stand-alone ghost fill just under and at the number of x rows (16384) from
which it fills the gaps between rows instead of their two faces: every kind of
face, different ones on the two sides, inflow with the other components, FP64 and
mixed, bit for bit as the oracle fills them."""
import numpy as np
import pytest

import oracle
from rhyme_amd import hydro, ics

pytestmark = pytest.mark.gpu

DIMS = [(3, [3, 128, 128]), (3, [3, 129, 127]), (3, [2, 16384, 2]), (2, [3, 16384]),
        (2, [3, 16383]), (2, [2, 20011])]
FACES = [[1, 2, 2, 1, 1, 2], [3, 3, 1, 2, 3, 3], [4, 2, 4, 1, 2, 4], [1, 4, 3, 3, 4, 1],
         [2, 4, 4, 4, 1, 1]]


@pytest.mark.parametrize("precision", [hydro.FP64, hydro.MIXED])
@pytest.mark.parametrize("faces", FACES)
@pytest.mark.parametrize("ndim,dims", DIMS)
def test_fill_equals_oracle(ndim, dims, faces, precision):
    ncmp = hydro.ncmp_for(ndim)
    inflows = np.random.default_rng(3).uniform(0.5, 2.0, size=(6, ncmp))
    p = hydro.make_params(ndim, bc=hydro.SamrBc(types=faces, cons_inflows=inflows))
    cells = ics.random_smooth(ndim, dims, seed=4)
    cells[ndim + 2:] = np.random.default_rng(5).uniform(size=cells[ndim + 2:].shape)
    if precision == hydro.MIXED:
        cells = cells.astype(np.float32).astype(np.float64)
    box = hydro.SamrBox(ndim, dims, precision=precision, cells=cells.copy())
    box.upload()
    hydro.rhyme_samr_bc_set_boundaries(p, box)
    got = box.download().copy()
    box.close()
    want = cells.copy()
    oracle.bc_set_boundaries(oracle.params_from(p), dims, want)
    if precision == hydro.MIXED:
        want = want.astype(np.float32).astype(np.float64)
    assert np.array_equal(got, want)
