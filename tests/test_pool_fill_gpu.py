"""The ghost fill of a pool whose boxes come at different times: with one new box
among many, as many as one fill names, one more, and all of them, every box
evolves bit for bit as it does alone."""
import numpy as np
import pytest

from rhyme_amd import hydro, ics
from rhyme_amd.batch import SamrPool

pytestmark = pytest.mark.gpu

FACES = [[1] * 6, [2] * 6, [3] * 6, [1, 1, 2, 2, 3, 3]]


def params(i, ndim):
    return hydro.make_params(
        ndim, rp=hydro.RiemannProblem(irs=hydro.Irs(n_iteration=100, tolerance=1e-6)),
        sl=hydro.SlopeLimiter(type=1 + i % 4), cfl=hydro.Cfl(0.2),
        bc=hydro.SamrBc(types=FACES[i % 4]))


@pytest.mark.parametrize("precision", [hydro.FP64, hydro.MIXED])
@pytest.mark.parametrize("ndim", [1, 2, 3])
@pytest.mark.parametrize("new", [1, 15, 16, 17, 24])
def test_boxes_equal_themselves_alone(new, ndim, precision):
    """24 boxes, `new` of them set again between two runs."""
    g = np.random.default_rng(new + ndim)
    dims = [[int(x) for x in g.integers(2, 20, size=ndim)] for _ in range(24)]
    cells = [ics.random_smooth(ndim, d, seed=i) for i, d in enumerate(dims)]
    again = sorted(g.choice(24, size=new, replace=False).tolist())
    pool = SamrPool(ndim, 1 << 28, precision=precision)
    slots = [pool.add(d, [0.1] * ndim, c, 1 + i % 4, FACES[i % 4])
             for i, (d, c) in enumerate(zip(dims, cells))]
    pool.run_async(params(0, ndim), 3)
    for i in again:
        pool.upload(slots[i], cells[i])
    pool.run_async(params(0, ndim), 2)
    pool.sync()
    for i, (d, c) in enumerate(zip(dims, cells)):
        box = hydro.SamrBox(ndim, d, cells=c.copy(), precision=precision)
        box.upload()
        hydro.run(params(i, ndim), box, [0.1] * ndim, 2 if i in again else 5)
        inner = (slice(0, ndim + 2),) + (slice(2, -2),) * ndim
        assert np.array_equal(pool.download(slots[i])[inner], box.download()[inner]), (i, d)
        box.close()
    pool.close()
