"""The 1D boxes whose steps run in one launch are those where that is faster:
at the sizes where the route changes a box takes no longer than a somewhat
larger one on the other route (the margin covers the clock's noise; past its
limit the one launch took 1.9 times as long)."""
import time

import numpy as np
import pytest

from rhyme_amd import hydro, ics

pytestmark = pytest.mark.gpu


def seconds(n, precision):
    p = hydro.make_params(1, sl=hydro.SlopeLimiter(type=hydro.VAN_LEER), cfl=hydro.Cfl(0.4),
                          rp=hydro.RiemannProblem(irs=hydro.Irs(n_iteration=100, tolerance=1e-6)),
                          bc=hydro.SamrBc(types=[hydro.PERIODIC] * 6))
    box = hydro.SamrBox(1, [n], precision=precision)
    drawing = dict(rho=1.0, v=[0.2], p=1.0, shapes=[], harmonics=[
        dict(axis=0, profile=ics.harmonic_profile(n, 0.1, 16.0), rho=0.5, v=[0.0], p=1.0)])
    times = []
    for _ in range(9):
        box.draw(p, drawing)
        hydro.run(p, box, [1.0 / n], 5)
        t = time.perf_counter()
        hydro.run(p, box, [1.0 / n], 100)
        times.append(time.perf_counter() - t)
    box.close()
    return float(np.median(times))


@pytest.mark.parametrize("precision,sizes", [(hydro.FP64, (1534, 1535, 2040)),
                                             (hydro.MIXED, (766, 767, 1534, 2040))])
def test_not_slower_than_a_larger_box(precision, sizes):
    large = seconds(3000, precision)
    for n in sizes:
        s = seconds(n, precision)
        print(n, precision, s, large, flush=True)
        assert s <= 1.3 * large, (n, s, large)
