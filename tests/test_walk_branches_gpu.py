"""Every branch of the FP64 walks' Riemann solve against the oracle: rows of
blocks of four equal cells, whose limited slopes are zero, so that the faces
between blocks hold exactly the problems put there.  Each pair of gases is
swept through mean velocities from supersonic on one side to supersonic on the
other; which part of the solution x/t = 0 falls into is worked out here and the
parts are counted, so that no case can miss its branch.

Tolerance: one step adds dt/dx (at most the Courant number 0.1 over the
fastest speed) times flux differences to the state.  A flux is a chain of some
30 operations of 1.1e-16 each around a Newton solution converged to 1e-13, so
the new state may differ by about 1e-13 of the largest flux change; 1e-12 of
each component's largest value covers it."""
import math

import numpy as np
import pytest

import oracle
from rhyme_amd import hydro, ics
from rhyme_amd.batch import SamrBatch

pytestmark = pytest.mark.gpu

BLOCK = 4
GAMMAS = [5.0 / 3.0, 7.0 / 5.0, 4.0 / 3.0, 1.5]
# rho, p on both sides and the velocity difference in units of the left sound speed
PAIRS = [((1.0, 1.0), (0.125, 0.1), 0.0),    # rarefaction, contact, shock
         ((0.3, 0.2), (1.0, 1.5), 0.0),      # shock, contact, rarefaction
         ((1.0, 1.0), (0.8, 0.9), -1.5),     # two shocks
         ((1.0, 1.0), (0.9, 1.1), 1.2),      # two rarefactions
         ((1.0, 1.0), (0.5, 1.0), 0.0)]      # a contact


def params(ndim, gamma, w_p=0.0, w_rho=0.0):
    p = hydro.make_params(
        ndim, rp=hydro.RiemannProblem(irs=hydro.Irs(n_iteration=200, tolerance=1e-13),
                                      w_vacuum_p=w_p, w_vacuum_rho=w_rho),
        sl=hydro.SlopeLimiter(type=hydro.SUPERBEE), cfl=hydro.Cfl(0.1),
        bc=hydro.SamrBc(types=[hydro.PERIODIC] * 6))
    p.gamma = gamma
    return p


def row_of(gamma, pairs=PAIRS):
    """Cells (rho, v, p) along the row: a block for either side of every
    problem, the mean velocity rising through the sweep and, for the mirror
    images, falling again (no block recedes from the next one's sweep)."""
    cells = []
    for (l, r, jump) in pairs:
        c = math.sqrt(gamma * l[1] / l[0])
        for sign in (1, -1):
            for m in np.linspace(-4.0, 4.0, 23):
                a, b = (l[0], m * c, l[1]), (r[0], (m + jump) * c, r[1])
                if sign < 0:
                    a, b = (b[0], -b[1], b[2]), (a[0], -a[1], a[2])
                cells += [a] * BLOCK + [b] * BLOCK
    return cells


def part(l, r, gamma):
    """(side, wave, part) of the solution at x/t = 0, or "vacuum generated"."""
    g1, g2 = gamma - 1.0, gamma + 1.0
    c = [math.sqrt(gamma * s[2] / s[0]) for s in (l, r)]
    if 2.0 * (c[0] + c[1]) / g1 <= r[1] - l[1]:
        return "vacuum generated"

    def f(p, s, cs):
        if p > s[2]:
            return (p - s[2]) * math.sqrt(2.0 / (g2 * s[0]) / (p + g1 / g2 * s[2]))
        return 2.0 * cs / g1 * ((p / s[2]) ** (g1 / (2.0 * gamma)) - 1.0)
    lo, hi = 1e-14, 1e4
    for _ in range(200):  # f is monotonic in p
        mid = math.sqrt(lo * hi)
        if f(mid, l, c[0]) + f(mid, r, c[1]) + r[1] - l[1] > 0.0:
            hi = mid
        else:
            lo = mid
    p = math.sqrt(lo * hi)
    us = 0.5 * (l[1] + r[1]) + 0.5 * (f(p, r, c[1]) - f(p, l, c[0]))
    side, s, cs, sign = ("right", r, c[1], 1.0) if us < 0.0 else ("left", l, c[0], -1.0)
    v, u = -sign * s[1], -sign * us  # as a left side
    if p > s[2] * (1.0 + 1e-9):
        speed = v - cs * math.sqrt(g2 / (2 * gamma) * p / s[2] + g1 / (2 * gamma))
        return side, "shock", "star" if speed < 0.0 else "ahead"
    tail = u - cs * (p / s[2]) ** (g1 / (2.0 * gamma))
    return (side, "rarefaction",
            "star" if tail < 0.0 else "fan" if v - cs < 0.0 else "ahead")


ALL_PARTS = {(s, w, q) for s in ("left", "right")
             for w, qs in (("shock", ("star", "ahead")), ("rarefaction", ("star", "fan", "ahead")))
             for q in qs}


def box_cells(ndim, axis, row, gamma):
    """The row along `axis` of an ndim box, three cells wide across; velocities
    across the axis differ from block to block."""
    dims = [3] * ndim
    dims[axis] = len(row)
    cells = np.zeros(hydro.box_shape(ndim, dims, hydro.ncmp_for(ndim)))
    shape = [1] * ndim
    shape[ndim - 1 - axis] = len(row)
    rho, v, p = (np.array(q).reshape(shape) for q in zip(*row))
    across = 0.1 * np.cos(np.arange(len(row)) // BLOCK).reshape(shape)
    inner = (slice(2, -2),) * ndim
    cells[(0,) + inner] = rho
    ke = 0.0
    for d in range(ndim):
        w = v if d == axis else across * (1.0 + d)
        w = np.where(rho > 0.0, w, 0.0)
        cells[(1 + d,) + inner] = rho * w
        ke = ke + 0.5 * rho * w * w
    cells[(ndim + 1,) + inner] = p / (gamma - 1.0) + ke
    return dims, cells


def step(ndim, axis, row, p):
    """One step on the device and with the oracle; returns the faces deferred."""
    dims, cells = box_cells(ndim, axis, row, p.gamma)
    dx = [1.0 / max(dims)] * ndim
    box = hydro.SamrBox(ndim, dims, cells=cells.copy())
    box.upload()
    hydro.run(p, box, dx, 1)
    out, deferred = box.download().copy(), box.last_deferred()
    box.close()
    ref = cells.copy()
    oracle.run(oracle.params_from(p), dims, ref, dx, 1)
    inner = (slice(2, -2),) * ndim
    assert np.isfinite(ref).all()
    for c in range(ndim + 2):
        a, b = out[(c,) + inner], ref[(c,) + inner]
        err = np.abs(a - b).max() / np.abs(b).max()
        print("ndim", ndim, "axis", axis, "component", c, "error", err, flush=True)
        assert err <= 1e-12
    return deferred


AXES = [(1, 0), (2, 0), (2, 1), (3, 0), (3, 1), (3, 2)]


@pytest.mark.parametrize("ndim,axis", AXES)
@pytest.mark.parametrize("gamma", GAMMAS)
def test_every_part_of_the_solution(gamma, ndim, axis):
    row = row_of(gamma)
    seen = {part(row[i], row[(i + 1) % len(row)], gamma) for i in range(len(row))
            if row[i] != row[(i + 1) % len(row)]}
    assert ALL_PARTS <= seen, ALL_PARTS - seen
    assert step(ndim, axis, row, params(ndim, gamma)) == 0


@pytest.mark.parametrize("ndim,axis", AXES)
def test_gas_under_the_pressure_floor(ndim, axis):
    """Pressures under w_vacuum's on one side or both are floored in the walk:
    none of their faces is left to the fixup."""
    gamma, floor = 5.0 / 3.0, 1e-3
    pairs = [((1.0, 2e-4), (0.5, 5e-4), 0.0), ((1.0, 2e-4), (0.7, 1.0), 0.0),
             ((0.6, 0.01), (1.0, 3e-4), 0.0), ((1.0, 4e-4), (0.9, 4e-4), -2.0)]
    row = row_of(gamma, pairs)
    assert step(ndim, axis, row, params(ndim, gamma, w_p=floor)) == 0


@pytest.mark.parametrize("w_rho,w_p", [(0.0, 0.0), (1e-3, 1e-4)])
@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.5, 4.0])
@pytest.mark.parametrize("ndim,axis", AXES)
def test_gas_beside_a_vacuum(ndim, axis, gamma, w_rho, w_p):
    """Vacuum on one side, at the velocities where each of the solver's answers
    holds; in the walk unless gamma > 3, where it may answer with a fan (small 1D
    boxes solve and count these faces on the spot)."""
    # (off v = -c and v = 2 c / (gamma - 1), where the answer jumps by a round-off)
    row = []
    for m in np.linspace(-5.03, 4.91, 21):
        for rho, p in ((1.0, 1.0), (0.4, 0.7)):
            c = math.sqrt(gamma * p / rho)
            row += [(rho, m * c, p)] * BLOCK + [(0.0, 0.0, 0.0)] * BLOCK
    deferred = step(ndim, axis, row, params(ndim, gamma, w_p=w_p, w_rho=w_rho))
    assert gamma > 3.0 or ndim == 1 or deferred == 0


@pytest.mark.parametrize("ndim,axis", AXES)
def test_vacuum_generated(ndim, axis):
    """Receding gases, the waves on either side of x/t = 0."""
    gamma = 5.0 / 3.0
    row = row_of(gamma, [((1.0, 1.0), (0.8, 0.9), 8.0)])
    step(ndim, axis, row, params(ndim, gamma))


@pytest.mark.parametrize("kind", ["vacuum", "floor"])
@pytest.mark.parametrize("ndim,dims", [(1, [[40], [700]]), (2, [[30, 21], [64, 9]]),
                                       (3, [[20, 17, 9], [40, 33, 27]])])
def test_batches_equal_boxes_alone(ndim, dims, kind):
    """Half empty boxes, and gas under the floor, in a batch (whose kernel leaves
    vacuum to the fixup, in a list of several parts) and alone."""
    p = params(ndim, 5.0 / 3.0, w_p=1e-3 if kind == "floor" else 0.0)
    cells = [ics.random_smooth(ndim, d, seed=8 + i) for i, d in enumerate(dims)]
    for c, d in zip(cells, dims):
        if kind == "floor":
            c[1:ndim + 2] *= 1e-4
        else:
            c[..., 2 + d[0] // 2:] = 0.0
    b = SamrBatch(ndim, dims, [[0.1] * ndim] * len(dims))
    for i, c in enumerate(cells):
        b.upload(i, c)
    dts = b.run(p, 3)
    assert kind == "floor" or b.last_deferred() > 0
    for i, (c, d) in enumerate(zip(cells, dims)):
        box = hydro.SamrBox(ndim, d, cells=c.copy())
        box.upload()
        assert np.array_equal(hydro.run(p, box, [0.1] * ndim, 3), dts[:, i])
        inner = (slice(0, ndim + 2),) + (slice(2, -2),) * ndim
        assert np.array_equal(box.download()[inner], b.download(i)[inner], equal_nan=True)
        box.close()
    b.close()
