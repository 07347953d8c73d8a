"""Host transfers of boxes and batches at the sizes where their route changes:
the direct copy, staged copies of a few chunks and of a partial last one, and
two threads that both ask for the staging memory.  What was uploaded comes
back bit for bit (mixed form: rounded to FP32 once)."""
import threading

import numpy as np
import pytest

from rhyme_amd import hydro
from rhyme_amd.batch import SamrBatch

pytestmark = pytest.mark.gpu

# 1D boxes of 6 planes: bytes of a state are 48 (n + 4) in FP64; the direct
# copy ends at 2 MiB, chunks are 256 KiB up to 4 MiB and 2 MiB from 32 MiB on
SIZES = [100, (2 << 20) // 48 - 5, (2 << 20) // 48 + 5, 100003, 700001, 1500007]


def cells_of(n, seed):
    g = np.random.default_rng(seed)
    return g.standard_normal(hydro.box_shape(1, [n], 6))


def round_trip(n, precision, seed):
    box = hydro.SamrBox(1, [n], 6, precision)
    cells = cells_of(n, seed)
    box.cells[...] = cells
    box.upload()
    box.cells[...] = 0.0
    got = box.download()
    want = cells.astype(np.float32).astype(np.float64) if precision == hydro.MIXED else cells
    assert np.array_equal(got, want), (n, precision)
    payload = box.snapshot()
    assert np.array_equal(payload.reshape(6, n), want[:, 2:-2].astype(np.float32)), n
    box.load_snapshot(payload[::-1].copy())
    got = box.download()[:, 2:-2]
    assert np.array_equal(got, payload[::-1].reshape(6, n).astype(np.float64)), n
    box.close()


@pytest.mark.parametrize("precision", [hydro.FP64, hydro.MIXED])
@pytest.mark.parametrize("n", SIZES)
def test_box(n, precision):
    round_trip(n, precision, n % 97)


@pytest.mark.parametrize("precision", [hydro.FP64, hydro.MIXED])
def test_batch(precision):
    dims = [[50], [60001], [100003]]
    b = SamrBatch(1, dims, [[1.0]] * 3, ncmp=6, precision=precision)
    cells = [cells_of(d[0], i) for i, d in enumerate(dims)]
    for i, c in enumerate(cells):
        b.upload(i, c)
    if precision == hydro.MIXED:
        cells = [c.astype(np.float32).astype(np.float64) for c in cells]
    for i, c in enumerate(cells):
        assert np.array_equal(b.download(i), c), i
    payload = b.snapshot()
    assert np.array_equal(payload, np.concatenate(
        [c[:, 2:-2].astype(np.float32).ravel() for c in cells]))
    b.load_snapshot(-payload)
    assert np.array_equal(b.snapshot(), -payload)
    b.close()


def test_threads():
    bad = []

    def work(seed):
        try:
            for _ in range(3):
                round_trip(300007, hydro.FP64, seed)
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            bad.append(e)
    ts = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
