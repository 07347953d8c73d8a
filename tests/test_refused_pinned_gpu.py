"""Where the runtime refuses pinned host memory everything still works: a child
process loads a library whose hipHostMalloc refuses ahead of the HIP runtime,
then takes a time step size, uploads, steps and downloads a box large enough to
be staged."""
import os
import subprocess
import sys

import numpy as np
import pytest

from rhyme_amd import hydro, ics

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = "int asked = 0; int hipHostMalloc(void** p, unsigned long n, unsigned f)" \
       "{ (void)n; (void)f; *p = 0; ++asked; return 2; }"
CHILD = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
sys.path.insert(0, sys.argv[2] + "/tests")
import test_refused_pinned_gpu as t
print("result", repr(t.work()), ctypes.c_int.in_dll(shim, "asked").value)
"""


def work():
    """The wave-speed dt, the dts of three steps and a sum of the state."""
    n = 112  # 12.6 M values: 50 MB up and down in the mixed form
    p = hydro.make_params(
        3, rp=hydro.RiemannProblem(irs=hydro.Irs(n_iteration=100, tolerance=1e-6)),
        sl=hydro.SlopeLimiter(type=hydro.MINMOD), cfl=hydro.Cfl(0.2),
        bc=hydro.SamrBc(types=[hydro.REFLECTIVE] * 6))
    box = hydro.SamrBox(3, [n] * 3, precision=hydro.MIXED,
                        cells=ics.blast_3d(dims=[n] * 3, seed=2))
    box.upload()
    dt = hydro.rhyme_cfl_time_step(p, box, [1.0 / n] * 3)
    dts = hydro.run(p, box, [1.0 / n] * 3, 3)
    out = box.download()
    total = [float(np.sum(out[c])) for c in range(5)]
    box.close()
    return [float(dt)] + [float(x) for x in dts] + total


def test_everything_works_without_pinned_memory(tmp_path):
    src, lib = str(tmp_path / "refuse.c"), str(tmp_path / "librefuse.so")
    with open(src, "w") as f:
        f.write(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", lib, src], check=True)
    r = subprocess.run([sys.executable, "-c", CHILD, lib, ROOT], capture_output=True, text=True,
                       timeout=100)
    print(r.stdout, r.stderr[-2000:], flush=True)
    assert r.returncode == 0
    line = [x for x in r.stdout.splitlines() if x.startswith("result ")][0]
    asked = int(line.rsplit(" ", 1)[1])
    assert asked >= 2  # for the wave speed and for the staging area
    assert line[len("result "):].rsplit(" ", 1)[0] == repr(work())
