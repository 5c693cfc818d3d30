"""Tiled passes with two rows and with pairs of columns a work-group, at lengths
of every kind of plan that takes them, 3072 among them (whose two layouts may
round differently): two iterations against the FP32 oracle, within twice the bar
of the one-iteration tests (relative L2 1e-5)."""
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from _helpers import ALG_IDS, random_case, rel

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parents[1]

CHILD = r"""
import sys
root, out, L, nx, nrec = sys.argv[1], sys.argv[2], *map(int, sys.argv[3:])
sys.path[:0] = [root, root + "/tests"]
import numpy as np
from libspimage_amd import spimage as sp
from _helpers import GpuPhaser, random_case
res = {}
obj, amp, meas, sup, g0 = random_case((5, L), seed=L)
for alg in ("hio", "dm"):
    with GpuPhaser(sp, alg, amp, meas, sup, g0, beta=0.9) as g:
        assert g.iterate(2) == 0
        assert sp.spx_phaser_tiled(g.ph) == 1
        res[alg] = g.get("model")
        res["gammas"] = np.array(g.gammas()) if alg == "dm" else 0
obj, amp, meas, sup, g0 = random_case((L, nx), seed=L)
b = sp.Batch((L, nx), nrec)
for r in range(nrec):
    b.set_data(r, amp, meas, sup)
    b.set_model(r, g0)
b.set_algorithm(sp.sp_phasing_hio_alloc(sp.smap([(0, 0.9)]), sp.SpNoConstraints))
b.iterate(2)
m = b.model()
b.close()
assert all(np.array_equal(m[0], x) for x in m)
res["columns"] = m[0]
np.savez(out, **res)
"""


@pytest.mark.parametrize("L,E", [(2016, 8), (2304, 16), (2592, 8), (2688, 8), (3072, 16), (3072, 8), (3456, 16),
                                 (3600, 8), (3888, 8), (4000, 8), (5184, 16), (7200, 16)])
def test_tiled_iterations(tmp_path, o32, L, E):
    env = dict(os.environ, SPX_T4="1", SPX_TR="0", SPX_FFT_E=str(E))
    for k in ("SPX_NO_TUNE", "SPX_NO_T4", "SPX_COL_WIDE", "SPX_NT", "SPX_TUNE_FILE"):
        env.pop(k, None)
    nx = 16 * E  # the narrowest tiled rows; more groups of 4 columns than CUs
    nrec = 256 // (nx // 4) + 1
    out = tmp_path / "models.npz"
    print(f"child process {L} E={E} nx={nx} x {nrec}", flush=True)
    r = subprocess.run([sys.executable, "-c", CHILD, str(ROOT), str(out), str(L), str(nx), str(nrec)], env=env,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    got = np.load(out)
    for key, alg, shape in (("hio", "hio", (5, L)), ("dm", "dm", (5, L)), ("columns", "hio", (L, nx))):
        obj, amp, meas, sup, g0 = random_case(shape, seed=L)
        gam = got["gammas"] if alg == "dm" else (0.0, 0.0)
        o = o32.phaser(shape)
        o.set_inputs(amp, meas, sup, g0)
        assert o.iterate(o32.alg(ALG_IDS[alg], 0, beta=[(0, 0.9)], gamma1=float(gam[0]), gamma2=float(gam[1])), 2) == 0
        assert rel(got[key], o.g1) < 2e-5, key
