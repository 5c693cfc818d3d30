"""Tuning records of choices between kernels that earlier builds did not have:
lines under the older names are passed over and the choice is timed and
recorded anew; under the newer names they are replayed."""
import json
import os
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parents[1]

CHILD = r"""
import json, sys
root, shape = sys.argv[1], tuple(json.loads(sys.argv[2]))
sys.path[:0] = [root, root + "/tests"]
from libspimage_amd import spimage as sp
from _helpers import GpuPhaser, random_case
obj, amp, meas, sup, g0 = random_case(shape, seed=1)
with GpuPhaser(sp, "hio", amp, meas, sup, g0) as g:
    print(json.dumps([sp.spx_phaser_tiled(g.ph), sp.spx_phaser_nt_hints(g.ph)]))
"""


def _child(path, shape, **extra):
    env = dict(os.environ, SPX_TUNE_FILE=str(path))
    for k in ("SPX_FFT_E", "SPX_NO_TUNE", "SPX_T4", "SPX_NO_T4", "SPX_TR", "SPX_COL_WIDE", "SPX_NT", "SPX_NO_VOL"):
        env.pop(k, None)
    env.update(extra)
    print(f"child process {shape} {extra}", flush=True)
    r = subprocess.run([sys.executable, "-c", CHILD, str(ROOT), json.dumps(shape)], env=env, capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.strip().splitlines()[-1])


# masks 5 and 1 are not among those the tuner times, so only the file can set them
@pytest.mark.parametrize("shape", [(128, 2048), (2048, 128)])
def test_lines_with_two_row_tiles(tmp_path, shape):
    ny, nx = shape
    f = tmp_path / "tune.txt"
    old = f"shape {nx} {ny} 1 8 8 0\npair {nx} {ny} 0 0 0 5\n"
    f.write_text(old)
    lay, hints = _child(f, shape)
    assert hints != 5
    new = f.read_text()[len(old):].splitlines()
    assert sorted(ln.rsplit(" ", 3)[0] for ln in new) == [f"pair2 {nx} {ny} 0", f"shape2 {nx} {ny} 1"]
    f.write_text(old + f"shape2 {nx} {ny} 1 8 8 0\npair2 {nx} {ny} 0 1 0 5\n")
    before = f.read_text()
    assert _child(f, shape) == [1, 5]
    assert f.read_text() == before


def test_two_pass_volumes(tmp_path):
    f = tmp_path / "tune.txt"
    old = "shape 64 64 64 8 8 8\nvolume 64 64 64 0 1\n"
    f.write_text(old)
    assert _child(f, (64, 64, 64))[1] != 1
    assert f.read_text()[len(old):].startswith("volume2 64 64 64 0 ")
    f.write_text(old + "volume2 64 64 64 0 5\n")
    before = f.read_text()
    assert _child(f, (64, 64, 64))[1] == 5
    # the passes per axis keep their records
    assert _child(f, (64, 64, 64), SPX_NO_VOL="1")[1] == 1
    assert f.read_text() == before
