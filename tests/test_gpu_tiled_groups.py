"""Tiled 2-D passes with two rows a work-group (lines too long for four in half
a CU's LDS) and with pairs of columns give the row-major passes' bits: odd
numbers of rows, single phasers, batches with per-reconstruction algorithms and
an idle slot, graph replays.  3072 is left to the comparison with the oracle:
its two layouts have always rounded differently (2e-7 an iteration)."""
import numpy as np
import pytest

from test_gpu_transposed import KEYS, _child

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("single,batch,E", [
    ([7, 1024], [1024, 128], "8"),
    ([2048, 256], [5, 2048], "16"),
    ([1536, 128], [5, 1536], "8"),
    ([3, 4096], [4096, 256], "16"),
    ([2, 8192], [8192, 256], "16"),
])
def test_tiled_equals_row_major(tmp_path, single, batch, E):
    shapes = {"single": single, "batch": batch}
    tiled = _child(tmp_path, "tiled", shapes, SPX_T4="1", SPX_TR="0", SPX_FFT_E=E)
    rm = _child(tmp_path, "row_major", shapes, SPX_NO_T4="1", SPX_TR="0", SPX_FFT_E=E)
    assert int(tiled["layout_single"]) == 1 and int(rm["layout_single"]) == 0
    for key in KEYS:
        assert np.array_equal(tiled[key], rm[key]), key
    assert bool(tiled["graph_equal"]) and bool(rm["graph_equal"])
