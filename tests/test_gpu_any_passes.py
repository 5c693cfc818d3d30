"""The fused passes of lines without a Stockham plan at the edges of their
padded lengths (the shortest and the longest line of each power of two), in
rows and in columns, against the FP32 oracle within the bar of the other
one-iteration tests (relative L2 1e-5); and the optional paths of those passes
(amplitude margins, the phased-amplitude objective, a Stockham axis beside)."""
import numpy as np
import pytest

from _helpers import ALG_IDS, GpuPhaser, random_case, rel

pytestmark = pytest.mark.gpu

# (padded length: shortest and longest line without a plan)
EDGES = [11, 13, 17, 31, 33, 62, 67, 127, 131, 254, 257, 511, 514, 1023, 1025, 2047, 2049, 4095]


@pytest.mark.parametrize("rows", [True, False])
@pytest.mark.parametrize("L", EDGES)
def test_one_iteration_at_the_edges(sp, o32, L, rows):
    shape = (5, L) if rows else (L, 5)
    obj, amp, meas, sup, g0 = random_case(shape, seed=L)
    for alg in ("hio", "dm"):
        with GpuPhaser(sp, alg, amp, meas, sup, g0, beta=0.9) as g:
            assert g.iterate(1) == 0
            gam = g.gammas() if alg == "dm" else (0.0, 0.0)
            o = o32.phaser(shape)
            o.set_inputs(amp, meas, sup, g0)
            assert o.iterate(o32.alg(ALG_IDS[alg], 0, beta=[(0, 0.9)], gamma1=gam[0], gamma2=gam[1]), 1) == 0
            assert rel(g.get("model"), o.g1) < 1e-5
            assert rel(g.get("fmodel"), np.fft.fftn(o.g1.astype(np.complex128))) < 1e-5
            assert abs(g.efourier()[0] - o.efourier()[0]) < 1e-4 * o.efourier()[0]


@pytest.mark.parametrize("shape", [(47, 37), (64, 37), (47, 64), (13, 11, 17)])
def test_margins_and_phased_amplitudes(sp, shape):
    """Against float64 numpy on the same inputs, one ER iteration."""
    obj, amp, meas, sup, g0 = random_case(shape, seed=2)
    g64 = g0.astype(np.complex128)
    F = np.fft.fftn(g64)
    lo, hi = (0.9 * amp).astype(np.float32), (1.2 * amp).astype(np.float32)
    m = np.clip(np.abs(F), lo, hi) / np.abs(F)
    want = np.where(sup, np.fft.ifftn(np.where(meas, F * m, F)), 0)
    with GpuPhaser(sp, "er", amp, meas, sup, g0, constraints=sp.SpAmplitudeErrorMargin) as g:
        sp.sp_phaser_set_amplitudes_margins(g.ph, g._img(lo), g._img(hi))
        assert g.iterate(1) == 0
        assert rel(g.get("model"), want) < 1e-5
    rng = np.random.default_rng(4)
    pa = (amp * np.exp(2j * np.pi * rng.random(shape))).astype(np.complex64)
    want = np.where(sup, np.fft.ifftn(np.where(meas, pa, F)), 0)
    with GpuPhaser(sp, "er", amp, meas, sup, g0) as g:
        sp.sp_phaser_set_phased_amplitudes(g.ph, g._img(pa, meas))
        sp.sp_phaser_set_objective(g.ph, sp.SpRecoverAmplitudes)
        assert g.iterate(1) == 0
        assert rel(g.get("model"), want) < 1e-5
