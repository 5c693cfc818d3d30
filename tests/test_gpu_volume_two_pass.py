"""Two-pass iterations of volumes (the 3-D transform split between a pass over
x and part of y and a pass over z and the rest of y) at every length that has
an instance, as the row pass's length and as the column pass's, against the
same iteration in float64 (scipy).  The bar is the other one-iteration tests'
relative L2 1e-5; metrics and the Fourier model likewise.  Margins, the
phased-amplitude objective and batches with mixed algorithms and idle slots
run the same kernels' optional paths."""
import numpy as np
import pytest
import scipy.fft

from _helpers import GpuPhaser, random_case, rel

pytestmark = pytest.mark.gpu

# (nz, n, n): column instance nz, row instance n
SHAPES = [(64, 256), (256, 64), (72, 240), (240, 72), (80, 216), (216, 80), (96, 200), (200, 96), (120, 192),
          (192, 120), (128, 160), (160, 128), (144, 144)]


def _fft(a, inverse=False):
    f = scipy.fft.ifftn if inverse else scipy.fft.fftn
    return f(a, workers=8)


def _project(F, amp, meas):
    with np.errstate(divide="ignore", invalid="ignore"):
        m = amp / np.abs(F)
    P = np.where(np.isfinite(m), F * np.where(np.isfinite(m), m, 0), amp)
    return np.where(meas, P, F)


def _step(alg, g, amp, meas, sup, beta, gam=(0, 0)):
    P = _fft(_project(_fft(g), amp, meas), True)
    if alg == "dm":
        Pf = _fft(_project(_fft(np.where(sup, g, -gam[0] * g)), amp, meas), True)
        return np.where(sup, g + beta * ((1 + gam[1]) * P - gam[1] * g), g) - beta * Pf
    out = {"er": 0 * g, "hio": g - beta * P, "raar": beta * g + (1 - 2 * beta) * P}[alg]
    return np.where(sup, P, out)


@pytest.mark.parametrize("nz,n", SHAPES)
def test_iterations_match_float64(sp, nz, n):
    shape = (nz, n, n)
    obj, amp, meas, sup, g0 = random_case(shape, seed=nz)
    a64, beta = amp.astype(np.float64), float(np.float32(0.9))
    for alg in ("hio", "dm"):
        with GpuPhaser(sp, alg, amp, meas, sup, g0, beta=0.9) as g:
            gam = g.gammas() if alg == "dm" else (0, 0)
            for _ in range(2):  # each from the engine's own iterate
                want = _step(alg, g.get("model").astype(np.complex128), a64, meas, sup, beta, gam)
                assert g.iterate(1) == 0
                assert rel(g.get("model"), want) < 1e-5
            F = _fft(g.get("model").astype(np.complex128))
            nom = ((np.abs(F) - a64)[meas] ** 2).sum()
            den = (a64[meas] ** 2).sum() + (np.abs(F[~meas]) ** 2).sum()
            assert abs(g.efourier()[0] - np.sqrt(nom / den)) < 1e-4 * np.sqrt(nom / den)
            assert rel(g.get("fmodel"), F) < 1e-5


@pytest.mark.parametrize("shape", [(64, 72, 72), (72, 64, 64), (80, 144, 144)])
def test_margins_and_phased_amplitudes(sp, shape):
    obj, amp, meas, sup, g0 = random_case(shape, seed=2)
    F = _fft(g0.astype(np.complex128))
    lo, hi = (0.9 * amp).astype(np.float32), (1.2 * amp).astype(np.float32)
    m = np.clip(np.abs(F), lo, hi) / np.abs(F)
    want = np.where(sup, _fft(np.where(meas, F * m, F), True), 0)
    with GpuPhaser(sp, "er", amp, meas, sup, g0, constraints=sp.SpAmplitudeErrorMargin) as g:
        sp.sp_phaser_set_amplitudes_margins(g.ph, g._img(lo), g._img(hi))
        assert g.iterate(1) == 0
        assert rel(g.get("model"), want) < 1e-5
    rng = np.random.default_rng(4)
    pa = (amp * np.exp(2j * np.pi * rng.random(shape))).astype(np.complex64)
    want = np.where(sup, _fft(np.where(meas, pa, F), True), 0)
    with GpuPhaser(sp, "er", amp, meas, sup, g0) as g:
        sp.sp_phaser_set_phased_amplitudes(g.ph, g._img(pa, meas))
        sp.sp_phaser_set_objective(g.ph, sp.SpRecoverAmplitudes)
        assert g.iterate(1) == 0
        assert rel(g.get("model"), want) < 1e-5


@pytest.mark.parametrize("shape", [(64, 64, 64), (64, 80, 80)])
def test_mixed_batch_with_idle_and_vacant_slots(sp, shape):
    algs, betas = ["hio", "raar", "er", "hio", "raar"], [0.9, 0.7, 0.0, 0.5, 0.8]
    pats = [random_case(shape, seed=40 + r) for r in range(5)]
    b = sp.Batch(shape, 5)
    for r, (_, a, m, s, g0) in enumerate(pats):
        b.set_data(r, a, m, s)
        b.set_model(r, g0)
    b.set_algorithm(sp.sp_phasing_hio_alloc(sp.smap([(0, 0.9)]), 0))
    ids = {"hio": sp.SpHIO, "raar": sp.SpRAAR, "er": sp.SpER}
    b.set_rec_algorithms(np.array([ids[a] for a in algs], np.int32), np.array(betas, np.float32))
    b.iterate(1)
    first = b.model()
    b.set_active([1, 0, 1, 2, 1])  # slot 1 idle, slot 3 vacant
    b.iterate(1)
    b.set_active(None)
    for r in (0, 1, 2, 4):
        _, a, m, s, g = pats[r]
        args = (a.astype(np.float64), m, s, float(np.float32(betas[r])))
        assert rel(first[r], _step(algs[r], g.astype(np.complex128), *args)) < 1e-5
        want = first[r] if r == 1 else _step(algs[r], first[r].astype(np.complex128), *args)
        assert rel(b.model(r), want) < 1e-5
        # the slot alone: the same bits
        with GpuPhaser(sp, algs[r], a, m, s, g, beta=betas[r]) as ph:
            assert ph.iterate(1 if r == 1 else 2) == 0
            assert np.array_equal(ph.get("model"), b.model(r))
    b.close()
