"""The area update's blur and select on sizes that are and are not whole
vectors of pixels, for one and several reconstructions, on either axis order,
and on models without a usable ranking, against the blur in float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIGMA, AREA = 2.0, 0.07


def _blur64(m):
    r2 = 0.0
    for ax, n in enumerate(m.shape):
        k = np.fft.fftfreq(n, 1.0 / n) / m.shape[-1]
        r2 = r2 + (k ** 2).reshape([-1 if a == ax else 1 for a in range(m.ndim)])
    return np.abs(np.fft.ifftn(np.fft.fftn(np.abs(m).astype(np.float64)) * np.exp(-2 * np.pi ** 2 * SIGMA ** 2 * r2)))


def _updated(sp, models):
    n, shape = len(models), models.shape[1:]
    b = sp.Batch(shape, n)
    try:
        keep = [sp.smap([(0, SIGMA)]), sp.smap([(0, AREA)])]
        ones = np.ones(models.shape)
        b.set_data(-1, ones.astype(np.float32), ones.astype(bool), np.zeros(models.shape, bool))
        b.set_algorithm(sp.sp_phasing_er_alloc(sp.SpNoConstraints))
        b.set_model(-1, models)
        b.set_support_schedule(sp.sp_support_array_init(sp.sp_support_area_alloc(*keep), 1))
        b.iterate(1)  # period 1: the update, no phasing
        return b.support(), b.support_fraction()
    finally:
        b.close()


@pytest.mark.parametrize("nrec", [1, 3])
@pytest.mark.parametrize("shape", [(16, 16), (45, 63), (30, 42), (2, 8), (512, 500), (1024, 1024), (24, 1, 36),
                                   (14, 18, 20), (64, 64, 64)])
def test_area_update(sp, shape, nrec):
    rng = np.random.default_rng(3)
    models = (rng.random((nrec,) + shape) + 1j * rng.random((nrec,) + shape)).astype(np.complex64)
    sup, fraction = _updated(sp, models)
    N = models[0].size
    k = int(np.float32(N) * np.float32(AREA))
    for r in range(nrec):
        b = _blur64(models[r])
        t = np.sort(b.ravel())[::-1][k]
        # float32 transforms are off by some eps log2 N of the largest value
        clear = np.abs(b - t) > 2e-6 * b.max()
        assert np.array_equal((sup[r] & 1).astype(bool)[clear], (b > t)[clear])
        count = int((sup[r] & 1).sum())
        assert k - 3 <= count <= k  # equal values at the threshold stay outside
        assert fraction[r] == np.float32(count) / np.float32(N)


@pytest.mark.parametrize("value", [0.0, np.nan])
def test_area_update_without_ranking(sp, value):
    sup, fraction = _updated(sp, np.full((2, 32, 32), value, np.complex64))
    assert not (sup & 1).any() and not np.any(fraction)
