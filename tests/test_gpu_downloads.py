"""Arrays come back from the device as they went there on both sides of 4 MiB
(up to which they pass through one of 4 pinned blocks), also with more threads
downloading at once than there are blocks."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(16, 16), (512, 1024), (512, 1050)])
@pytest.mark.parametrize("threads", [1, 7])
def test_models_return_unchanged(sp, shape, threads):
    good = []

    def work(k):
        rng = np.random.default_rng(k)
        b = sp.Batch(shape, 1)
        try:
            for n in range(5):
                m = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)
                b.set_model(0, m)
                if np.array_equal(b.model()[0], m):
                    good.append((k, n))
        finally:
            b.close()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert sorted(good) == [(k, n) for k in range(threads) for n in range(5)]
