"""Uploads of one thread while another captures its iterations into graphs:
both succeed, and the captured iterations give what they give alone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE, NREC, CAPTURES = (64, 64), 2, 150


def _captured_runs(sp):
    """Models of a batch whose beta changes before every call, so that every
    call captures its iterations anew, right behind an upload."""
    rng = np.random.default_rng(5)
    start = rng.random((NREC,) + SHAPE).astype(np.complex64)
    amp = np.abs(np.fft.fft2(start)).astype(np.float32)
    b = sp.Batch(SHAPE, NREC)
    out = []
    try:
        b.use_graphs(True)
        for k in range(CAPTURES):
            b.set_model(-1, start)
            b.set_data(-1, amp, np.ones(amp.shape, np.int32), (start.real > 0.5).astype(np.float32))
            b.set_algorithm(sp.sp_phasing_hio_alloc(sp.smap([(0, 0.5 + 0.002 * k)]), sp.SpNoConstraints))
            b.iterate(4)
            out.append(b.model())
    finally:
        b.close()
    return np.array(out)


def test_uploads_beside_captures(sp):
    alone = _captured_runs(sp)
    stop = threading.Event()
    errors, sent = [], []

    def upload(seed):
        a = np.random.default_rng(seed).random((128, 128)).astype(np.float32)
        b = sp.Batch((128, 128), 1)
        try:
            while not stop.is_set():
                b.set_data(0, a, np.ones(a.shape, np.int32), a > 0.5)
                sent.append(np.array_equal(b.support(0) != 0, a > 0.5))
        except RuntimeError as e:
            errors.append(e)
        finally:
            b.close()

    threads = [threading.Thread(target=upload, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    try:
        beside = _captured_runs(sp)
    finally:
        stop.set()
        for t in threads:
            t.join()
    assert not errors and sent and all(sent)
    assert np.array_equal(beside, alone)
