"""PRTF of more reconstructions than the spectra kept at once (4 of 1024 x
1024): what a reconstruction is aligned to does not depend on where the groups
end, and the transforms over several groups add up."""
import numpy as np
import pytest

from _helpers import rel
from test_gpu_prtf import _copies

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("translate", [True, False])
def test_prtf_over_groups(translate):
    from libspimage_amd import prtf as gp
    imgs, masks = _copies((1024, 1024), 9, seed=5, reflect=translate)
    masks[8] = 0
    few = gp.prtf(imgs[:4], masks[:4], translate=translate, full_out=True)
    all_ = gp.prtf(imgs, masks, translate=translate, full_out=True)
    assert np.array_equal(all_["images"][:4], few["images"])
    assert np.array_equal(all_["masks"][:4], few["masks"])
    # the sums, in float64 from the aligned reconstructions
    a = all_["images"].astype(np.complex128)
    assert rel(all_["super_image"], a.sum(0)) < 1e-5
    F = np.fft.fftn(a, axes=(1, 2))
    assert rel(all_["prtf"], np.fft.fftshift(np.abs((F / np.abs(F)).mean(0)))) < 1e-5
    counted = masks.reshape(9, -1).sum(1) > 0
    assert np.array_equal(all_["super_mask"], ((all_["masks"] == 0) & counted[:, None, None])[1:].any(0))
