"""A model set on a phaser is in its device array when the call returns, also
behind queued iterations: a program that holds the array reads it on streams of
its own."""
import ctypes as C

import numpy as np
import pytest
import torch

from _helpers import GpuPhaser, random_case

pytestmark = pytest.mark.gpu


class _Array:
    def __init__(self, address, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<c8", "data": (address, False), "version": 3}


# on both sides of 16 MiB, up to which uploads pass through pinned memory
@pytest.mark.parametrize("shape", [(64, 64), (1024, 1024), (1536, 1536), (61, 67), (64, 64, 64)])
def test_model_is_in_the_device_array(sp, shape):
    _, amp, meas, sup, g0 = random_case(shape, seed=2)
    with GpuPhaser(sp, "hio", amp, meas, sup, g0) as g:
        for k in range(3):
            assert g.iterate(400) == 0
            model = np.roll(g0, k + 1, axis=0)
            sp.sp_phaser_set_model(g.ph, g._img(model))
            g1 = C.c_void_p()
            assert sp.spx_phaser_device_arrays(g.ph, C.byref(g1), None, None) == 0
            got = torch.as_tensor(_Array(g1.value, shape), device="cuda").cpu().numpy()
            assert np.array_equal(got, model)
