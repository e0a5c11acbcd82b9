"""prh_spectral_iterate_* with the result over the density, and over a source that is the density too: the bits of the
same call into a buffer of its own (the header lets out be src or delta)."""
import ctypes

import numpy as np
import pytest

from test_gpu_half_spectrum import OBLIQUE, Setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('los', [None, OBLIQUE])
@pytest.mark.parametrize('dtype', ['f4', 'f8'])
@pytest.mark.parametrize('shape', [(2, 3, 4), (15, 9, 25), (48, 40, 36)])
def test_over_the_density(shape, dtype, los):
    from pyrecon_amd import DeviceArray
    s = Setup(shape, dtype)
    lib = s._lib
    scratch = s.scratch(lib.SPECTRAL_LOCAL if los is None else lib.SPECTRAL_GLOBAL)
    bc, bc_ptr = lib.vec3(s.boxcenter, dtype)
    bs, bs_ptr = lib.vec3(s.boxsize, dtype)
    los_c = None if los is None else (ctypes.c_double * 3)(*los)
    fn = getattr(lib.lib, 'prh_spectral_iterate_' + s.sfx)

    def iterate(src, delta, out):
        lib.check(fn(s.ws.handle, src.ptr, delta.ptr, out.ptr, s.nm_ptr, bs_ptr, bc_ptr, los_c, 0.7, scratch.ptr,
                     scratch.nbytes, None))
        return out.numpy()

    src, delta, out = DeviceArray.from_numpy(s.source), DeviceArray.from_numpy(s.delta), DeviceArray(shape, dtype)
    apart = iterate(src, delta, out)
    assert np.array_equal(iterate(src, delta, delta), apart)
    delta = DeviceArray.from_numpy(s.delta)
    same = iterate(delta, delta, out)
    assert np.array_equal(iterate(delta, delta, delta), same)
