"""Half-spectrum calls of the FFT reconstructions (prh_spectral_iterate_*, prh_spectral_displacements_*)
against numpy's c2c transforms in float64, as pyrecon/iterative_fft.py:30-82 and
pyrecon/plane_parallel_fft.py:41-55 use them.

White noise, so that the Nyquist planes, whose c2c result is not Hermitian, carry their share; even and
odd axes; every radix (2 to 8 and 10), the longest line of each axis and several slabs.  Bounds: a
transform's relative rounding grows with the square root of its number of passes, a few eps in all
(FP64 2e-16, FP32 1.2e-7): 1e-13 and 2e-6, those of the c2c transforms' own tests.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(2, 3, 4), (8, 7, 10), (16, 16, 16), (12, 14, 20), (15, 9, 25), (9, 12, 21), (20, 15, 18), (48, 40, 36), (49, 50, 27),
          (1024, 9, 10), (12, 1024, 9), (9, 10, 1024), (10, 9, 875), (64, 256, 224)]
TOL = {'f4': 2e-6, 'f8': 1e-13}


def rel_l2(a, b):
    # (an axis of two cells has no displacement at all: both sides are zero)
    return np.sqrt(np.sum((np.asarray(a, 'f8') - b)**2) / max(np.sum(np.asarray(b, 'f8')**2), 1e-300))


class Setup(object):

    def __init__(self, shape, dtype):
        from pyrecon_amd import DeviceArray, Workspace, _lib
        self._lib, self.shape, self.dtype = _lib, shape, dtype
        self.boxsize = np.array([7., 6., 8.], dtype=dtype) * np.array(shape, dtype=dtype)
        self.boxcenter = np.array([50., -30., 900.], dtype=dtype)
        rng = np.random.RandomState(sum(shape))
        self.delta = rng.normal(size=shape).astype(dtype)
        self.source = rng.normal(size=shape).astype(dtype)
        self.ws = Workspace(shape, dtype, flags=_lib.WS_FFT)
        self.sfx = 'f32' if dtype == 'f4' else 'f64'
        self.nm, self.nm_ptr = _lib.size3(shape)
        k = [2 * np.pi * np.fft.fftfreq(n, d=float(b) / n) for n, b in zip(shape, self.boxsize)]
        self.k = np.meshgrid(*k, indexing='ij')
        self.k2 = sum(kk**2 for kk in self.k)
        self.k2[0, 0, 0] = 1.

    def over_k2(self, mesh):
        spectrum = np.fft.fftn(mesh.astype('f8')) / self.k2
        spectrum[0, 0, 0] = 0.
        return spectrum

    def scratch(self, kind):
        from pyrecon_amd import DeviceArray
        nbytes = ctypes.c_size_t()
        self._lib.check(self._lib.lib.prh_spectral_scratch(self.nm_ptr, self._lib.dtype_code(self.dtype), kind,
                                                           ctypes.byref(nbytes)))
        assert nbytes.value > 0
        return DeviceArray((nbytes.value,), np.uint8)

    def iterate(self, los, factor, in_place):
        from pyrecon_amd import DeviceArray
        scratch = self.scratch(self._lib.SPECTRAL_LOCAL if los is None else self._lib.SPECTRAL_GLOBAL)
        src, delta = DeviceArray.from_numpy(self.source), DeviceArray.from_numpy(self.delta)
        out = src if in_place else DeviceArray(self.shape, self.dtype)
        los_c = None if los is None else (ctypes.c_double * 3)(*los)
        bc, bc_ptr = self._lib.vec3(self.boxcenter, self.dtype)
        bs, bs_ptr = self._lib.vec3(self.boxsize, self.dtype)
        fn = getattr(self._lib.lib, 'prh_spectral_iterate_' + self.sfx)
        args = lambda nscratch: (self.ws.handle, src.ptr, delta.ptr, out.ptr, self.nm_ptr, bs_ptr, bc_ptr, los_c, factor,
                                 scratch.ptr, nscratch, None)
        assert fn(*args(scratch.nbytes - 1)) == self._lib.ERR_CAPACITY
        self._lib.check(fn(*args(scratch.nbytes)))
        return out.numpy()

    def displacements(self, los, beta):
        from pyrecon_amd import DeviceArray
        scratch = self.scratch(self._lib.SPECTRAL_DISPLACEMENTS)
        delta = DeviceArray.from_numpy(self.delta)
        psis = [DeviceArray(self.shape, self.dtype) for _ in range(3)]
        los_c = None if los is None else (ctypes.c_double * 3)(*los)
        bs, bs_ptr = self._lib.vec3(self.boxsize, self.dtype)
        fn = getattr(self._lib.lib, 'prh_spectral_displacements_' + self.sfx)
        self._lib.check(fn(self.ws.handle, delta.ptr, *[p.ptr for p in psis], self.nm_ptr, bs_ptr, los_c, beta,
                           scratch.ptr, scratch.nbytes, None))
        assert np.array_equal(delta.numpy(), self.delta)
        return [p.numpy() for p in psis]


OBLIQUE = np.array([0.3, 0.4, np.sqrt(0.75)])


@pytest.mark.parametrize('dtype', ['f4', 'f8'])
@pytest.mark.parametrize('shape', SHAPES)
def test_half_spectrum(shape, dtype):
    s = Setup(shape, dtype)
    factor, beta = 0.7, 0.4
    spectrum = s.over_k2(s.source)
    # local line of sight
    offset = (s.boxcenter - s.boxsize / s.boxsize.dtype.type(2)).astype('f8')
    x = np.meshgrid(*[o + float(b) / n * np.arange(n) for o, b, n in zip(offset, s.boxsize, shape)], indexing='ij')
    x2 = sum(xx**2 for xx in x)
    expect = s.delta.astype('f8')
    for a in range(3):
        for b in range(3):
            expect -= factor * x[a] * x[b] / x2 * np.fft.ifftn(s.k[a] * s.k[b] * spectrum).real
    for in_place in (False, True):
        assert rel_l2(s.iterate(None, factor, in_place), expect) < TOL[dtype]
    # global lines of sight, along an axis and not
    for los in (np.array([0., 0., 1.]), OBLIQUE):
        kl = sum(kk * ll for kk, ll in zip(s.k, los))
        expect = s.delta.astype('f8') - factor * np.fft.ifftn(kl**2 * spectrum).real
        assert rel_l2(s.iterate(los, factor, True), expect) < TOL[dtype]
        den = 1. + beta * kl**2 / s.k2
        for psi, kk in zip(s.displacements(los, beta), s.k):
            assert rel_l2(psi, np.fft.ifftn(1j * kk * s.over_k2(s.delta) / den).real) < TOL[dtype]
    for psi, kk in zip(s.displacements(None, 0.), s.k):
        assert rel_l2(psi, np.fft.ifftn(1j * kk * s.over_k2(s.delta)).real) < TOL[dtype]


@pytest.mark.parametrize('shape', [(16, 22, 16), (16, 16, 1250), (16, 16, 13)])
def test_shapes_left_to_c2c(shape):
    """A prime factor above 7, too long a line: no scratch size, and the classes still run."""
    from pyrecon_amd import IterativeFFTReconstruction, _lib
    nm, nm_ptr = _lib.size3(shape)
    nbytes = ctypes.c_size_t(1)
    _lib.check(_lib.lib.prh_spectral_scratch(nm_ptr, _lib.F64, _lib.SPECTRAL_LOCAL, ctypes.byref(nbytes)))
    assert nbytes.value == 0
    recon = IterativeFFTReconstruction(f=0.8, bias=2., los='x', nmesh=shape, boxsize=10. * np.array(shape),
                                       boxcenter=(0., 0., 0.))
    rng = np.random.RandomState(3)
    positions = rng.uniform(-0.5, 0.5, (2000, 3)) * 10. * np.array(shape)
    recon.assign_data(positions)
    recon.set_density_contrast(smoothing_radius=15.)
    recon.run()
    assert np.isfinite(recon.read_shifted_positions(positions)).all()
