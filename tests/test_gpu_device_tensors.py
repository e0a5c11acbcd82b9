"""Device tensors (objects with data_ptr() and is_cuda, as torch's) given to the FFT reconstructions, periodic or
not: the shifts of the same positions as numpy arrays, bit for bit, and the same catalogs assigned."""
import numpy as np
import pytest

from test_gpu_point_algebra import BOX, CENTER, assert_same, points

pytestmark = pytest.mark.gpu


class Tensor(object):
    """What the package uses of a device tensor; like torch's, it has no numpy form."""
    is_cuda = True

    def __init__(self, array):
        from pyrecon_amd import DeviceArray
        self.array = DeviceArray.from_numpy(array)
        self.shape, self.dtype, self.ndim = self.array.shape, 'torch.' + self.array.dtype.name, self.array.ndim

    def __len__(self):
        return self.shape[0]

    def data_ptr(self):
        return self.array.ptr

    def is_contiguous(self):
        return True

    def __array__(self, dtype=None, copy=None):
        raise TypeError("can't convert cuda device type tensor to numpy")


@pytest.mark.parametrize('wrap', [False, True])
@pytest.mark.parametrize('dtype,pdtype', [('f8', 'f8'), ('f4', 'f4'), ('f8', 'f4')])
@pytest.mark.parametrize('algorithm', ['IterativeFFT', 'PlaneParallelFFT', 'IterativeFFTParticle'])
def test_same_as_numpy(algorithm, dtype, pdtype, wrap):
    import pyrecon_amd
    center = CENTER.astype(pdtype)
    inside = lambda n, seed: (0.9 * (points(n, pdtype, wrap, seed) - center) + center).astype(pdtype)
    data, x, weights = inside(5000, 1), inside(1000, 2), np.random.RandomState(3).uniform(0.5, 1.5, 5000).astype(pdtype)

    def run(given):
        recon = getattr(pyrecon_amd, algorithm + 'Reconstruction')(f=0.8, bias=2., los='z', nmesh=(32, 24, 40), boxsize=BOX,
                                                                   boxcenter=CENTER, dtype=dtype, wrap=wrap)
        recon.assign_data(given(data), given(weights))
        recon.set_density_contrast(smoothing_radius=30.)
        recon.run()
        out = []
        for field in ('disp', 'rsd', 'disp+rsd'):
            out += [recon.read_shifts(given(x), field), recon.read_shifted_positions(given(x), field)]
        if wrap or algorithm == 'IterativeFFTParticle': assert all(isinstance(o, np.ndarray) for o in out)
        return [o if isinstance(o, np.ndarray) else o.numpy() for o in out]

    for a, b in zip(run(Tensor), run(np.asarray)): assert_same(a, b)
