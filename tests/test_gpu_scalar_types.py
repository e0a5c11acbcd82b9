"""Growth rates and biases that are numpy scalars (a cosmology's f is a numpy f8): the dtypes and bits of the
reference's numpy algebra (pyrecon/recon.py:255-325, pyrecon/iterative_fft_particle.py:104-239), which an f8
scalar takes from f4 to f8 while Python's numbers leave it in f4."""
import numpy as np
import pytest

from test_gpu_point_algebra import BOX, CENTER, assert_same, points

pytestmark = pytest.mark.gpu

SCALARS = [(np.float64(0.8), 2.), (np.float32(0.8), 2.), (0.8, np.float64(2.)), (1, 2), (np.array(0.8), 2.)]


def promoted(f):
    return np.result_type(np.float32(1.) * f)


@pytest.mark.parametrize('f,bias', SCALARS)
@pytest.mark.parametrize('los', ['x', None])
def test_wrapped_shifts(f, bias, los):
    from pyrecon_amd import IterativeFFTReconstruction
    recon = IterativeFFTReconstruction(f=f, bias=bias, los=los, nmesh=(32, 24, 40), boxsize=BOX, boxcenter=CENTER,
                                       dtype='f4', wrap=True)
    recon.assign_data(points(20000, 'f4', True, 1))
    recon.set_density_contrast(smoothing_radius=30.)
    recon.run()
    x = points(1000, 'f4', True, 2)
    for field in ('disp', 'rsd', 'disp+rsd'):
        expect = recon._host_shifts(x, field)
        assert expect.dtype == (promoted(f) if field == 'rsd' else np.float32)
        assert_same(recon.read_shifts(x, field), expect)
        assert_same(recon.read_shifted_positions(x, field), recon.info.wrap(x - expect))


@pytest.mark.parametrize('f,bias', SCALARS)
@pytest.mark.parametrize('dtype,wrap,los', [('f4', False, 'x'), ('f4', True, None), ('f8', False, None)])
def test_particle(f, bias, dtype, wrap, los):
    from pyrecon_amd import IterativeFFTParticleReconstruction

    def run(device):
        recon = IterativeFFTParticleReconstruction(f=f, bias=bias, los=los, nmesh=(32, 24, 40), boxsize=BOX,
                                                   boxcenter=CENTER, dtype=dtype, wrap=wrap)
        if not device: recon._on_device = lambda dtype: False
        center = CENTER.astype('f4')
        recon.assign_data(np.float32(0.9) * (points(5000, 'f4', wrap, 1) - center) + center)
        recon.set_density_contrast(smoothing_radius=30.)
        recon.run()
        x = np.float32(0.9) * (points(1000, 'f4', wrap, 2) - center) + center
        out = [recon._positions_rec_data]
        for given in ('data', x):
            for field in ('disp', 'rsd', 'disp+rsd'):
                out += [recon.read_shifts(given, field), recon.read_shifted_positions(given, field)]
        return out

    out = run(True)
    assert out[0].dtype == promoted(f)
    for a, b in zip(out, run(False)): assert_same(a, b)


@pytest.mark.parametrize('algorithm', ['IterativeFFT', 'IterativeFFTParticle'])
def test_own_line_of_sight(algorithm):
    """A line of sight in f8 that a program put in the place of an f4 reconstruction's: f8 shifts, as numpy has them."""
    import pyrecon_amd
    recon = getattr(pyrecon_amd, algorithm + 'Reconstruction')(f=0.8, bias=2., los='x', nmesh=(32, 24, 40), boxsize=BOX,
                                                               boxcenter=CENTER, dtype='f4', wrap=True)
    recon.los = np.array([0.3, 0.4, np.sqrt(0.75)])
    recon.assign_data(points(20000, 'f4', True, 1))
    recon.set_density_contrast(smoothing_radius=30.)
    recon.run()
    x = points(1000, 'f4', True, 2)
    for field in ('rsd', 'disp+rsd'):
        expect = recon._host_shifts(x, field)
        if field == 'rsd' or algorithm == 'IterativeFFTParticle': assert expect.dtype == np.float64
        assert_same(recon.read_shifts(x, field), expect)
        assert_same(recon.read_shifted_positions(x, field), recon.info.wrap(x - expect))
    if algorithm == 'IterativeFFTParticle': assert recon._positions_rec_data.dtype == np.float64
