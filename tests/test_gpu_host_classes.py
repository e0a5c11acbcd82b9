"""Host positions of a class of their own (masked arrays, host tensors) given to the FFT reconstructions: shifted
positions are numpy's difference with them (pyrecon/recon.py:304-325, pyrecon/iterative_fft_particle.py:214-239) and
keep their class, with the values, bit for bit, of plain arrays."""
import numpy as np
import pytest

from test_gpu_point_algebra import BOX, CENTER, assert_same, points

pytestmark = pytest.mark.gpu


@pytest.mark.filterwarnings('ignore:__array_wrap__')
@pytest.mark.parametrize('algorithm,wrap', [('PlaneParallelFFT', True), ('IterativeFFT', True), ('IterativeFFTParticle', True),
                                            ('IterativeFFTParticle', False)])
def test_class_kept(algorithm, wrap):
    import torch
    import pyrecon_amd
    recon = getattr(pyrecon_amd, algorithm + 'Reconstruction')(f=0.8, bias=2., los='z', nmesh=(32, 24, 40), boxsize=BOX,
                                                               boxcenter=CENTER, wrap=wrap)
    inside = lambda n, seed: 0.9 * (points(n, 'f8', wrap, seed) - CENTER) + CENTER
    recon.assign_data(inside(5000, 1))
    recon.set_density_contrast(smoothing_radius=30.)
    recon.run()
    x = inside(1000, 2)
    masked = np.ma.masked_array(x, mask=np.zeros(x.shape, dtype=bool))
    masked.mask[::5] = True
    for field in ('disp', 'rsd', 'disp+rsd'):
        expect = recon.read_shifted_positions(x, field)
        out = recon.read_shifted_positions(torch.from_numpy(x), field)
        assert isinstance(out, torch.Tensor)
        assert_same(out.numpy(), expect)
        out = recon.read_shifted_positions(masked, field)
        assert isinstance(out, np.ma.MaskedArray) and np.array_equal(out.mask, masked.mask)
        assert_same(out.data[~out.mask], expect[~out.mask])
        for given in (torch.from_numpy(x), masked):
            assert type(recon.read_shifts(given, field)) is np.ndarray
