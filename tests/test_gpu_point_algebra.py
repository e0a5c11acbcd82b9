"""The device's per-point algebra against the host's numpy on the same displacement meshes, bit for bit:
wrapped shifts of the FFT reconstructions (pyrecon/recon.py:255-325) and the particle reconstruction's
iteration and shifts (pyrecon/iterative_fft_particle.py:104-239), for every field, line of sight, wrap and
dtype combination, those that numpy promotes beyond the positions dtype (and that stay on the host)
included; below and above the size from which reads bin their points.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOX, CENTER = np.array([800., 600., 1000.]), np.array([0., 100., 900.])
COMBINATIONS = [(p, m, los, wrap) for p in ('f4', 'f8') for m in ('f4', 'f8')
                for los in (None, 'x', [0.3, 0.4, np.sqrt(0.75)]) for wrap in (False, True)]


def bits(array):
    return np.ascontiguousarray(array).view('u4' if array.dtype == np.float32 else 'u8')


def assert_same(a, b):
    assert a.dtype == b.dtype and a.shape == b.shape
    assert np.array_equal(bits(a), bits(b))


def points(n, dtype, wrap, seed):
    rng = np.random.RandomState(seed)
    x = rng.uniform(-0.48, 0.48, (n, 3)) * BOX + CENTER
    if wrap: x[::7] += BOX * [1., -1., 2.]
    return x.astype(dtype)


@pytest.mark.parametrize('n', [1000, 70000])
@pytest.mark.parametrize('pdtype,dtype,los,wrap', [c for c in COMBINATIONS if c[2] is not None])
def test_wrapped_shifts(pdtype, dtype, los, wrap, n):
    from pyrecon_amd import DeviceArray, PlaneParallelFFTReconstruction
    recon = PlaneParallelFFTReconstruction(f=0.8, bias=2., los=los, nmesh=(32, 24, 40), boxsize=BOX, boxcenter=CENTER,
                                           dtype=dtype, wrap=wrap)
    recon.assign_data(points(20000, pdtype, wrap, 1))
    recon.set_density_contrast(smoothing_radius=30.)
    recon.run()
    for local in (False, True):
        if local: recon.los = None  # the local line of sight on the same meshes
        x = points(n, pdtype, wrap, 2)
        for field in ('disp', 'rsd', 'disp+rsd'):
            expect = recon._host_shifts(x, field)
            moved = x - expect
            if wrap: moved = recon.info.wrap(moved)
            for given in (x, DeviceArray.from_numpy(x)):
                out = [recon.read_shifts(given, field), recon.read_shifted_positions(given, field)]
                out = [o if isinstance(o, np.ndarray) else o.numpy() for o in out]
                assert_same(out[0], expect)
                assert_same(out[1], moved)


@pytest.mark.parametrize('n', [1000, 70000])
@pytest.mark.parametrize('pdtype,dtype,los,wrap', COMBINATIONS)
def test_particle(pdtype, dtype, los, wrap, n):
    from pyrecon_amd import IterativeFFTParticleReconstruction

    def run(device):
        recon = IterativeFFTParticleReconstruction(f=0.8, bias=2., los=los, nmesh=(32, 24, 40), boxsize=BOX,
                                                   boxcenter=CENTER, dtype=dtype, wrap=wrap)
        if not device: recon._on_device = lambda dtype: False
        rng = np.random.RandomState(3)
        recon.assign_data(0.9 * (points(n, pdtype, wrap, 1) - CENTER.astype(pdtype)) + CENTER.astype(pdtype),
                          rng.uniform(0.5, 1.5, n).astype(pdtype))
        recon.set_density_contrast(smoothing_radius=30.)
        recon.run()
        x = 0.9 * (points(n, pdtype, wrap, 2) - CENTER.astype(pdtype)) + CENTER.astype(pdtype)
        out = [recon._positions_rec_data]
        for given in ('data', x):
            for field in ('disp', 'rsd', 'disp+rsd'):
                out += [recon.read_shifts(given, field), recon.read_shifted_positions(given, field)]
        return out

    for a, b in zip(run(True), run(False)): assert_same(a, b)
