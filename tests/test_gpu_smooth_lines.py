"""Gaussian smoothing over the line transforms of prh_fft.hpp at the edges of their tiles, against numpy's
c2c transform in float64 (pyrecon/mesh.py:655-680).

Partial tiles (rows not a multiple of 16 or 32 cells), odd rows (pairs not aligned, a last line alone), an
odd number of rows, lines long enough for 64-byte tile rows, single-pass lengths, and a mesh that does not
start on a 16-byte boundary.  The bounds are those of test_smooth_gaussian.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(8, 10, 7), (15, 20, 33), (16, 18, 34), (9, 5, 512), (512, 6, 18), (12, 512, 10), (1000, 2, 9), (3, 1000, 8),
          (4, 3, 1000), (1024, 2, 16), (2, 1024, 10), (5, 7, 1024), (972, 3, 4), (48, 96, 192), (2, 3, 2)]


@pytest.mark.parametrize('dtype', ['f4', 'f8'])
@pytest.mark.parametrize('shape', SHAPES)
def test_smooth_lines(shape, dtype):
    from pyrecon_amd import DeviceArray, MeshInfo, RealMesh
    rng = np.random.RandomState(sum(shape))
    boxsize, radius = 9. * np.array(shape), 12.
    value = rng.uniform(0., 3., shape).astype(dtype)
    gain = 1.
    for d, (n, b) in enumerate(zip(shape, boxsize)):
        g = np.exp(-0.5 * (radius * 2. * np.pi * np.fft.fftfreq(n, d=b / n))**2)
        gain = gain * g.reshape([-1 if i == d else 1 for i in range(3)])
    expect = np.fft.ifftn(np.fft.fftn(value.astype('f8')) * gain).real
    info = MeshInfo(nmesh=shape, boxsize=boxsize, boxcenter=0., dtype=dtype)
    # the mesh in a buffer of its own, and one element into a larger one
    padded = DeviceArray.from_numpy(np.concatenate([value.ravel()[:1], value.ravel()]))
    for buffer in (DeviceArray.from_numpy(value), padded.rows(1, value.size + 1)):
        mesh = RealMesh(info=info)
        mesh.value = buffer
        mesh.smooth_gaussian(radius)
        got = mesh.value.astype('f8')
        assert np.sqrt(np.sum((got - expect)**2) / np.sum(expect**2)) < (1e-13 if dtype == 'f8' else 2e-6)
