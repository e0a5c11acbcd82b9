"""Displacement meshes that a program puts in the place of an FFT reconstruction's own, of another shape, box or
dtype: each is read by its own geometry (prh_shift_algebra_* or numpy's algebra after), bit for bit the reads of
the single meshes and the reference's numpy (pyrecon/recon.py:255-325, pyrecon/iterative_fft_particle.py:141-239).
"""
import numpy as np
import pytest

from test_gpu_point_algebra import BOX, CENTER, assert_same, points

pytestmark = pytest.mark.gpu

# coarser, finer, of the other dtype, in a larger box, the three unlike each other
KINDS = ['coarse', 'fine', 'dtype', 'box', 'mixed']


def replaced(recon, kind):
    from pyrecon_amd import RealMesh
    meshes = []
    for axis in range(3):
        nmesh, boxsize, dtype = np.array(recon.info.shape), recon.info.boxsize, recon.info.dtype
        this = KINDS[axis] if kind == 'mixed' else kind
        if this == 'coarse': nmesh = nmesh // 2
        if this == 'fine': nmesh = nmesh + 7
        if this == 'dtype': dtype = 'f4' if dtype == np.float64 else 'f8'
        if this == 'box': boxsize = 1.25 * boxsize
        mesh = RealMesh(nmesh=nmesh, boxsize=boxsize, boxcenter=recon.info.boxcenter, dtype=dtype)
        mesh.value = np.random.RandomState(axis).normal(size=tuple(nmesh))
        meshes.append(mesh)
    return meshes


@pytest.mark.parametrize('kind', KINDS)
@pytest.mark.parametrize('wrap,los', [(False, None), (False, 'x'), (True, 'x')])
@pytest.mark.parametrize('dtype', ['f4', 'f8'])
@pytest.mark.parametrize('algorithm', ['iterative', 'particle'])
def test_replaced_meshes(algorithm, dtype, wrap, los, kind):
    from pyrecon_amd import DeviceArray, IterativeFFTReconstruction, IterativeFFTParticleReconstruction
    cls = IterativeFFTReconstruction if algorithm == 'iterative' else IterativeFFTParticleReconstruction
    recon = cls(f=0.8, bias=2., los=los, nmesh=(32, 24, 40), boxsize=BOX, boxcenter=CENTER, dtype=dtype, wrap=wrap)
    recon.assign_data(0.9 * (points(5000, 'f8', False, 1) - CENTER) + CENTER)
    recon.set_density_contrast(smoothing_radius=30.)
    recon.run()
    recon.mesh_psi = replaced(recon, kind)
    x = 0.9 * (points(3000, 'f8', wrap, 2) - CENTER) + CENTER
    for field in ('disp', 'rsd', 'disp+rsd'):
        expect = recon._host_shifts(x, field)
        moved = x - expect
        if wrap: moved = recon.info.wrap(moved)
        for given in (x, DeviceArray.from_numpy(x)):
            out = [recon.read_shifts(given, field), recon.read_shifted_positions(given, field)]
            out = [o if isinstance(o, np.ndarray) else o.numpy() for o in out]
            assert_same(out[0], expect)
            assert_same(out[1], moved)
    if algorithm == 'particle':
        where = recon._positions_rec_data
        expect = np.stack([psi.read_cic(where, wrap=True) for psi in recon.mesh_psi], axis=-1)
        assert_same(recon.read_shifts('data', 'disp'), expect)
        expect = recon._positions_data - (expect + (recon._positions_data - where))
        if wrap: expect = recon.info.wrap(expect)
        assert_same(recon.read_shifted_positions('data'), expect)
