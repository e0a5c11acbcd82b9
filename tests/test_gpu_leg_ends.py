"""The last sweep with the residual and its restriction, and the correction with the first sweep, on tiles of
8^3 cells, bit for bit against the CPU oracle (src/multigrid.c:270-300): levels just above the whole legs' and
up to 64^3 cells, tiles that the level does not fill, the thinnest levels, one to six sweeps, groups of solves.
The fast FP32 forms (rows of 64 cells): a mixed solve tracks the plain FP64 one to 1e-4 of the potential's norm.
"""
import numpy as np
import pytest

from test_gpu_kernels import BOX, LOS, assert_bitexact

pytestmark = pytest.mark.gpu

SHAPES = [(28, 28, 28), (12, 44, 40), (30, 36, 38), (14, 130, 140), (62, 66, 62), (64, 64, 64), (48, 64, 56), (66, 64, 64)]


@pytest.mark.parametrize('dtype', ['f4', 'f8'])
@pytest.mark.parametrize('shape', SHAPES)
def test_leg_ends(gpu, oracle, dtype, shape):
    rng = np.random.RandomState(sum(shape))
    f, v = (rng.normal(size=shape).astype(dtype) for _ in range(2))
    for los in LOS[::2]:
        for niter in (1, 2, 3, 6):
            a, b = v.copy(), v.copy()
            oracle.vcycle(a, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, los)
            gpu.vcycle(b, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, los)
            assert_bitexact(a, b, 'vcycle')
    # zero starts below a finer level
    f = rng.normal(size=2 * np.array((28, 30, 26))).astype(dtype)
    for niter in (1, 2):
        assert_bitexact(oracle.fmg(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, 2, los=None),
                        gpu.fmg(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, 2, los=None), 'fmg')


@pytest.mark.parametrize('shape', [(16, 32, 64), (64, 64, 64), (32, 64, 128), (28, 28, 28)])
def test_fast_leg_ends(gpu, shape):
    f = np.random.RandomState(sum(shape)).normal(size=shape)
    f -= f.mean()
    for los in LOS[::2]:
        for niter in (1, 2, 5):
            a = gpu.fmg(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, 2, los=los)
            b, _ = gpu.fmg_mixed(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, 2, los=los)
            a, b = a - a.mean(), b - b.mean()
            assert np.linalg.norm(a - b) < 1e-4 * np.linalg.norm(a)


@pytest.mark.parametrize('precision', ['plain', 'mixed'])
def test_group_of_leg_ends(precision):
    from pyrecon_amd import MultiGridReconstruction, run_group
    shape = (32, 32, 64)

    def make(i):
        recon = MultiGridReconstruction(f=0.8, bias=2., los=[None, 'x', None][i], nmesh=shape, boxsize=8. * np.array(shape),
                                        boxcenter=(0., 10. * i, 500.), precision=precision)
        recon.mesh_delta = recon.mesh_data.__class__(info=recon.info, workspace=recon.workspace)
        recon.mesh_delta.value = np.random.RandomState(i).normal(size=shape)
        return recon

    group = [make(i) for i in range(3)]
    run_group(group, precision=precision)
    for i, recon in enumerate(group):
        alone = make(i)
        alone.run()
        assert_bitexact(alone.mesh_phi.value, recon.mesh_phi.value, 'job {:d}'.format(i))
