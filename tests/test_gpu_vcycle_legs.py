"""V-cycles and full multigrid through the leg kernels and the single-workgroup levels, bit for bit against
the CPU oracle (src/multigrid.c:270-328): levels from the smallest extent the legs take to the largest
size, tiles that the level does not fill, levels just outside (too thin, too large, an odd coarser level),
one to six sweeps, a given iterate and a zero one, groups of solves.
"""
import numpy as np
import pytest

from test_gpu_kernels import BOX, LOS, assert_bitexact

pytestmark = pytest.mark.gpu

SHAPES = [(12, 12, 12), (12, 14, 18), (16, 16, 16), (20, 28, 26), (26, 26, 28), (28, 26, 28), (10, 16, 16), (12, 40, 40),
          (54, 18, 20), (32, 32, 32), (8, 12, 64), (16, 16, 2), (24, 24, 36), (14, 48, 96)]


@pytest.mark.parametrize('dtype', ['f4', 'f8'])
@pytest.mark.parametrize('shape', SHAPES)
def test_vcycle_legs(gpu, oracle, dtype, shape):
    rng = np.random.RandomState(sum(shape))
    f, v = (rng.normal(size=shape).astype(dtype) for _ in range(2))
    for los in LOS[::2]:
        for niter in (1, 2, 5, 6):
            a, b = v.copy(), v.copy()
            oracle.vcycle(a, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, los)
            gpu.vcycle(b, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, los)
            assert_bitexact(a, b, 'vcycle')
        assert_bitexact(oracle.fmg(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, 5, 2, los=los),
                        gpu.fmg(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, 5, 2, los=los), 'fmg')


@pytest.mark.parametrize('precision', ['plain', 'mixed'])
def test_group_of_legs(precision):
    # jobs with different sources, and local and global lines of sight in one group
    from pyrecon_amd import MultiGridReconstruction, run_group
    shape = (24, 32, 28)

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
