"""The residual and its restriction in one launch, bit for bit against the CPU oracle (src/multigrid.c:44-262):
FP64 and FP32 levels in 64-wide tiles, FP32 whole rows with a global line of sight; one tile along y or z, the
shortest run of planes, several runs with a shorter last one, planes no multiple of 16 rows (separate launches).
The fast FP32 forms: a mixed solve tracks the plain FP64 one to 1e-4 of the potential's norm.
"""
import numpy as np
import pytest

from test_gpu_kernels import BOX, LOS, assert_bitexact

pytestmark = pytest.mark.gpu

SHAPES = [(6, 112, 448), (270, 16, 64), (18, 64, 256), (30, 48, 192), (10, 64, 512), (84, 32, 128), (38, 80, 320),
          (30, 56, 192), (6, 48, 1024)]


@pytest.mark.parametrize('dtype', ['f4', 'f8'])
@pytest.mark.parametrize('shape', SHAPES)
def test_residual_restrict(gpu, oracle, dtype, shape):
    rng = np.random.RandomState(sum(shape))
    f, v = (rng.normal(size=shape).astype(dtype) for _ in range(2))
    for los in LOS[::2]:
        for niter in (1, 3):
            a, b = v.copy(), v.copy()
            oracle.vcycle(a, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, los)
            gpu.vcycle(b, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, los)
            assert_bitexact(a, b, 'vcycle')


@pytest.mark.parametrize('shape', SHAPES)
def test_fast_residual_restrict(gpu, shape):
    f = np.random.RandomState(sum(shape)).normal(size=shape)
    f -= f.mean()
    for los in LOS[::2]:
        a = gpu.fmg(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, 5, 2, los=los)
        b, _ = gpu.fmg_mixed(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, 5, 2, los=los)
        a, b = a - a.mean(), b - b.mean()
        assert np.linalg.norm(a - b) < 1e-4 * np.linalg.norm(a)
