"""V-cycles of levels that one workgroup takes whole, bit for bit against the CPU oracle (src/multigrid.c:270-300):
1025 to 4096 cells whose columns along x are too many for the workgroup's threads, so that they run along y or z, or
have no thread each."""
import numpy as np
import pytest

from test_gpu_kernels import BOX, LOS, assert_bitexact

pytestmark = pytest.mark.gpu

ALONG_X = [(16, 16, 16), (12, 12, 14), (10, 20, 20)]
ALONG_Y = [(10, 80, 5), (10, 48, 8), (7, 80, 7), (3, 32, 40), (5, 28, 28)]
ALONG_Z = [(7, 14, 40), (14, 14, 20), (3, 3, 448), (2, 2, 640)]
NEITHER = [(10, 14, 29), (15, 15, 18)]


@pytest.mark.parametrize('dtype', ['f4', 'f8'])
@pytest.mark.parametrize('shape', ALONG_X + ALONG_Y + ALONG_Z + NEITHER)
def test_vcycle(gpu, oracle, dtype, shape):
    rng = np.random.RandomState(sum(shape))
    f, v = (rng.normal(size=shape).astype(dtype) for _ in range(2))
    for los in LOS:
        for niter in (1, 5):
            a, b = v.copy(), v.copy()
            oracle.vcycle(a, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, los)
            gpu.vcycle(b, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, los)
            assert_bitexact(a, b, 'vcycle')
