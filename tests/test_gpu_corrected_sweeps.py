"""The coarser level's correction added inside the first sweep that follows it, bit for bit against the CPU
oracle (src/multigrid.c:270-300): FP64 levels in 64-wide tiles, FP32 ones in whole rows of 64, 128, 256 and
512 cells and in tiles, runs of planes of odd length, the fewest planes and rows, one sweep (the correction
by itself) and several.  The fast FP32 forms: a mixed solve tracks the plain FP64 one to FP32 rounding, 1e-4
of the potential's norm for sources of unit variance (a misplaced correction costs 1e-1).
"""
import numpy as np
import pytest

from test_gpu_kernels import BOX, LOS, assert_bitexact

pytestmark = pytest.mark.gpu

SHAPES = [(6, 136, 384), (68, 72, 64), (130, 40, 64), (34, 64, 128), (22, 56, 256), (10, 64, 512), (30, 56, 192),
          (6, 48, 1024), (10, 2048, 64), (120, 8, 320)]


@pytest.mark.parametrize('dtype', ['f4', 'f8'])
@pytest.mark.parametrize('shape', SHAPES)
def test_corrected_sweeps(gpu, oracle, dtype, shape):
    rng = np.random.RandomState(sum(shape))
    f, v = (rng.normal(size=shape).astype(dtype) for _ in range(2))
    for los in LOS[::2]:
        for niter in (1, 2, 3):
            a, b = v.copy(), v.copy()
            oracle.vcycle(a, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, los)
            gpu.vcycle(b, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, los)
            assert_bitexact(a, b, 'vcycle')


@pytest.mark.parametrize('shape', SHAPES)
def test_corrected_fast_sweeps(gpu, shape):
    f = np.random.RandomState(sum(shape)).normal(size=shape)
    f -= f.mean()
    for los in LOS[::2]:
        for niter in (2, 5):
            a = gpu.fmg(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, 2, los=los)
            b, _ = gpu.fmg_mixed(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, niter, 2, los=los)
            a, b = a - a.mean(), b - b.mean()
            assert np.linalg.norm(a - b) < 1e-4 * np.linalg.norm(a)
