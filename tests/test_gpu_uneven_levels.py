"""Sweeps and residuals on levels that the 64-wide tiles do not cover, bit for bit against the CPU oracle
(src/multigrid.c:44-164): FP64 levels of 500 000 cells and more in tiles of any extent (one tile a row and
several, partial last tiles along each axis, few rows, few planes), FP32 ones in columns of two cells (odd
extents along x), and smaller ones a cell a thread.
"""
import numpy as np
import pytest

from test_gpu_kernels import BOX, LOS, assert_bitexact

pytestmark = pytest.mark.gpu

SHAPES = [(79, 81, 79), (80, 75, 84), (101, 64, 80), (64, 100, 96), (90, 7, 800), (9, 300, 190), (3, 420, 400),
          (400, 31, 41), (2400, 15, 14), (2, 512, 500), (25, 31, 20), (11, 9, 130), (2, 40, 40), (2, 2, 2), (5, 3, 2)]


@pytest.mark.parametrize('dtype', ['f4', 'f8'])
@pytest.mark.parametrize('shape', SHAPES)
def test_uneven_levels(gpu, oracle, dtype, shape):
    rng = np.random.RandomState(sum(shape))
    f, v = (rng.normal(size=shape).astype(dtype) for _ in range(2))
    for los in LOS[::2]:
        a, b = v.copy(), v.copy()
        oracle.jacobi(a, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, 2, los)
        gpu.jacobi(b, f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, 2, los)
        assert_bitexact(a, b, 'jacobi')
        assert_bitexact(oracle.residual(v, f, BOX['boxsize'], BOX['boxcenter'], 0.4, los),
                        gpu.residual(v, f, BOX['boxsize'], BOX['boxcenter'], 0.4, los), 'residual')


@pytest.mark.parametrize('dtype', ['f4', 'f8'])
def test_uneven_solve(gpu, oracle, dtype):
    shape = (80, 72, 88)
    f = np.random.RandomState(4).normal(size=shape).astype(dtype)
    assert_bitexact(oracle.fmg(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, 5, 6, los=None),
                    gpu.fmg(f, BOX['boxsize'], BOX['boxcenter'], 0.4, 0.4, 5, 6, los=None), 'fmg')
