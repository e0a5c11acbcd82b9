"""Grouped multigrid solves over the sizes where a group's levels change kernels, against the same problems solved alone,
bit for bit: levels whose legs, one-workgroup launches or launches for the whole group depend on the number of problems
(12^3, 14 x 12 x 16, 16^3, 20^3, 24^3, 20 x 24 x 28), below and above each limit."""
import numpy as np
import pytest

from test_gpu_group import JOBS, bits, solve_alone, solve_group, sources

pytestmark = pytest.mark.gpu

SHAPES = [((48, 48, 48), (2, 4, 5)), ((56, 48, 64), (2, 4, 8)), ((32, 32, 32), (4, 8)), ((40, 40, 40), (2, 3, 5)),
          ((20, 24, 28), (2, 3, 8))]


def check_group(shape, count, dtype, mixed):
    jobs = (JOBS * 3)[:count]
    fs = sources(shape, dtype, count, seed=count)
    for f, job, group in zip(fs, jobs, solve_group(fs, jobs, dtype, mixed=mixed)):
        assert np.array_equal(bits(group), bits(solve_alone(f, job, dtype, mixed=mixed)))


@pytest.mark.parametrize('dtype,mixed', [('f4', False), ('f8', False), ('f8', True)])
@pytest.mark.parametrize('shape,count', [(shape, count) for shape, counts in SHAPES for count in counts])
def test_equals_alone(shape, count, dtype, mixed):
    check_group(shape, count, dtype, mixed)


@pytest.mark.parametrize('dtype,mixed', [('f4', False), ('f8', False), ('f8', True)])
@pytest.mark.parametrize('shape', [(80, 96, 112), (96, 112, 116), (96, 112, 120), (96, 128, 120), (96, 128, 124)])
def test_finest_level_equals_alone(shape, dtype, mixed):
    """Meshes of 860 160 cells to 1 523 712, on both sides of where the finest level of a group is no longer relaxed in
    one launch for it (1.25 million cells in FP64, 1.5 in FP32)."""
    check_group(shape, 2, dtype, mixed)


@pytest.mark.parametrize('dtype,mixed', [('f4', False), ('f8', False), ('f8', True)])
@pytest.mark.parametrize('shape', [(16, 96, 192), (32, 128, 120), (32, 128, 128)])
def test_residual_restriction_equals_alone(shape, dtype, mixed):
    """Levels in 64-wide tiles and not, below and above the size from which a group's residuals are restricted at once."""
    check_group(shape, 2, dtype, mixed)
