"""The composite residual's march over a refined rectangle and its layers of
coarse-fine cells, through the projection that it decides the convergence of,
against the oracle's direct solve at the tolerances of the projection's own
tests: rows of more lanes than a wave, several chunks of planes, a single
coarse cell between the rectangle and its periodic image, rectangles that
meet a seam without spanning it, and ones of two coarse cells."""
import pytest

from maestro_amd import workloads as W

from . import test_gpu_ml as M

pytestmark = pytest.mark.gpu

P, WALL, OUT = W.PERIODIC, W.SLIP_WALL, W.OUTLET


@pytest.mark.parametrize("dim,n,bc,lo,hi", [
    (2, 72, [[P, P], [WALL, OUT]], [0, 32], [129, 103]),
    (2, 72, [[WALL, OUT], [P, P]], [2, 0], [143, 143]),
    (2, 16, [[P, P], [P, P]], [2, 2], [31, 31]),
    (3, 10, [[P, P], [P, P], [P, P]], [0, 2, 2], [17, 19, 19]),
    (3, 10, [[OUT, WALL], [P, P], [P, P]], [0, 0, 4], [7, 19, 19]),
    (3, 8, [[P, P], [WALL, OUT], [OUT, WALL]], [6, 6, 6], [9, 9, 9]),
])
def test_ml_rectangles_match_oracle(gpu, oracle_lib, dim, n, bc, lo, hi):
    M.test_ml_projection_matches_oracle(oracle_lib, dim, n, bc, lo, hi, 1)
