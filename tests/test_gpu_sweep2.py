"""Two sweeps in one pass over memory against the oracle's single sweeps,
bitwise in FP64 and FP32: tiles (24 x 24 columns in FP64, 56 x 24 in FP32) cut
by the domain's end on each side, chunks of planes of every remainder, domains
below a tile's halo and periods that a tile spans more than once."""
import numpy as np
import pytest

from maestro_amd import workloads as W

from . import test_gpu_solve as S
from .test_gpu_kernels import fp32_reference, make_plan, push_level, rand_level, ref_omega

pytestmark = pytest.mark.gpu

P, WALL, OUT = W.PERIODIC, W.SLIP_WALL, W.OUTLET
BCS = [[[P, P], [P, P], [P, P]], [[WALL, OUT], [P, P], [WALL, OUT]], [[P, P], [OUT, WALL], [P, P]],
       [[OUT, OUT], [OUT, WALL], [WALL, WALL]]]


@pytest.mark.parametrize("omega", [0.0, 1.25])
@pytest.mark.parametrize("n", [(4, 4, 4), (2, 6, 10), (24, 24, 4), (26, 25, 5), (56, 48, 6), (58, 23, 7), (120, 6, 33),
                               (10, 130, 18)])
@pytest.mark.parametrize("bc", BCS)
def test_two_sweeps_bitwise(gpu, oracle_lib, n, bc, omega):
    O = oracle_lib
    bc = [[WALL, OUT] if m % 2 and kind[0] == P else kind for m, kind in zip(n, bc)]
    g = O.make_grid(n, [1.0 / n[0]] * 3, bc)
    b, phi, rhs = rand_level(g, n, 3, np.random.default_rng(41), O)
    plan = make_plan(n, bc, omega=omega)
    for op, want in (("gsrb", O.gsrb(g, b, phi, rhs, sweeps=4, omega=ref_omega(n, omega))),
                     ("gsrb32", fp32_reference(O, n, bc, b, phi, rhs, 4, omega=ref_omega(n, omega)))):
        push_level(plan, 0, bc, n, b, phi, rhs, 3)
        plan.debug_op(0, op, 4)
        assert np.array_equal(plan.debug_get(0, "phi").reshape(phi.shape), want)


# from a zero iterate (level 0 of the FP32 cycles; level 1 of the FP64 one) and
# with alpha, at the tolerances of the solver's own tests
ELL = [[S.PER, S.PER], [S.NEU, S.DIR], [S.DIR, S.NEU]]


@pytest.mark.parametrize("n,box,prec", [((72, 64, 72), 8, 0), ((72, 64, 72), 8, 1), ((144, 128, 128), 16, 0)])
@pytest.mark.parametrize("alpha", ["rand", None])
def test_two_sweeps_in_the_solver(gpu, oracle_lib, n, box, prec, alpha):
    S.test_solve_matches_oracle(gpu, oracle_lib, n, box, ELL, alpha, prec, True)


@pytest.mark.parametrize("prec", [0, 1])
def test_two_over_relaxed_sweeps_in_the_solver(gpu, oracle_lib, prec):
    S.test_solve_over_relaxed_matches_oracle(gpu, oracle_lib, (72, 64, 72), 8, ELL, prec)
