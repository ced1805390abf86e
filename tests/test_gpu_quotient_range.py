"""Sweeps on levels whose diagonals lie at the ends of the exponent range, where
a reciprocal is not a normal number: the pairs of sweeps, the legs and the
single-workgroup cycle."""
import numpy as np
import pytest

from maestro_amd import workloads as W

from .test_gpu_kernels import fp32_reference, make_plan, push_level, rand_level

pytestmark = pytest.mark.gpu

P, WALL, OUT = W.PERIODIC, W.SLIP_WALL, W.OUTLET


# A diagonal is 6 ih2 b with b in [0.5, 2): with 12 ih2 b up to the factor
# below, [2^(top - 2), 2^top) where no face is closed.
@pytest.mark.parametrize("n", [(10, 12, 14), (58, 24, 6)])
@pytest.mark.parametrize("bc", [[[P, P]] * 3, [[P, P], [P, P], [WALL, WALL]]])
def test_two_sweeps_at_the_ends_of_the_range(gpu, oracle_lib, n, bc):
    """Bit for bit: every diagonal's reciprocal is out of the normal range
    (or, beside a closed face at the upper end, the products are exact)."""
    O = oracle_lib
    g = O.make_grid(n, [1.0 / n[0]] * 3, bc)
    b, phi, rhs = rand_level(g, n, 3, np.random.default_rng(71), O)
    unit = 1.0 / (6 * 2.0 * n[0] ** 2)   # b in [0.5, 2) to a diagonal in [1/4, 1)
    phi *= 2.0 ** -6
    for op, tops in (("gsrb32", (-126, 128)), ("gsrb", (-1022, 1024))):
        for top in tops:
            s = float(np.ldexp(unit, top))
            bs, rs = [x * s for x in b], rhs * 2.0 ** (top - 8)
            plan = make_plan(n, bc)
            push_level(plan, 0, bc, n, bs, phi, rs, 3)
            plan.debug_op(0, op, 4)
            got = plan.debug_get(0, "phi").reshape(phi.shape)
            want = O.gsrb(g, bs, phi, rs, sweeps=4) if op == "gsrb" else fp32_reference(O, n, bc, bs, phi, rs, 4)
            finite, same = bool(np.isfinite(want).all()), np.array_equal(got, want)
            assert finite and same, (op, top)


@pytest.mark.parametrize("n", [(6, 6, 6), (12, 10, 14), (38, 50, 46), (72, 64, 72), (66, 70), (18, 20)])
@pytest.mark.parametrize("top", [-126, 128])
@pytest.mark.parametrize("cycle", [2, 3])
def test_fp32_cycle_at_the_ends_of_the_range(gpu, oracle_lib, n, top, cycle):
    """One FP32 cycle on weights and right side scaled by a power of two, which
    leaves the solution alone: exactly at the upper end.  At the lower one the
    weights and diagonals are denormal but exact, and only small terms of a sum
    round differently, by less than 2^-24 of the largest, which a domain of m
    cells across amplifies by at most m^2."""
    torch, O = gpu, oracle_lib
    dim = len(n)
    m = list(n)
    while all(x % 2 == 0 and x >= 4 for x in m):
        m = [x // 2 for x in m]
    # an odd period has no colouring
    bc = [[P, P] if m[d] % 2 == 0 and d < dim - 1 else [WALL, OUT] for d in range(dim)]
    g = O.make_grid(n, [1.0] * dim, bc)
    b, _, rhs = rand_level(g, n, dim, np.random.default_rng(73), O)
    b = [np.floor(4.0 * x) / 4.0 for x in b]   # at most 1.75: diagonals and sums of four faces below 16
    rhs *= 2.0 ** (-12 if top > 0 else 12)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    got = []
    for k in (0, top - 4):
        plan = make_plan(n, bc, dx=[1.0] * dim, precision=1, inner_cycles=1, max_iter=1, eps_rel=1e-300,
                         cycle_type=cycle, device_ptrs=1)
        z = [t(np.zeros(O.face_shape(g, d))) for d in range(dim)] + [None] * (3 - dim)
        bt = [t(x * 2.0 ** k) for x in b] + [None] * (3 - dim)
        ph = t(np.zeros(O.cell_shape(g)))
        plan.project_level(*z, ph, *bt, t(rhs * 2.0 ** k), check=False)
        got.append(ph.cpu().numpy())
    assert np.isfinite(got[0]).all() and np.abs(got[0]).max() > 0.0
    tol = 0.0 if top > 0 else max(n) ** 2 * 2.0 ** -24
    err, scale = float(np.abs(got[1] - got[0]).max()), float(np.abs(got[0]).max())
    assert err <= tol * scale
