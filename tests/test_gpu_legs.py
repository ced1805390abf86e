"""The fused legs (two sweeps with the residual restriction, or with the
prolongation, in one launch) and the single-workgroup cycle against the
oracle's single operators.  FP64 is bitwise: the same operations per cell in
the same order."""
import numpy as np
import pytest

from maestro_amd import workloads as W

from .test_gpu_kernels import fp32_reference, make_plan, push_level, rand_level, ref_omega

pytestmark = pytest.mark.gpu

P, WALL, OUT = W.PERIODIC, W.SLIP_WALL, W.OUTLET
BCS = [[[P, P], [P, P], [WALL, OUT]], [[WALL, OUT], [P, P], [P, P]], [[OUT, OUT], [OUT, WALL], [WALL, WALL]]]
# just above the single-workgroup cycle (4096 cells), tiles cut by the domain's
# end in each direction, extents below a tile's halo, both tile sizes
SIZES = [(18, 16, 16), (20, 12, 28), (4, 36, 34), (70, 6, 12), (38, 50, 46), (64, 48, 40), (94, 44), (66, 70), (640, 10)]


def level(O, n, bc, seed):
    g = O.make_grid(n, [1.0 / n[0]] * len(n), bc[:len(n)])
    return (g, *rand_level(g, n, len(n), np.random.default_rng(seed), O))


def half(n):
    return [x // 2 for x in n] + [1] * (3 - len(n))


def views(O, g, n, b, phi, rhs, e):
    return O.LevelView(g, b, phi.copy(), rhs), O.LevelView(g, [np.zeros(1)] * len(n), e, np.zeros_like(e), n=half(n))


def restricted(O, g, n, b, phi, rhs):
    res, _ = O.residual(g, b, phi, rhs)
    shape = half(n)[::-1]
    c = O.LevelView(g, [np.zeros(1)] * len(n), np.zeros(shape), np.zeros(shape), n=half(n))
    O.level_restrict(g, O.LevelView(g, b, phi, rhs, res=res), c)
    return c.rhs


def prolonged(O, g, n, b, phi, rhs, e):
    f, c = views(O, g, n, b, phi, rhs, e)
    O.level_prolong(g, c, f)
    return f.phi


@pytest.mark.parametrize("omega", [0.0, 1.25])
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("bc", BCS)
def test_legs_bitwise(gpu, oracle_lib, n, bc, omega):
    """One V-cycle: the right side that the way down leaves on level 1, and
    the way up from the correction that level 1 ends with."""
    O = oracle_lib
    dim = len(n)
    g, b, phi, rhs = level(O, n, bc, 31)
    plan = make_plan(n, bc[:dim], omega=omega)
    push_level(plan, 0, bc[:dim], n, b, phi, rhs, dim)
    lev = 0
    while True:
        try:
            plan.level_dims(lev + 1)
        except Exception:
            break
        plan.debug_op(lev, "coarsen")
        lev += 1
    plan.debug_op(0, "vcycle")
    w = ref_omega(n, omega)
    down = O.gsrb(g, b, phi, rhs, sweeps=2, omega=w)
    want = restricted(O, g, n, b, down, rhs)
    assert np.array_equal(plan.debug_get(1, "rhs"), want.ravel())
    e = plan.debug_get(1, "phi").reshape(want.shape)
    want = O.gsrb(g, b, prolonged(O, g, n, b, down, rhs, e), rhs, sweeps=2, omega=w)
    assert np.array_equal(plan.debug_get(0, "phi"), want.ravel())


@pytest.mark.parametrize("n", [(20, 12, 28), (38, 50, 46), (64, 48, 40), (94, 44), (66, 70)])
@pytest.mark.parametrize("bc", BCS)
def test_legs_fp32(gpu, oracle_lib, n, bc):
    """The FP32 cycle of one refinement step (from a zero iterate): the
    sweeps are the oracle's FP32 ones; the residual and the interpolation are
    formed here in FP64 from FP32 values, so each of their some 20 rounded
    operations on terms of size 6 w ih2 |phi| adds 2^-24 of that."""
    torch = gpu
    O = oracle_lib
    dim = len(n)
    g, b, _, rhs = level(O, n, bc, 33)
    plan = make_plan(n, bc[:dim], precision=1, inner_cycles=1, max_iter=1, device_ptrs=1)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    z = [t(np.zeros(O.face_shape(g, d))) for d in range(dim)] + [None] * (3 - dim)
    bt = [t(x) for x in b] + [None] * (3 - dim)
    ph = t(np.zeros(O.cell_shape(g)))
    plan.project_level(*z, ph, *bt, t(rhs), check=False)
    r0 = plan.debug_get(0, "rhs").reshape(O.cell_shape(g))   # less its mean where singular
    zero = np.zeros_like(r0)
    down = fp32_reference(O, n, bc[:dim], b, zero, r0, 2)
    want = restricted(O, g, n, b, down, r0)
    tol = 20 * 2.0 ** -24 * 6 * 2.0 * n[0] ** 2 * np.abs(down).max()
    assert np.abs(plan.debug_get(1, "rhs", copy="f32") - want.ravel()).max() <= tol
    e = plan.debug_get(1, "phi", copy="f32").reshape(want.shape)
    up = prolonged(O, g, n, b, down, r0, e).astype(np.float32)
    want = fp32_reference(O, n, bc[:dim], b, up, r0, 2)
    scale = max(np.abs(down).max(), np.abs(e).max())
    assert np.abs(plan.debug_get(0, "phi", copy="f32") - want.ravel()).max() <= 20 * 2.0 ** -24 * scale


@pytest.mark.parametrize("cycle", [1, 2, 3])
@pytest.mark.parametrize("bottom", [0, 1, 2])
@pytest.mark.parametrize("n", [(12, 10, 14), (10, 6, 6), (16, 16, 16), (8, 4, 2), (4, 4, 4), (14, 18, 10), (12, 20), (64, 60),
                               (62, 62), (2, 2), (70, 66)])
def test_bottoms(gpu, oracle_lib, n, bottom, cycle):
    """One cycle whose bottom is solved by every form (2 cells per direction,
    one wave, one block, global memory) against the oracle's.  Both reach a
    relative residual of 1e-15 there, so they differ by at most the bottom
    operator's condition number times that: the weights span a factor of 4 and
    the smoothest mode of m cells has (pi / 2m)^2 of the 4 dim of the roughest,
    which makes 6.5 dim m^2.  A direction is periodic where its bottom extent
    is even (an odd period has no red-black colouring)."""
    O = oracle_lib
    dim = len(n)
    m = list(n)
    while all(x % 2 == 0 and x >= 4 for x in m):
        m = [x // 2 for x in m]
    bc = [[P, P] if m[d] % 2 == 0 and d != 1 else [WALL, OUT] for d in range(dim)]
    g, b, phi, rhs = level(O, n, bc, 35)
    opts = dict(bottom_eps=1e-15, cycle_type=cycle, bottom_solver=bottom)
    plan = make_plan(n, bc, bottom_max_iter=400, **opts)
    push_level(plan, 0, bc, n, b, phi, rhs, dim)
    lev = 0
    while True:
        try:
            plan.level_dims(lev + 1)
        except Exception:
            break
        plan.debug_op(lev, "coarsen")
        lev += 1
    plan.debug_op(0, "vcycle")
    ref, _, _, _ = O.mg_solve(g, b, phi, rhs, O.default_opts(max_iter=1, eps_rel=1e-300, bottom_maxit=400, **opts))
    got = plan.debug_get(0, "phi").reshape(phi.shape)
    assert np.abs(got - ref).max() <= max(1e-12, 6.5 * dim * max(m) ** 2 * 1e-15) * np.abs(ref).max()


@pytest.mark.parametrize("bottom", [1, 2])
@pytest.mark.parametrize("n", [(11, 7, 9), (9, 9, 8), (27, 31), (19, 27), (32, 31)])
def test_bottom_sums_beyond_512_cells(gpu, oracle_lib, n, bottom):
    """A singular bottom of 513 to 1024 cells: the solution is the oracle's but
    for a constant, and the same bits on every call."""
    O = oracle_lib
    dim = len(n)
    bc = [[WALL, WALL]] * dim
    g, b, _, rhs = level(O, n, bc, 37)
    rhs -= rhs.mean()
    got = []
    opts = dict(bottom_eps=1e-13, bottom_solver=bottom)
    for _ in range(2):
        plan = make_plan(n, bc, bottom_max_iter=400, **opts)
        push_level(plan, 0, bc, n, b, np.zeros_like(rhs), rhs, dim)
        plan.debug_op(0, "vcycle")
        got.append(plan.debug_get(0, "phi").reshape(rhs.shape))
    ref, _, _, _ = O.mg_solve(g, b, np.zeros_like(rhs), rhs, O.default_opts(max_iter=1, eps_rel=1e-300, bottom_maxit=400, **opts))
    assert np.array_equal(got[0], got[1])
    d, e = got[0] - got[0].mean(), ref - ref.mean()
    assert np.abs(d - e).max() <= 6.5 * dim * max(n) ** 2 * 1e-13 * np.abs(e).max()
