"""Bottoms of more than 1024 cells with an odd period, across which two cells
of one colour are neighbours: a half-sweep updates a colour from its old values,
so that the result does not depend on the order of the cells."""
import numpy as np
import pytest

from maestro_amd import workloads as W

from .test_gpu_kernels import make_plan, push_level, rand_level

pytestmark = pytest.mark.gpu

P, WALL, OUT = W.PERIODIC, W.SLIP_WALL, W.OUTLET
# level 1 is the bottom
CASES = [((30, 22, 18), [[P, P], [P, P], [WALL, OUT]]), ((40, 18, 22), [[P, P], [WALL, WALL], [P, P]]),
         ((70, 66), [[P, P], [WALL, OUT]]), ((80, 62), [[P, P], [P, P]])]


def level(O, n, bc):
    g = O.make_grid(n, [1.0 / n[0]] * len(n), bc)
    b, phi, rhs = rand_level(g, n, len(n), np.random.default_rng(81), O)
    for d in range(len(n)):
        if bc[d][0] == P:   # one face on both sides of a period
            np.moveaxis(b[d], 2 - d, 0)[-1] = np.moveaxis(b[d], 2 - d, 0)[0]
    return g, b, phi, rhs


def colour_sweeps(dim, bc, ih2, w, rhs, sweeps):
    """From zero, on folded weights w (bx, .. as the library keeps a level)."""
    shape = rhs.shape
    faces, den = [], np.zeros(shape)
    for d in range(dim):
        ax = 2 - d
        lo = w["bx by bz".split()[d]].reshape(shape)
        high = np.expand_dims(w["bxh byh bzh".split()[d]].reshape(tuple(np.delete(shape, ax))), ax)
        hi = np.concatenate([np.take(lo, np.arange(1, shape[ax]), ax), high], ax)
        faces.append((lo, hi))
        den += ih2 * (lo + hi)
    k, j, i = np.indices(shape)
    x = np.zeros(shape)
    for h in range(2 * sweeps):
        num = rhs.copy()
        for d in range(dim):
            for s, wt in zip((1, -1), faces[d]):
                p = np.roll(x, s, 2 - d)
                if bc[d][0] != P:
                    sl = [slice(None)] * 3
                    sl[2 - d] = 0 if s == 1 else -1
                    p[tuple(sl)] = 0.0
                num += ih2 * wt * p
        x = np.where((i + j + k) % 2 == h % 2, num / den, x)
    return x


@pytest.mark.parametrize("n,bc", CASES)
def test_sweeps_of_an_odd_period(gpu, oracle_lib, n, bc):
    dim = len(n)
    g, b, phi, rhs = level(oracle_lib, n, bc)
    plan = make_plan(n, bc, bottom_solver=0, nub=3)
    push_level(plan, 0, bc, n, b, phi, rhs, dim)
    plan.debug_op(0, "coarsen")
    plan.debug_op(0, "vcycle")
    shape = tuple(m // 2 if m > 1 else 1 for m in phi.shape)
    w = {k: plan.debug_get(1, k) for k in ("bx", "bxh", "by", "byh", "bz", "bzh")[:2 * dim]}
    want = colour_sweeps(dim, bc, n[0] ** 2 / 4.0, w, plan.debug_get(1, "rhs").reshape(shape), 6)
    # 12 half-sweeps, each a mean of values with some 15 roundings
    err = float(np.abs(plan.debug_get(1, "phi").reshape(shape) - want).max())
    assert err <= 12 * 15 * 2.0 ** -53 * max(1.0, float(np.abs(want).max()))


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n,bc", CASES[:3])
def test_solves_of_an_odd_period_repeat(gpu, oracle_lib, n, bc, prec):
    """The same bits on every call, and the residual asked for."""
    torch, O = gpu, oracle_lib
    dim = len(n)
    g, b, _, rhs = level(O, n, bc)
    if bc[-1][1] != OUT:
        rhs -= rhs.mean()
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    got = []
    for _ in range(3):
        plan = make_plan(n, bc, precision=prec, device_ptrs=1)
        z = [t(np.zeros(O.face_shape(g, d))) for d in range(dim)] + [None] * (3 - dim)
        ph = t(np.zeros(O.cell_shape(g)))
        st = plan.project_level(*z, ph, *[t(x) for x in b], *[None] * (3 - dim), t(rhs), check=False)
        assert st["converged"]
        got.append(ph.cpu().numpy())
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    res, _ = O.residual(g, b, got[0], rhs)
    tol = 1e-10 * np.abs(rhs).max() + 20 * 2.0 ** -53 * 12 * 2.0 * n[0] ** 2 * np.abs(got[0]).max()
    assert float(np.abs(res).max()) <= tol
