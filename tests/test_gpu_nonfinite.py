"""A residual with NaN in it is not a small one: solves that overflow, and right
sides that are not finite, never count as converged.  The differentiable entries
pass the latter on as NaN."""
import math

import numpy as np
import pytest

from maestro_amd import autograd
from maestro_amd import mac
from maestro_amd import workloads as W

from .helpers import run_gpu
from .test_gpu_kernels import make_plan, rand_level

pytestmark = pytest.mark.gpu

P, WALL, OUT = W.PERIODIC, W.SLIP_WALL, W.OUTLET


@pytest.mark.parametrize("cfg,n", [(1, (64, 64, 64)), (1, (128, 64, 64)), (0, (384, 256))])
def test_diverging_solve_is_not_converged(gpu, cfg, n):
    """An outlet above a beta0 contrast of 1e4, where the V-cycle diverges (the
    oracle's too): the FP32 cycles overflow."""
    wl = W.make_workload(cfg, n=n, box=64)
    wl["dx"] = [1.0 / max(n)] * len(n)
    wl["bc"] = wl["bc"][:-1] + [[WALL, OUT]]
    m = n[-1]
    wl["beta0"] = np.exp(-math.log(1e4) * (np.arange(m) + 0.5) / m)
    wl["beta0_edge"] = np.exp(-math.log(1e4) * np.arange(m + 1) / m)
    b0 = wl["beta0"].reshape((-1, 1, 1) if len(n) == 3 else (1, -1, 1))
    rho = b0 * (1.0 + 0.01 * np.random.default_rng(91).standard_normal(wl["phi"].shape))
    wl["rho"] = W._fill_rho_ghosts(rho, wl["bc"], len(n))
    out = run_gpu(wl, precision=mac.PREC_MIXED, check=False)
    finite = bool(np.isfinite(out["phi"]).all())
    print(out["stats"]["iters"], out["stats"]["res"], finite)
    assert not out["stats"]["converged"]


@pytest.mark.parametrize("prec", [mac.PREC_FP64, mac.PREC_MIXED])
@pytest.mark.parametrize("n", [(128, 8, 8), (16, 12, 10), (15, 10, 12), (32, 24), (33, 20)])
@pytest.mark.parametrize("value", [math.nan, math.inf])
def test_right_side_not_finite(gpu, oracle_lib, n, value, prec):
    torch, O = gpu, oracle_lib
    dim = len(n)
    bc = [[WALL, OUT]] * dim
    g = O.make_grid(n, [1.0 / n[0]] * dim, bc)
    b, phi, rhs = rand_level(g, n, dim, np.random.default_rng(93), O)
    rhs.flat[rhs.size // 3] = value
    plan = make_plan(n, bc, precision=prec, max_iter=5, device_ptrs=1)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    z = [t(np.zeros(O.face_shape(g, d))) for d in range(dim)] + [None] * (3 - dim)
    ph = t(0.0 * phi)
    st = plan.project_level(*z, ph, *[t(x) for x in b], *[None] * (3 - dim), t(rhs))
    assert bool(torch.isnan(ph).all()) and not st["converged"]


def test_gradient_not_finite(gpu):
    torch = gpu
    n = (16, 12, 10)
    plan = autograd.level_plan(n, (1.0 / 16,) * 3, [[P, P], [WALL, WALL], [WALL, WALL]], precision=mac.PREC_FP64)
    rng = np.random.default_rng(95)
    shape = lambda d: tuple(n[e] + (e == d) for e in (2, 1, 0))
    t = lambda a: torch.from_numpy(a).cuda().requires_grad_(True)
    U = [t(np.zeros(shape(d))) for d in range(3)]
    B = [t(rng.uniform(0.5, 2.0, shape(d))) for d in range(3)]
    phi, *u = autograd.mac_project(plan, *U, *B)
    weight = torch.ones_like(phi)
    weight[3, 4, 5] = math.nan
    grads = torch.autograd.grad((weight * phi).sum(), U)
    assert all(bool(torch.isnan(x).any()) for x in grads)
