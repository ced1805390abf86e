"""Finest levels kept in rho form or in bfloat16 that are small enough for the
single-workgroup cycle, or that have no coarser level: the cycle reads the
stored FP32 weights and right side, which those forms do not write."""
import numpy as np
import pytest

from maestro_amd import mac
from maestro_amd import workloads as W

from .helpers import rel_err, run_gpu, run_oracle
from .test_gpu_kernels import make_plan, rand_level

pytestmark = pytest.mark.gpu

P, WALL, OUT = W.PERIODIC, W.SLIP_WALL, W.OUTLET


@pytest.mark.parametrize("cycle", [mac.CYCLE_V, mac.CYCLE_F, mac.CYCLE_W])
@pytest.mark.parametrize("prec", [mac.PREC_MIXED, mac.PREC_MIXED_BF16])
@pytest.mark.parametrize("top", [W.SLIP_WALL, W.OUTLET])
def test_finest_level_of_4096_cells(gpu, oracle_lib, prec, cycle, top):
    """128 x 4 x 8 cells: the one extent whose finest level takes either form
    and fits the single-workgroup cycle."""
    wl = W.make_workload(1, n=(128, 4, 8), box=4)
    wl["dx"] = [1.0 / 128] * 3
    wl["bc"] = [wl["bc"][0], wl["bc"][1], [W.SLIP_WALL, top]]
    truth = run_oracle(wl, eps=1e-13)
    same = run_oracle(wl, eps=1e-10)
    out = run_gpu(wl, precision=prec, cycle_type=cycle)
    sing = top != W.OUTLET
    e_phi = rel_err(out["phi"], truth["phi"], remove_mean=sing)
    e_ref = rel_err(same["phi"], truth["phi"], remove_mean=sing)
    e_u = max(rel_err(out["faces"][d], truth["faces"][d]) for d in range(3))
    print(f"prec {prec} cycle {cycle}: {out['stats']['iters']} steps, phi {e_phi:.2e} (oracle {e_ref:.2e}), "
          f"U {e_u:.2e}")
    assert out["stats"]["converged"]
    # NaN fails both; the bounds are those of the parity tests
    assert e_phi <= max(1e-8, 2.0 * e_ref)
    assert e_u <= 1e-8


@pytest.mark.parametrize("n,levels", [((128, 3, 8), 0), ((256, 3, 9), 0), ((128, 4, 8), 1), ((128, 12, 16), 1)])
@pytest.mark.parametrize("bc", [[[P, P], [WALL, WALL], [WALL, OUT]], [[OUT, WALL], [WALL, OUT], [WALL, WALL]]])
def test_bf16_of_one_level(gpu, oracle_lib, n, levels, bc):
    """MAC_PREC_MIXED_BF16 where the finest level is the bottom."""
    torch, O = gpu, oracle_lib
    g = O.make_grid(n, [1.0 / n[0]] * 3, bc)
    b, phi, rhs = rand_level(g, n, 3, np.random.default_rng(61), O)
    plan = make_plan(n, bc, precision=mac.PREC_MIXED_BF16, max_levels=levels, device_ptrs=1)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    ph = t(np.zeros_like(phi))
    z = [t(np.zeros(O.face_shape(g, d))) for d in range(3)]
    st = plan.project_level(*z, ph, *[t(x) for x in b], t(rhs), check=False)
    res, _ = O.residual(g, b, ph.cpu().numpy(), rhs)
    print(n, st["iters"], np.abs(res).max())
    # the tolerance asked for, and the rounding of a residual: some 20 operations on terms of 6 w ih2 |phi|
    tol = 1e-10 * np.abs(rhs).max() + 20 * 2.0 ** -53 * 12 * 2.0 * n[0] ** 2 * np.abs(ph.cpu().numpy()).max()
    assert st["converged"] and np.abs(res).max() <= tol
