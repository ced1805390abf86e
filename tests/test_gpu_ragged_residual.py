"""The FP64 residual passes on levels of any even row length against the
oracle's residual, bitwise: its maximum after one cycle and the FP32 right side
of the next one, for rows of fewer and of more pairs than a wave has lanes, a
last wave that is part empty, and chunks of planes of every remainder."""
import numpy as np
import pytest

from maestro_amd import workloads as W

from .test_gpu_kernels import make_plan
from .test_gpu_legs import level

pytestmark = pytest.mark.gpu

P, WALL, OUT = W.PERIODIC, W.SLIP_WALL, W.OUTLET
BCS = [[[P, P], [P, P], [WALL, OUT]], [[WALL, OUT], [P, P], [P, P]], [[OUT, OUT], [OUT, WALL], [WALL, WALL]]]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [(8, 4, 4), (20, 12, 16), (62, 20, 14), (66, 34, 30), (132, 16, 24), (190, 10, 72), (640, 10),
                               (40, 24)])
@pytest.mark.parametrize("bc", BCS)
def test_residual_passes_bitwise(gpu, oracle_lib, n, bc, precision):
    torch = gpu
    O = oracle_lib
    dim = len(n)
    g, b, phi, rhs = level(O, n, bc, 43)
    plan = make_plan(n, bc[:dim], precision=precision, inner_cycles=1, max_iter=1, device_ptrs=1)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    z = [t(np.zeros(O.face_shape(g, d))) for d in range(dim)] + [None] * (3 - dim)
    bt = [t(x) for x in b] + [None] * (3 - dim)
    ph = t(np.zeros(O.cell_shape(g)))
    st = plan.project_level(*z, ph, *bt, t(rhs), check=False)
    got = plan.debug_get(0, "phi").reshape(phi.shape)
    r0 = plan.debug_get(0, "rhs").reshape(phi.shape)
    res, norm = O.residual(g, b, got, r0)
    assert st["res"] == norm == np.abs(res).max()
    if precision == 1:
        assert np.array_equal(plan.debug_get(0, "rhs", copy="f32"), res.astype(np.float32).ravel())
