"""Radial profiles of every size class (copied to LDS, read in memory) and
values (zeros, magnitudes whose quotients leave the normal range) in
make_macrhs and make_s0mac, bit for bit against the oracle, on boxes that cut
the kernels' rows, tiles and plane chunks raggedly."""
import numpy as np
import pytest

from maestro_amd import boxes as BX
from maestro_amd import mac
from maestro_amd import workloads as W

from .test_gpu_inputs import OUT, per_box, plan_for, to_dev

pytestmark = pytest.mark.gpu


def radial(n, bins):
    """dr (bins per cell), number of bins, centre, corner."""
    dx = 1.0 / n[0]
    ext = [m * dx for m in n]
    return dx, dx / bins, int(0.5 * np.sqrt(sum(e * e for e in ext)) * bins / dx) + 2, [0.5 * e for e in ext], [0.0] * 3


def profile(kind, nr, rng):
    p = np.sort(rng.uniform(1e-3, 2.0, nr))[::-1].copy()
    if kind == "zeros":
        p[nr // 3:] = 0.0
    elif kind == "tiny":
        p *= np.where(np.arange(nr) % 2 == 0, 1e-300, 1e-150)
    return p


@pytest.mark.parametrize("kind", ["normal", "zeros", "tiny"])
@pytest.mark.parametrize("n,box,bins,interp", [((90, 90, 90), 90, 5, 3), ((90, 90, 90), 30, 100, 3), ((34, 34, 34), 17, 5, 2),
                                               ((6, 6, 6), 3, 4, 3), ((24, 24, 24), 24, 400, 2), ((24, 24, 24), 24, 400, 1)])
def test_s0mac_profiles_bitwise(gpu, oracle_lib, n, box, bins, interp, kind):
    torch = gpu
    dx, dr, nr, ctr, plo = radial(n, bins)
    s0 = profile(kind, nr, np.random.default_rng(interp))
    ref = oracle_lib.make_s0mac(n, s0, dr, ctr, plo, (dx,) * 3, interp)
    plan = plan_for(n, box, [[OUT, OUT]] * 3)
    boxes = W.box_list(n, box)
    out = [[torch.full(BX.box_shape(lo, hi, 1, 3, face_dir=d), float("nan"), dtype=torch.float64, device="cuda")
            for d in range(3)] for lo, hi in boxes]
    plan.make_s0mac(torch.from_numpy(s0).cuda(), mac.sphr(dr, nr, ctr, plo, interp), out)
    for (lo, hi), box_f in zip(boxes, out):
        for d in range(3):
            e = [hi[q] - lo[q] + 3 + (q == d) for q in range(3)]
            want = ref[d][lo[2]:lo[2] + e[2], lo[1]:lo[1] + e[1], lo[0]:lo[0] + e[0]]
            assert np.array_equal(box_f[d].cpu().numpy(), want), (lo, d)
    plan.close()


@pytest.mark.parametrize("kind", ["normal", "zeros", "tiny"])
@pytest.mark.parametrize("n,box,bins,interp,dpdt", [((34, 34, 34), 34, 5, 3, 0.5), ((34, 34, 34), 17, 100, 3, 0.5),
                                                    ((34, 34, 34), 17, 100, 2, -1.0), ((6, 6, 6), 3, 4, 1, 0.5)])
def test_macrhs_profiles_bitwise(gpu, oracle_lib, n, box, bins, interp, dpdt, kind):
    torch = gpu
    dx, dr, nr, ctr, plo = radial(n, bins)
    rng = np.random.default_rng(interp)
    shp = tuple(reversed(n))
    S, dg, dp, dchi = (rng.standard_normal(shp) for _ in range(4))
    Sbar, beta0, rho0 = (profile(kind, nr, rng) for _ in range(3))
    g1, p0 = (profile("normal", nr, rng) for _ in range(2))
    ref_chi = dchi.copy()
    ref = oracle_lib.make_macrhs(n, S, dg, Sbar, beta0, gamma1bar=g1, p0=p0, rho0=rho0, dp=dp, dchi=ref_chi, dt=0.3,
                                 dpdt_factor=dpdt, base_cutoff_density=0.2, is_predictor=False,
                                 sph=(dr, ctr, plo, interp), dx=(dx,) * 3)
    plan = plan_for(n, box, [[OUT, OUT]] * 3)
    boxes = W.box_list(n, box)
    dev = lambda a: to_dev(torch, per_box(a, boxes, 0, 3, [[OUT, OUT]] * 3))
    rhs, chi = dev(np.zeros(shp)), dev(dchi)
    one = to_dev(torch, [Sbar, beta0, g1, p0, rho0])
    on = dpdt >= 0.0
    plan.make_macrhs(rhs, dev(S), dev(dg), one[0], one[1], delta_p_term=dev(dp) if on else None,
                     delta_chi=chi if on else None, gamma1bar=one[2], p0=one[3], rho0=one[4], dt=0.3,
                     dpdt_factor=dpdt, base_cutoff_density=0.2, is_predictor=False,
                     sph=mac.sphr(dr, nr, ctr, plo, interp))
    cells = lambda bs: BX.gather_cells([b.cpu().numpy() for b in bs], boxes, 0, list(n), 3).reshape(shp)
    assert np.array_equal(cells(rhs), ref)
    if on:
        assert np.array_equal(cells(chi), ref_chi)
    plan.close()
