"""SOR solves with arguments at the ends of their ranges."""
import numpy as np
import pytest

from osinco3d_amd import capi
from tests.helpers import rand_fields

pytestmark = pytest.mark.gpu


# Resting tiles and the march: solves of more than one batch of launches.
@pytest.mark.parametrize("shape", [(20, 24, 40), (40, 130, 58)])
@pytest.mark.parametrize("kmax", [1 << 30, (1 << 31) - 1])
def test_any_kmax(shape, kmax):
    rhs, p0 = rand_fields(shape, 2, seed=77)
    rhs -= rhs.mean()
    got = []
    for k in (5000, kmax):
        p = p0.copy()
        got.append((capi.poisson(p, rhs, (0.3, 0.35, 0.4), 1.6, 1e-6, k, 0, "0000"), p))
    assert got[0][0] == got[1][0] and 20 < got[0][0][0] < 5000
    assert np.array_equal(got[0][1], got[1][1])


# One block, resting tiles, the march.  The one-iteration kernel's largest update leaves
# out NaN, so a solve with omega = NaN ends on eps once the field is NaN.
@pytest.mark.parametrize("shape", [(12, 12, 16), (20, 24, 40), (20, 90, 264)])
@pytest.mark.parametrize("idyn", [0, 1])
@pytest.mark.parametrize("omega", [np.nan, np.inf])
def test_omega_not_finite(shape, idyn, omega):
    rhs, p0 = [a.astype(np.float32) for a in rand_fields(shape, 2, seed=78)]
    got = []
    for variant in (0, 2):
        p = p0.copy()
        it, dmax, reason, om = capi.poisson_f32(p, rhs, (0.3, 0.35, 0.4), omega, 1e-6, 12, idyn,
                                                "0000", variant=variant)
        got.append((it, dmax, reason, p, om))
    assert got[0][:3] == got[1][:3]
    assert np.array_equal(got[0][3], got[1][3], equal_nan=True)
    assert np.array_equal(got[0][4], got[1][4], equal_nan=True)


# idyn = 1: where omega changes after a pair's first iteration the next launch runs the
# pair again; the timing counts each iteration of the solve once.
def test_timed_iterations_of_changing_omega():
    from osinco3d_amd.config import tgv_config
    from osinco3d_amd.solver import FP64, Solver, taylor_green
    cfg = tgv_config(48, 1, 2, kmax=40)
    cfg.idyn, cfg.omega = 1, 4.0  # above 2 the updates grow, and omega falls with each
    s = Solver(cfg, FP64)
    s.upload(*taylor_green(cfg))
    done = s.step(1)["sor_exit_iter"] - 1
    ms, sweeps, launches = s.sor_timing(launches=True)
    print(f"iterations {done}, timed {sweeps[0]} in {launches[0]} launches, {ms[0]:.3f} ms")
    assert done == 40 and 0 < sweeps[0] <= done and ms[0] > 0
    s.close()
