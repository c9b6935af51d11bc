"""The two-iterations-per-launch SOR kernel at the edges of its tiles: iterates,
dmax, omega and exit equal the oracle's (FP64) and the one-iteration kernel's
(FP32) bit for bit, for even and odd counts of sweeps."""
import numpy as np
import pytest

from osinco3d_amd import capi

from tests.helpers import rand_fields

pytestmark = pytest.mark.gpu


# FP64 tiles own 56 x 16 nodes and chunks of an even number of planes; resting tiles
# 24 x 8 x 8.
@pytest.mark.parametrize("solver,shape", [("0000", (6, 6, 6)), ("0000", (8, 16, 56)),
                                          ("0000", (10, 18, 58)), ("0011", (8, 33, 114)),
                                          ("111111", (9, 17, 56)), ("0011", (42, 15, 10)),
                                          ("111111", (11, 7, 70)),
                                          # One round of resting tiles, more: the
                                          # march with 16 rows, with 24 rows.
                                          ("0011", (40, 130, 58)), ("0000", (66, 66, 130)),
                                          ("111111", (51, 67, 100)),
                                          ("0011", (130, 145, 116)), ("111111", (129, 128, 128))])
@pytest.mark.parametrize("idyn", [0, 1])
def test_pair_f64_equals_oracle(orc, solver, shape, idyn):
    rhs, p0 = rand_fields(shape, 2, seed=61)
    rhs -= rhs.mean()
    d = (0.3, 0.35, 0.4)
    runs = ((1e-4, 300), (1e-2, 300), (1e-30, 1), (1e-30, 6), (1e-30, 7))
    for eps, kmax in runs[3:] if rhs.size > 1e6 else runs:
        pg, po = p0.copy(), p0.copy()
        it, dm, rs, om = capi.poisson(pg, rhs, d, 1.6, eps, kmax, idyn, solver)
        ito, dmo, rso, omo, _ = orc.sor(po, rhs, d, solver, 1.6, eps, kmax, idyn, red_black=True)
        assert (it, rs, dm, om) == (ito, rso, dmo, omo), (eps, kmax)
        assert np.array_equal(pg, po), (eps, kmax)


# Resting tiles of 24 x 8 x 8 nodes, then the march: its narrow FP32 tile owns 56 x
# 40 nodes; the last shape is beyond the size where the wide one (120 x 24) takes over.
@pytest.mark.parametrize("solver,shape", [("0000", (20, 90, 264)), ("0011", (16, 121, 280)),
                                          ("0000", (24, 40, 72)), ("111111", (25, 39, 128)),
                                          ("0000", (10, 40, 56)), ("0011", (10, 81, 64)),
                                          ("111111", (13, 41, 120)),
                                          ("0011", (258, 289, 304))])
def test_pair_f32_equals_single(solver, shape):
    rhs, p0 = [a.astype(np.float32) for a in rand_fields(shape, 2, seed=62)]
    d = (0.3, 0.35, 0.4)
    for kmax in (5, 6):
        pa, pb = p0.copy(), p0.copy()
        a = capi.poisson_f32(pa, rhs, d, 1.7, 1e-30, kmax, 0, solver, variant=0)
        b = capi.poisson_f32(pb, rhs, d, 1.7, 1e-30, kmax, 0, solver, variant=2)
        assert a == b, kmax
        assert np.array_equal(pa, pb), kmax


# Grids of one block, up to its largest of every number of pairs per thread.
@pytest.mark.parametrize("solver,shape", [("0000", (16, 16, 16)), ("111111", (17, 16, 16)),
                                          ("0011", (16, 13, 38)), ("0000", (16, 16, 32))])
def test_block_f64_equals_oracle(orc, solver, shape):
    rhs, p0 = rand_fields(shape, 2, seed=63)
    rhs -= rhs.mean()
    d = (0.3, 0.35, 0.4)
    for omega, eps, kmax, idyn in ((1.6, 1e-4, 300, 0), (1.6, 1e-2, 300, 1), (1.6, 1e-30, 1, 0),
                                   (1.6, 1e-30, 8, 1),
                                   # More iterations than one launch runs.
                                   (1.0, 1e-30, 701, 0)):
        pg, po = p0.copy(), p0.copy()
        got = capi.poisson(pg, rhs, d, omega, eps, kmax, idyn, solver)
        it, dm, rs, om, _ = orc.sor(po, rhs, d, solver, omega, eps, kmax, idyn, red_black=True)
        assert got == (it, dm, rs, om), (omega, eps, kmax)
        assert np.array_equal(pg, po), (omega, eps, kmax)


@pytest.mark.parametrize("solver,shape", [("0000", (6, 6, 8)), ("0011", (16, 11, 24)),
                                          ("111111", (9, 29, 24)), ("0000", (16, 16, 64))])
def test_block_f32_equals_single(solver, shape):
    rhs, p0 = [a.astype(np.float32) for a in rand_fields(shape, 2, seed=64)]
    d = (0.3, 0.35, 0.4)
    for kmax in (5, 600):
        pa, pb = p0.copy(), p0.copy()
        a = capi.poisson_f32(pa, rhs, d, 1.0, 1e-30, kmax, 0, solver, variant=0)
        b = capi.poisson_f32(pb, rhs, d, 1.0, 1e-30, kmax, 0, solver, variant=2)
        assert a == b, kmax
        assert np.array_equal(pa, pb), kmax
