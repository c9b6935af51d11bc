"""Multigrid last levels whose colours meet (an odd axis that wraps makes cells 0
and m - 1 neighbours of one colour): every kernel reads a colour whole before it
writes it, so V-cycles equal the float32 restatement bit for bit and two runs of
one program agree."""
import numpy as np
import pytest

from osinco3d_amd import capi
from osinco3d_amd.config import mixing_layer_config
from osinco3d_amd.solver import MIXED, WARM_EXTRAPOLATE, Solver, mixing_layer
from tests.helpers import rand_fields
from tests.test_gpu_mg_sweep import F, _vcycle

pytestmark = pytest.mark.gpu


# (nz, ny, nx) and the last level's cells.  One block: 3 x 5 x 17, 5 x 3 x 6, 3 x 3 x 17,
# 9 x 15 x 20 (three cells per thread), 5 x 9 x 22.  In a group of small levels: 7 x 7 x 7
# and 5 x 6 x 6.  Launches per colour (more than 40 cells wide): 17 x 7 x 65, 5 x 21 x 44.
# Rows in LDS: 13 x 9 x 36.
@pytest.mark.parametrize("shape", [(12, 20, 68), (40, 24, 48), (6, 6, 34), (18, 30, 40),
                                   (20, 36, 88), (28, 28, 28), (20, 24, 24), (34, 14, 130),
                                   (10, 42, 88), (26, 18, 72)])
@pytest.mark.parametrize("per", [(1, 1, 1), (1, 0, 1), (0, 1, 1)])
def test_vcycles_equal_restatement(shape, per):
    f, = rand_fields(shape, 1, seed=74)
    f = f.astype(F)
    h = (0.1, 0.12, 0.11)
    u = np.zeros(shape, F)
    capi.multigrid(u, f, h, per, 2)
    if not all(per):
        # The library solves for the part of f with zero mean: its own f32 mean.
        f = f - F(f.astype(np.float64).sum() / f.size)
    ref = np.zeros(shape, F)
    for _ in range(2):
        ref = _vcycle(ref, f, h, per)
    if all(per):
        assert np.array_equal(u, ref)
    else:
        # The mean's last bit may differ with the order of its sum.
        assert np.abs(u - ref).max() <= 1e-5 * np.abs(ref).max()


# Last levels of 29 x 15 x 12, 27 x 11 x 8 and 19 x 13 x 48 cells.
@pytest.mark.parametrize("nx,ny,nz", [(48, 60, 116), (32, 44, 108), (192, 52, 76)])
def test_two_runs_agree(nx, ny, nz):
    cfg = mixing_layer_config(nx, ny, nz, 2, lengths=(60.0 * nx / 384, 40.0 * ny / 256,
                                                      20.0 * nz / 128))
    got = []
    for _ in range(2):
        s = Solver(cfg, MIXED, WARM_EXTRAPOLATE, coarse_cycles=2, smooth_sweeps=8, adaptive=1)
        s.upload(*mixing_layer(cfg))
        for it in (1, 2):
            s.step(it)
        got.append(s.download())
        s.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("shape", [(16, 28, 144), (34, 46, 16), (30, 54, 96)])
def test_two_solves_agree(shape):
    rhs, = rand_fields(shape, 1, seed=75)
    rhs = rhs - rhs.mean()
    got = []
    for _ in range(2):
        p = np.zeros(shape)
        capi.poisson_multigrid(p, rhs, (0.3, 0.32, 0.35), "0000", tol=1e-6, max_cycles=20)
        got.append(p)
    assert np.array_equal(*got)
