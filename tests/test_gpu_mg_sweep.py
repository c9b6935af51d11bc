"""The fused multigrid level kernels (one launch per red-black sweep, with the
prolongation before it or the restriction after it): V(2, 2) cycles equal a
float32 restatement bit for bit on full and partial tiles with wrapped and
mirrored axes, and V(1, 1) cycles solve the pressure problem."""
import numpy as np
import pytest

from osinco3d_amd import capi
from tests.helpers import rand_fields

pytestmark = pytest.mark.gpu
F = np.float32


def _nb(u, axis, step, per):
    """Neighbour values along numpy axis: wrapped, or the edge cell itself."""
    r = np.roll(u, -step, axis)
    if not per:
        e = [slice(None)] * 3
        e[axis] = -1 if step > 0 else 0
        r[tuple(e)] = u[tuple(e)]
    return r


class Level:
    def __init__(self, shape, h, per):
        self.shape, self.h, self.per = shape, h, per
        self.c = [F(1.0 / (a * a)) for a in h]
        self.diag = F(-2.0) * (self.c[0] + self.c[1] + self.c[2])
        self.invd = F(1.0) / self.diag
        z, y, x = np.indices(shape)
        self.odd = (x + y + z) & 1

    def lap(self, u):
        s = [_nb(u, 2 - a, -1, self.per[a]) + _nb(u, 2 - a, 1, self.per[a]) for a in range(3)]
        return (self.c[0] * s[0] + self.c[1] * s[1]) + self.c[2] * s[2]

    def sweep(self, u, f):
        for colour in (0, 1):
            u = np.where(self.odd == colour, (f - self.lap(u)) * self.invd, u)
        return u

    def restrict(self, u, f):
        r = f - (self.lap(u) + self.diag * u)
        s = np.zeros(tuple(n // 2 for n in self.shape), F)
        for c in range(8):
            s = s + r[c >> 2::2, (c >> 1) & 1::2, c & 1::2]
        return F(0.125) * s

    def prolong(self, uc):
        for axis in (2, 1, 0):
            n, per = self.shape[axis], self.per[2 - axis]
            x = 0.5 * np.arange(n) - 0.25
            i0 = np.floor(x).astype(int)
            w = (x - i0).astype(F)
            i1 = i0 + 1
            m = n // 2
            if per:
                i0, i1 = i0 % m, i1 % m
            else:
                w[(i0 < 0) | (i1 >= m)] = 0
                i0, i1 = np.maximum(i0, 0), np.minimum(i1, m - 1)
            w = w.reshape([-1 if a == axis else 1 for a in range(3)])
            uc = (F(1) - w) * uc.take(i0, axis) + w * uc.take(i1, axis)
        return uc


def _vcycle(u, f, h, per, top=True, inside=False):
    """V(2, 2): 10 sweeps on the last level of a group of small levels (at most
    four levels of at most 4096 cells, 4680 together), 30 or 60 elsewhere."""
    L = Level(f.shape, h, per)

    def shapes(s):
        out = [s]
        while np.prod(s) > 64 and all(n % 2 == 0 and n >= 4 for n in s):
            s = tuple(n // 2 for n in s)
            out.append(s)
        return out

    below = shapes(f.shape)
    if len(below) == 1:
        n = f.size
        for _ in range(10 if inside else (30 if n <= 64 else 60)):
            u = L.sweep(u, f)
        return u
    cells = [int(np.prod(s)) for s in below]
    inside = inside or (not top and len(below) <= 4 and max(cells) <= 4096 and sum(cells) <= 4680)
    for _ in range(2):
        u = L.sweep(u, f)
    fc = L.restrict(u, f)
    uc = _vcycle(np.zeros_like(fc), fc, tuple(2 * a for a in h), per, False, inside)
    u = u + L.prolong(uc)
    for _ in range(2):
        u = L.sweep(u, f)
    return u


# (nz, ny, nx): one tile, partial tiles on every axis, several tiles of 4 and
# of 8 planes (512 tiles of 8 planes and more), two levels only; last levels of 17 x
# 18 x 25, 25 x 21 x 33 and 5 x 33 x 40 cells (more than a block holds).  Other last
# levels have even axes or at most 64 cells: on an odd axis that wraps two cells of one
# colour are neighbours, and the in-place sweeps of a block of several waves take
# them in no fixed order.
@pytest.mark.parametrize("shape", [(4, 8, 32), (4, 12, 72), (12, 12, 24), (40, 24, 32),
                                   (128, 64, 256), (6, 10, 6), (34, 36, 50), (50, 42, 66),
                                   (10, 66, 80)])
@pytest.mark.parametrize("per", [(1, 1, 1), (1, 0, 1), (0, 0, 0)])
def test_vcycles_equal_restatement(shape, per):
    f, = rand_fields(shape, 1, seed=71)
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
        # The mean's last bit may differ with the order of its sum; two cycles
        # pass a change of one ulp of the mean on as at most a few of u.
        assert np.abs(u - ref).max() <= 1e-5 * np.abs(ref).max()


# Levels of one block whose cells of a colour do not meet: axes that wrap are even.
@pytest.mark.parametrize("shape,per", [((36, 30, 48), (1, 0, 0)), ((20, 60, 98), (0, 1, 0)),
                                       ((16, 24, 90), (0, 1, 1))])
def test_one_block_last_level(shape, per):
    f, = rand_fields(shape, 1, seed=73)
    f = f.astype(F)
    u = np.zeros(shape, F)
    capi.multigrid(u, f, (0.1, 0.12, 0.11), per, 2)
    f = f - F(f.astype(np.float64).sum() / f.size)
    ref = np.zeros(shape, F)
    for _ in range(2):
        ref = _vcycle(ref, f, (0.1, 0.12, 0.11), per)
    # As above: the mean's last bit.
    assert np.abs(u - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("solver,shape", [("0000", (16, 16, 64)), ("0011", (24, 40, 72)),
                                          ("111111", (16, 12, 16))])
def test_v11_solves(orc, solver, shape):
    q, = rand_fields(shape, 1, seed=72)
    d = (0.3, 0.32, 0.35)
    rhs = -orc.residual(q, np.zeros(shape), d, solver)
    p = np.zeros(shape)
    cycles, rmax = capi.poisson_multigrid(p, rhs, d, solver, npre=1, npost=1, tol=1e-9,
                                          max_cycles=200)
    assert rmax < 1e-9 and np.abs(orc.residual(p, rhs, d, solver)).max() < 1.01e-9
    assert cycles < 200
