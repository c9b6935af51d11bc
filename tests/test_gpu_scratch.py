"""Scratch kept between calls: results do not depend on what a block held
before, the idle blocks are bounded, and o3d_release_scratch gives them back."""
import numpy as np
import pytest

from osinco3d_amd import capi
from tests.helpers import rand_fields

pytestmark = pytest.mark.gpu


def _call(torch, shape, seed):
    phi, src = rand_fields(shape, 2, seed=seed)
    u = rand_fields(shape, 3, seed=seed + 1)
    g = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    p, f = g(np.clip(phi, 0, 1)), torch.zeros((3,) + shape, dtype=torch.float64, device="cuda")
    capi.transeq(p, [g(a) for a in u], g(src), f, 100.0, 0.7, [0.01] * 3, [0.0] * 3, [0.0] * 3, 1,
                 1, (0.1, 0.2, 0.3), 0, None, (0, 0, 0))
    return p.cpu().numpy(), f.cpu().numpy()


def test_kept_blocks_do_not_show_in_results():
    import torch
    lib = capi.load()
    shapes = [(12, 20, 40), (30, 40, 50), (12, 20, 40), (13, 21, 33)]
    lib.o3d_release_scratch()
    fresh = []
    for s, shape in enumerate(shapes):
        fresh.append(_call(torch, shape, 80 + s))
        assert lib.o3d_release_scratch() == 0
    kept = [_call(torch, shape, 80 + s) for s, shape in enumerate(shapes)]
    for a, b in zip(fresh, kept):
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


def test_idle_blocks_are_bounded_and_given_back():
    import torch
    lib = capi.load()
    _call(torch, (16, 16, 16), 90)
    lib.o3d_release_scratch()
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    phi = torch.zeros((160, 400, 400), dtype=torch.float64, device="cuda")  # 205 MB a field
    f = torch.zeros((1,) + phi.shape, dtype=torch.float64, device="cuda")
    used = free0 - torch.cuda.mem_get_info()[0]
    for n in (400, 200, 100, 64, 40, 30):
        v = phi.reshape(-1)[: 160 * 400 * n].reshape(160, 400, n)
        capi.transeq(v, [v, v, v], v, f.reshape(-1), 100.0, 0.7, [0.01] * 3, [0.0] * 3, [0.0] * 3,
                     1, 1, (0.1, 0.2, 0.3), 0, None, (0, 0, 0))
    held = free0 - torch.cuda.mem_get_info()[0] - used
    assert 0 < held <= (1 << 30) + (64 << 20)
    lib.o3d_release_scratch()
    assert free0 - torch.cuda.mem_get_info()[0] - used <= 64 << 20
