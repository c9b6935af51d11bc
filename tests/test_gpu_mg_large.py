"""The multigrid solve of a grid whose FP32 fields exceed the 2 GiB that the pair
kernel's buffer descriptors address: a periodic problem made of copies of a small one
has copies of its solution, bit for bit, as the small one's pair kernel leaves it."""
import pytest

from osinco3d_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npre,npost", [(2, 1), (1, 1)])
def test_copies_beyond_two_gib(npre, npost):
    import torch
    if torch.cuda.mem_get_info()[0] < 32 << 30:
        pytest.skip("needs 32 GiB of device memory")
    g = torch.Generator(device="cuda").manual_seed(76)
    shape, copies = (64, 32, 128), (8, 32, 8)
    rhs = torch.rand(shape, generator=g, dtype=torch.float64, device="cuda") - 0.5
    p = torch.zeros_like(rhs)
    # Two levels: deeper ones would end on other grids.
    kw = dict(npre=npre, npost=npost, tol=0.0, max_cycles=1, nlevels=2, with_reason=True)
    d = (0.3, 0.32, 0.35)
    small = capi.poisson_multigrid(p, rhs, d, "0000", **kw)
    big_rhs = rhs.repeat(copies)
    assert big_rhs.numel() == 1 << 29
    big = torch.zeros_like(big_rhs)
    assert capi.poisson_multigrid(big, big_rhs, d, "0000", **kw) == small
    del big_rhs
    tiles = big.reshape(8, 64, 32, 32, 8, 128)
    for a in range(8):
        assert bool((tiles[a] == p.reshape(64, 1, 32, 1, 128)).all())
    del big, tiles
    capi.load().o3d_release_scratch()
    torch.cuda.empty_cache()
