"""The network's padding is periodic, so moving input and target by 8 voxels (one voxel
of the coarsest level) leaves every gradient as it is but for the order of its FP32
sums: activations and their gradients are the same values at other places.  A tap, run
or wrapped neighbour left out at an edge shows as the share of the voxels it serves
(one column of 40: 9 %).

Bound: FP32 sums of n = 15360 terms of random sign are off by 2^-24 sqrt(n / 2) = 5e-6
of their norm; 1e-3 leaves room for sums that cancel to a part in 200."""
import pytest

from osinco3d_amd import warmstart

pytestmark = pytest.mark.gpu

LAYERS = [(16, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128),
          (128, 64), (64, 64), (64, 32), (32, 32), (32, 16), (16, 16)]


@pytest.mark.parametrize("shift", [(0, 0, 8), (0, 0, 16), (0, 8, 0), (8, 0, 0), (8, 16, 24)])
def test_gradients_do_not_move(shift):
    import torch
    nz, ny, nx = 16, 24, 40
    gen = torch.Generator(device="cuda").manual_seed(79)
    inp = torch.randn((2, nz, ny, nx), generator=gen, device="cuda")
    tgt = torch.randn((nz, ny, nx), generator=gen, device="cuda")

    def grads(by):
        net = warmstart.Network(nx, ny, nz, 3)
        x = torch.roll(inp, by, (1, 2, 3)).reshape(2, -1).contiguous()
        t = torch.roll(tgt, by, (0, 1, 2)).reshape(-1).contiguous()
        out, d = torch.empty_like(t), torch.empty_like(t)
        net.zero_grad()
        net.forward(x, out)
        net.mse(out, t, d)
        net.backward(d)
        g = torch.from_numpy(net.grads()).double()
        net.close()
        return g

    a, b = grads((0, 0, 0)), grads(shift)
    at = 0
    for li, (ci, co) in enumerate(LAYERS):
        for what, n in (("weights", co * 27 * ci), ("bias", co)):
            off = float((a[at:at + n] - b[at:at + n]).norm() / a[at:at + n].norm())
            at += n
            assert off <= 1e-3, (li, what, off)
    assert float((a[at:] - b[at:]).norm() / a[at:].norm()) <= 1e-3
