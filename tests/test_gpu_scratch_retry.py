"""Allocations of the library's own give back the scratch it keeps between calls
before they fail: a network is created on a device whose last memory that scratch
holds."""
import numpy as np
import pytest

from osinco3d_amd import capi, warmstart

pytestmark = pytest.mark.gpu


def test_network_takes_the_kept_scratch():
    import torch
    lib = capi.load()
    lib.o3d_release_scratch()
    # Idle scratch of about 0.8 GB: the tendency and the sums of a 100 M-node field.
    phi = torch.zeros((100, 1000, 1000), dtype=torch.float64, device="cuda")
    f = torch.zeros((1,) + phi.shape, dtype=torch.float64, device="cuda")
    capi.transeq(phi, [phi, phi, phi], phi, f, 100.0, 0.7, [0.01] * 3, [0.0] * 3, [0.0] * 3, 1, 1,
                 (0.1, 0.2, 0.3), 0, None, (0, 0, 0))
    del phi, f
    torch.cuda.empty_cache()
    # A 96x96x48 network takes about 0.6 GB; leave less than that free.
    warmstart.Network(16, 16, 16).close()
    hold, left = [], torch.cuda.mem_get_info()[0]
    for _ in range(4):  # memory of the calls before comes back with a delay
        if left <= 256 << 20:
            break
        hold.append(torch.empty(left - (192 << 20), dtype=torch.uint8, device="cuda"))
        left = torch.cuda.mem_get_info()[0]
    print(f"left free {left >> 20} MB")
    assert left <= 256 << 20
    net = warmstart.Network(96, 96, 48)
    x = torch.zeros((2, 96 * 96 * 48), dtype=torch.float32, device="cuda")
    out = torch.empty_like(x[0])
    net.forward(x, out)
    assert np.isfinite(float(out.sum()))
    net.close()
    del hold
    torch.cuda.empty_cache()
    lib.o3d_release_scratch()


# The SOR solve asks for three fields of scratch and does with two, for an even and an
# odd number of launches; the multigrid solve for three FP32 fields and the levels (3.4
# fields of 64 MiB) and does with one less.
def test_solves_with_a_field_less_of_scratch():
    import torch
    lib = capi.load()
    g = torch.Generator(device="cuda").manual_seed(80)
    rhs = torch.rand((256, 256, 256), generator=g, dtype=torch.float64, device="cuda") - 0.5
    runs = [((0.3, 0.35, 0.4), 1.6, 1e-30, kmax, 0, "0000") for kmax in (5, 8)]
    ref = [torch.zeros_like(rhs) for _ in runs]
    want = [capi.poisson(p, rhs, *args) for p, args in zip(ref, runs)]
    mg = ((0.3, 0.35, 0.4), "0000")
    ref.append(torch.zeros_like(rhs))
    want.append(capi.poisson_multigrid(ref[2], rhs, *mg, tol=0.0, max_cycles=2))
    p = [torch.zeros_like(rhs) for _ in ref]
    torch.cuda.synchronize()
    lib.o3d_release_scratch()
    torch.cuda.empty_cache()
    hold, left = [], torch.cuda.mem_get_info()[0]
    for _ in range(4):
        if left <= 380 << 20:  # a field is 128 MiB
            break
        hold.append(torch.empty(left - (350 << 20), dtype=torch.uint8, device="cuda"))
        left = torch.cuda.mem_get_info()[0]
    print(f"left free {left >> 20} MB")
    assert 260 << 20 < left <= 380 << 20
    got = [capi.poisson(a, rhs, *args) for a, args in zip(p, runs)]
    lib.o3d_release_scratch()
    left = torch.cuda.mem_get_info()[0]
    hold.append(torch.empty(left - (190 << 20), dtype=torch.uint8, device="cuda"))
    print(f"then {torch.cuda.mem_get_info()[0] >> 20} MB")
    assert torch.cuda.mem_get_info()[0] < 216 << 20
    got.append(capi.poisson_multigrid(p[2], rhs, *mg, tol=0.0, max_cycles=2))
    del hold
    torch.cuda.empty_cache()
    assert got == want
    for a, b in zip(p, ref):
        assert torch.equal(a, b)
    lib.o3d_release_scratch()
