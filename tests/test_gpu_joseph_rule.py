"""GPU: which Joseph forward projections are staged.

Slice counts that are no multiple of 16 run the staged kernel or the direct one,
which give the same bits.  A staged block is full only where 16 angles share a
chunk; with few angles over a wide volume it holds one, and the direct kernel is
up to three times as fast.  The direct kernel's launches are counted apart.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz,n_ang,direct", [(2048, 4, 30, True), (1024, 4, 60, True), (1024, 12, 20, True),
                                                (700, 4, 90, True), (128, 20, 60, True), (300, 12, 60, True),
                                                (300, 20, 200, False), (400, 4, 360, False), (1024, 12, 180, False),
                                                (512, 24, 90, False), (256, 20, 180, False), (512, 16, 20, False)])
def test_rule(dev, nx, nz, n_ang, direct):
    import imagingsuite_amd._lib as L
    from recon_autograd import Geometry
    ang = (np.arange(n_ang) * (180.0 / n_ang)).astype(np.float32)
    geo = Geometry(nx, nz, nx, ang, nx / 2 + 0.3)
    vol = torch.randn((nx, nx, nz), device=dev)
    L.profile_reset()
    L.profile(True)
    try:
        out = geo.forward(vol)
        torch.cuda.synchronize()
        launches = L.profile_query("joseph_forward_direct")[1]
    finally:
        L.profile(False)
        L.profile_reset()
    print(f"{nx} {nz} {n_ang} direct launches {launches}", flush=True)
    assert (launches > 0) == direct
    # the other kernel's bits: a few angles alone, and the slices among 16
    some = [0, n_ang // 3, n_ang - 1]
    few = Geometry(nx, nz, nx, ang[some], nx / 2 + 0.3).forward(vol)
    assert torch.equal(out[some], few)
