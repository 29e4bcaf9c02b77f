"""Slice tiles of the back-projection's adjoint: 32 slices a line at a time, 16,
8 and 4 two lines at a time, with partial last tiles.

A slice's sums do not depend on the slices beside it, so the adjoint of nv slices
equals, bit for bit, that of its slices in groups of 4.  Widths are odd and even
(the last step of two lines is then half empty), slices at or beyond 4 (nv / 4)
get no gradient.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["MultiProjBPparallel", "NearestNeighborBP"])
@pytest.mark.parametrize("nu,nv", [(2, 8), (33, 12), (64, 20), (101, 45), (90, 64), (57, 7)])
def test_tiles_equal_groups_of_four(dev, name, nu, nv):
    from imagingsuite_amd.recon import BackProjector
    n_p = 50
    rng = np.random.default_rng(nu + nv)
    ang = (np.arange(n_p) * 7.3).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n_p).astype(np.float32)
    g = torch.from_numpy(rng.standard_normal((nu, nu, nv)).astype(np.float32)).to(dev)
    print(f"adjoint tiles {name} {nu} {nv}", flush=True)
    got = BackProjector(name, nu, nv, nu / 2 + 0.4, buffer_size=0).adjoint(g, ang, w)
    assert got.shape == (n_p, nv, nu)
    part = BackProjector(name, nu, 4, nu / 2 + 0.4, buffer_size=0)
    for z in range(0, nv // 4 * 4, 4):
        ref = part.adjoint(g[:, :, z:z + 4].contiguous(), ang, w)
        assert torch.equal(got[:, z:z + 4], ref), z
    assert not got[:, nv // 4 * 4:].any()
    if nu > 2:
        assert bool(got.any())
