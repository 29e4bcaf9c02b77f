"""The staged Joseph projector pair on every slice count: against the same
geometry with the slices split over calls that take the other kernels.

A slice's sums do not depend on the slices beside it, so projecting a volume of
nz slices must equal, bit for bit, projecting its slices in groups of 4 through
the direct kernels (a grid of few blocks or tiles takes them: the reference
projects few angles, or a few voxel rows, at a time) - and slice counts that are
multiples of 16 must equal the same slices inside a larger multiple.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _geometry(nx, nz, n_det, ang):
    from recon_autograd import Geometry
    return Geometry(nx, nz, n_det, ang, nx / 2 + 0.7)


# 8-, 16- and 32-slice tiles with rests, odd widths, both stepping classes
@pytest.mark.parametrize("nx,nz,n_ang", [(300, 4, 100), (260, 8, 130), (257, 12, 100), (350, 20, 130), (350, 36, 97),
                                         (170, 44, 90)])
def test_any_slice_count_equals_direct_kernels(dev, nx, nz, n_ang):
    print(f"joseph staged {nx} {nz} {n_ang}", flush=True)
    ang = (np.arange(n_ang) * (180.0 / n_ang) + 0.1).astype(np.float32)
    nd = nx + 5
    g = torch.Generator().manual_seed(nx + nz)
    vol = torch.randn((nx, nx, nz), generator=g).to(dev)
    sino = torch.randn((n_ang, nd, nz), generator=g).to(dev)
    fwd = _geometry(nx, nz, nd, ang).forward(vol)
    adj = _geometry(nx, nz, nd, ang).adjoint(sino)
    # direct forward kernel: 4 slices of 3 angles at a time (fewer than 128 blocks)
    for z in range(0, nz, 4):
        part = vol[:, :, z:z + 4].contiguous()
        for i in range(0, n_ang, 3):
            ref = _geometry(nx, 4, nd, ang[i:i + 3]).forward(part)
            assert torch.equal(fwd[i:i + 3, :, z:z + 4], ref), (z, i)
    # direct adjoint kernel: 4 slices (fewer than 512 tiles at these widths;
    # the whole of 350^2 x 20 and x 36 is staged)
    assert ((nx + 15) // 16) ** 2 < 512
    for z in range(0, nz, 4):
        ref = _geometry(nx, 4, nd, ang).adjoint(sino[:, :, z:z + 4].contiguous())
        assert torch.equal(adj[:, :, z:z + 4], ref), z


@pytest.mark.parametrize("nx,n_ang", [(129, 50), (256, 33)])
def test_slice_tiles_agree(dev, nx, n_ang):
    """16 slices (two lines per barrier) against the same slices among 48 and 32."""
    ang = (np.arange(n_ang) * (180.0 / n_ang) + 0.1).astype(np.float32)
    vol = torch.randn((nx, nx, 96), generator=torch.Generator().manual_seed(nx)).to(dev)
    out = {}
    for nz in (16, 32, 48, 96):
        out[nz] = _geometry(nx, nz, nx, ang).forward(vol[:, :, :nz].contiguous())
    for nz in (16, 32, 48):
        assert torch.equal(out[nz], out[96][:, :, :nz]), nz


@pytest.mark.parametrize("nz", [4, 8])
def test_adjoint_eight_slice_tiles(dev, nz):
    """368^2 has 529 tiles: 8-slice tiles against the same slices among 16."""
    nx, n_ang = 368, 21
    ang = (np.arange(n_ang) * (180.0 / n_ang) + 0.1).astype(np.float32)
    sino = torch.randn((n_ang, nx + 1, 16), generator=torch.Generator().manual_seed(nz)).to(dev)
    part = _geometry(nx, nz, nx + 1, ang).adjoint(sino[:, :, :nz].contiguous())
    assert torch.equal(part, _geometry(nx, 16, nx + 1, ang).adjoint(sino)[:, :, :nz])
