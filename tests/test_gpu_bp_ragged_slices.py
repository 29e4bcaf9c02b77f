"""Slice counts that no slice tile divides: the last tile's rest.

The slices past the last whole group of four belong to the last tile that has
one; tiles of 16 and 32 slices store what whole vectors do not fit through LDS;
a stack of one group of four runs 4-slice tiles at every grid size.  Counts on
both sides of the tiles' edges, widths that are no multiple of 16, every module
and its tilt branch, bit for bit against the oracle; accumulation leaves the
slices that no group holds as they are.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# width, slices, projections: tiles of 8 (one group: 4), 8, 16 and 32 slices
SHAPES = [(530, 4, 35), (500, 5, 20), (530, 7, 33), (500, 11, 33), (530, 13, 21), (515, 17, 33), (515, 19, 20),
          (520, 31, 9), (515, 33, 18), (530, 35, 7), (515, 50, 10), (515, 67, 6)]


@pytest.mark.parametrize("name", ["MultiProjBPparallel", "MultiProjBP", "NearestNeighborBP"])
@pytest.mark.parametrize("nu,nv,n_p", SHAPES)
def test_ragged_slices_bitexact(orc, dev, nu, nv, n_p, name):
    from imagingsuite_amd.recon import BackProjector
    rng = np.random.default_rng(nu + nv)
    proj = rng.normal(size=(n_p, nv, nu)).astype(np.float32)
    ang = np.sort(rng.uniform(0, 180, n_p)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n_p).astype(np.float32)
    c = nu / 2 + 0.75
    bp = BackProjector(name, nu, nv, c, buffer_size=0)
    vol = torch.full((nu, nu, nv), 9.0, dtype=torch.float32, device=dev)
    bp.process(torch.from_numpy(proj).to(dev), ang, w, volume=vol)
    ref = orc.bp_parallel_f32(proj, ang, w, c, 0, "nearest" if name == "NearestNeighborBP" else "linear", 0,
                              name == "MultiProjBP")
    print(f"{bp.kernel} {nu} {nv} {n_p}", flush=True)
    assert np.array_equal(vol.cpu().numpy(), ref)
    # a second half added on: the sums go on, the slices without a group stay
    half = n_p // 2
    vol.fill_(9.0)
    bp.process(torch.from_numpy(proj[:half]).to(dev), ang[:half], w[:half], volume=vol)
    assert not vol[:, :, nv // 4 * 4:].any()
    vol[:, :, nv // 4 * 4:] = 3.0
    bp.process(torch.from_numpy(proj[half:]).to(dev), ang[half:], w[half:], volume=vol, accumulate=True)
    got = vol.cpu().numpy()
    assert np.array_equal(got[:, :, :nv // 4 * 4], ref[:, :, :nv // 4 * 4])
    assert bool((got[:, :, nv // 4 * 4:] == 3.0).all())


@pytest.mark.parametrize("name", ["MultiProjBPparallel", "MultiProjBP", "NearestNeighborBP"])
@pytest.mark.parametrize("nu,nv,n_p", [(260, 4, 18), (100, 20, 18), (530, 36, 6)])
def test_tilt_groups_equal_their_padded_stack(dev, nu, nv, n_p, name):
    """A stack with up to three more slices gives the tilt branch the same groups of four."""
    from imagingsuite_amd.recon import BackProjector
    rng = np.random.default_rng(nv)
    ang = np.sort(rng.uniform(0, 180, n_p)).astype(np.float32)
    w = np.ones(n_p, np.float32)
    full = torch.from_numpy(rng.normal(size=(n_p, nv + 3, nu)).astype(np.float32)).to(dev)
    kw = dict(buffer_size=0, correct_tilt=True, tilt_angle=0.4, tilt_pivot=nv / 2, tilt_rows=nv)
    ref = BackProjector(name, nu, nv, nu / 2, **kw).process(full[:, :nv].contiguous(), ang, w)
    for extra in (1, 3):
        if name == "MultiProjBP":
            break   # its second column lies 4 (nv / 4) on: another layout
        got = BackProjector(name, nu, nv + extra, nu / 2, **kw).process(full[:, :nv + extra].contiguous(), ang, w)
        assert torch.equal(got[:, :, :nv], ref), extra
        assert not got[:, :, nv:].any()
