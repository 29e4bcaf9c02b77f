"""The slice-lane FDK back-projection (lanes = slices, the detector window of an
8 x 8 patch of voxel columns staged in LDS) against the column kernel, which a
plan made under MR_FDK_COLUMN=1 keeps: bit-identical volumes.

Sizes: whole and ragged 256-slice groups (a group of 224 slices or more is
padded, a shorter rest goes to the column kernel), widths that leave partial
patches, windows far taller and shorter than the slab's shadow (rows outside
count as zero), slabs at the first detector rows (where r + 0.5 is rounded
before the floor), an off-centre axis, an ROI mask, anisotropic voxels, a
window around no row at all, and calls that stay with the column kernel.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# width, (row0, row1) of the slab, window rows, projections, changes to the
# geometry, whether the slice-lane kernel takes part
CASES = [
    (512, (0, 256), 256, 9, {}, True),
    (520, (40, 345), 330, 8, {"direction": 1}, True),
    (601, (0, 230), 241, 9, {"center": 4.25}, True),
    (513, (0, 224), 224, 8, {"matrix_roi": (20, 9, 377, 490)}, True),
    (512, (0, 223), 224, 8, {}, False),
    (511, (0, 256), 256, 8, {}, False),
    (530, (0, 512), 37, 7, {}, True),
    (514, (0, 300), 700, 7, {"voxel": (0.13, 0.09, 0.05), "filter": "shepp-logan", "cosine_weight": True}, True),
    (512, (0, 256), 11, 6, {"ppoint": (250.5, -3.0)}, True),
    (520, (0, 256), 255, 10, {"sod": 150.0, "sdd": 300.0}, True),
    (520, (0, 256), 255, 10, {"sod": 60.0, "sdd": 300.0}, False),
]


def _plan(width, rows, kw):
    from imagingsuite_amd.recon import FDKbp_single
    kw = dict(kw)
    center = width / 2 + kw.pop("center", 0.0)
    args = (kw.pop("sod", 500.0), kw.pop("sdd", 1000.0), (0.2, 0.2), kw.pop("voxel", (0.1, 0.1, 0.1)),
            kw.pop("ppoint", (width / 2, (rows[0] + rows[1]) / 2)), center, (0, rows[0], width, rows[1]),
            max(rows[1], width) - 1)
    return FDKbp_single(*args, **kw)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("width,rows,win,n_p,geometry,lanes", CASES)
def test_slice_lanes_equal_column_threads(dev, monkeypatch, fused, width, rows, win, n_p, geometry, lanes):
    print(f"fdk slice lanes {width} {rows} {win} {n_p} {geometry} fused={fused}", flush=True)
    kw = dict(geometry, fused=fused)
    g = torch.Generator().manual_seed(width + win)
    proj = torch.randn((n_p, win, width), generator=g) + 1.0
    angles = (np.arange(n_p) * (360.0 / n_p) + 0.3).astype(np.float32)
    weights = np.linspace(0.5, 1.5, n_p).astype(np.float32) / n_p
    monkeypatch.delenv("MR_FDK_COLUMN", raising=False)
    a = _plan(width, rows, kw)
    monkeypatch.setenv("MR_FDK_COLUMN", "1")
    b = _plan(width, rows, kw)
    from imagingsuite_amd import _lib
    for _ in range(2):   # the second call reuses the plan's copy of the projections
        pa, pb = proj.to(dev), proj.to(dev)
        _lib.profile(True)
        _lib.profile_reset()
        va = a.process(pa, angles, weights, volume=torch.full((a.nz, width, width), 7.0, device=dev))
        launches = _lib.profile_query("fdk_transpose")[1]
        _lib.profile(False)
        assert launches == int(lanes)   # the copy only the slice-lane kernel needs
        vb = b.process(pb, angles, weights, volume=torch.full((a.nz, width, width), -3.0, device=dev))
        assert float(vb.abs().max()) > 0
        assert torch.equal(va, vb), int((va != vb).sum())
        assert torch.equal(pa, pb)
