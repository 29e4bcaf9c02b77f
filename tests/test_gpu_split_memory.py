"""GPU: calls whose fast form needs a copy that does not fit the device's free memory.

The matrix-core form pads slices to 16 (20 slices: 32, float samples 20).  Where
only the float samples fit, plans and batches run on the vector kernel, with its
bits, instead of failing.  An FDK plan that had no room for its transposed
projections makes the copy at the next call that has.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

NU, NV, NP = 1024, 20, 2400
FLOAT = 4 * NP * NU * 20          # bytes of the float sinogram
SPLIT = 4 * NP * NU * 32          # of the split one (118 MB more)
SLACK = 32 << 20                  # tables, filter plans, allocation granularity


def _fits(dev, n):
    try:
        x = torch.empty(n, dtype=torch.uint8, device=dev)
    except torch.OutOfMemoryError:
        return False
    del x
    torch.cuda.empty_cache()
    return True


def _squeeze(dev, fits, fails):
    """Takes the device's memory until an allocation of `fails` bytes does not succeed, one of `fits` does."""
    torch.cuda.empty_cache()
    held = []
    while True:   # most of it at once (what is reported free can lag behind)
        have, _total = torch.cuda.mem_get_info(dev)
        if have - fails < (256 << 20):
            break
        held.append(torch.empty(have - fails - (128 << 20), dtype=torch.uint8, device=dev))
    while _fits(dev, fails):
        held.append(torch.empty(16 << 20, dtype=torch.uint8, device=dev))
    assert _fits(dev, fits)
    return held


def _stack(dev):
    t = torch.randn((NP, NV, NU), device=dev, generator=torch.Generator(device=dev).manual_seed(3))
    ang = (np.arange(NP) * (180.0 / NP)).astype(np.float32)
    return t, ang, np.full(NP, 1.0 / NP, np.float32)


def test_plan_falls_back(dev, monkeypatch):
    from imagingsuite_amd.recon import BackProjector
    t, ang, w = _stack(dev)
    vol = torch.empty((NU, NU, NV), dtype=torch.float32, device=dev)
    bp = BackProjector("MultiProjBPparallel", NU, NV, NU / 2, buffer_size=0, fused=True)
    rest = _squeeze(dev, FLOAT + SLACK, SPLIT)
    bp.process(t, ang, w, volume=vol)
    torch.cuda.synchronize()
    del rest
    torch.cuda.empty_cache()
    assert bp.kernel.startswith("bp_lds_kernel")
    monkeypatch.setenv("MR_BP_STAGE64", "1")
    ref = BackProjector("MultiProjBPparallel", NU, NV, NU / 2, buffer_size=0, fused=True)
    assert torch.equal(vol, ref.process(t, ang, w))


def test_batch_falls_back(dev, monkeypatch):
    from imagingsuite_amd.recon import BackProjector, BatchReconstructor, ProjectionFilterSingle
    t, ang, w = _stack(dev)
    small = t[:400, :17].contiguous()
    stacks = [dict(proj=t, angles=ang, weights=w, center=NU / 2, buffer_size=0),
              dict(proj=small, angles=ang[:400], weights=w[:400], center=NU / 2, buffer_size=0)]
    vols = 4 * NU * NU * (NV + 17)
    # volumes (rounded up by the allocator), filtered rows of both stacks and their float samples
    base = vols + 4 * (t.numel() + small.numel()) + 4 * 400 * NU * 20
    rest = _squeeze(dev, base + FLOAT + SLACK, base + SPLIT - SLACK)
    br = BatchReconstructor(stacks, tune=False, fused=True)
    del rest
    torch.cuda.empty_cache()
    assert br.slice_tile != 64   # 64: every stack on the matrix cores
    br.run()
    torch.cuda.synchronize()
    monkeypatch.setenv("MR_BP_STAGE64", "1")
    for s, v in zip(stacks, br.volumes):
        n_p, nv, nu = s["proj"].shape
        f = ProjectionFilterSingle(nu, "Hamming").process(s["proj"].clone())
        ref = BackProjector("MultiProjBPparallel", nu, nv, nu / 2, buffer_size=0, fused=True)
        assert torch.equal(v, ref.process(f, s["angles"], s["weights"]))
    br.close()
    # with room the same stacks run on the matrix cores
    assert BatchReconstructor(stacks, tune=False, fused=True).slice_tile == 64


def test_fdk_plan_takes_its_copy_later(dev):
    from imagingsuite_amd import _lib
    from imagingsuite_amd.recon import FDKbp_single
    n, rows, n_p = 512, 256, 400
    copy = 4 * n_p * n * rows          # without the rows behind the window
    fdk = FDKbp_single(500.0, 1000.0, (0.2, 0.2), (0.1, 0.1, 0.1), (n / 2, rows / 2), n / 2, (0, 0, n, rows), n - 1)
    proj = torch.randn((n_p, rows, n), device=dev, generator=torch.Generator(device=dev).manual_seed(7))
    angles = (np.arange(n_p) * (360.0 / n_p)).astype(np.float32)
    weights = np.full(n_p, 1.0 / n_p, np.float32)
    vols = [torch.empty((rows, n, n), device=dev) for _ in range(2)]
    work = [proj.clone(), proj]
    launches = []
    rest = _squeeze(dev, SLACK, copy)
    for w, v in zip(work, vols):
        _lib.profile(True)
        _lib.profile_reset()
        fdk.process(w, angles, weights, volume=v)
        launches.append(_lib.profile_query("fdk_transpose")[1])
        _lib.profile(False)
        rest = None
        torch.cuda.empty_cache()
    assert launches == [0, 1]
    assert torch.equal(vols[0], vols[1])
