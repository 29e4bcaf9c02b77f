"""GPU: which fused stacks run on the matrix cores, and what their ragged ends hold.

The rule asks for about two blocks per CU in each launch, so stacks of small
width stay with the vector kernel whatever their depth (with fewer blocks the
matrix-core form took up to 3 times as long).  Slice counts whose last group of
four ends a tile leave the one to three slices past it to that tile.  Values are
compared with the vector kernel's: both stay within 1e-6 of the range of the
oracle (test_gpu_bp_mfma.py, test_gpu_bp_kernels.py), so 2e-6 of each other.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# width, slices, projections, whether on the matrix cores
RULE = [(128, 100, 916, False), (256, 80, 287, False), (150, 200, 334, False), (64, 1024, 358, False),
        (256, 32, 720, False), (300, 64, 261, False), (330, 36, 400, False), (350, 24, 511, False),
        (400, 20, 500, True), (350, 32, 409, True), (350, 36, 350, True), (350, 64, 192, True), (350, 80, 154, True), (256, 128, 179, True),
        (200, 256, 147, True)]


@pytest.mark.parametrize("nu,nv,n_p,mfma", RULE)
def test_rule(dev, nu, nv, n_p, mfma):
    from imagingsuite_amd.recon import BackProjector
    bp = BackProjector("MultiProjBPparallel", nu, nv, nu / 2, buffer_size=0, fused=True)
    ang = (np.arange(n_p) * (180.0 / n_p)).astype(np.float32)
    bp.process(torch.zeros((n_p, nv, nu), dtype=torch.float32, device=dev), ang, np.ones(n_p, np.float32))
    print(f"{nu} {nv} {n_p} {bp.kernel}", flush=True)
    assert bp.kernel.startswith("bp_mfma_kernel") == mfma


@pytest.mark.parametrize("nu,nv,n_p", [(641, 17, 240), (641, 19, 240), (520, 33, 180), (520, 35, 180), (520, 50, 130),
                                       (520, 65, 100), (520, 67, 100)])
def test_ragged_ends(dev, monkeypatch, nu, nv, n_p):
    from imagingsuite_amd.recon import BackProjector
    rng = np.random.default_rng(nv)
    t = torch.from_numpy(rng.normal(size=(n_p, nv, nu)).astype(np.float32)).to(dev)
    ang = (np.arange(n_p) * (180.0 / n_p)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n_p).astype(np.float32)
    vols = []
    for vector in ("0", "1"):
        monkeypatch.setenv("MR_BP_STAGE64", vector)
        bp = BackProjector("MultiProjBPparallel", nu, nv, nu / 2 + 1.25, buffer_size=0, fused=True)
        vol = torch.full((nu, nu, nv), 5.0, dtype=torch.float32, device=dev)
        bp.process(t, ang, w, volume=vol)
        assert bp.kernel.startswith("bp_lds_kernel" if vector == "1" else "bp_mfma_kernel")
        vols.append(vol)
    assert not vols[0][:, :, nv // 4 * 4:].any()
    span = float(vols[1].max() - vols[1].min())
    err = float((vols[0] - vols[1]).double().pow(2).mean().sqrt()) / span
    assert err <= 2e-6, err
    # samples that do not fit the split: the vector kernel, the same ends (the float sinogram has more slices
    # than the split one here)
    t[3, nv - 1, 7] = float("inf")
    t[5, 2, 9] = float("nan")
    monkeypatch.setenv("MR_BP_STAGE64", "0")
    a = BackProjector("MultiProjBPparallel", nu, nv, nu / 2 + 1.25, buffer_size=0, fused=True).process(t, ang, w)
    monkeypatch.setenv("MR_BP_STAGE64", "1")
    b = BackProjector("MultiProjBPparallel", nu, nv, nu / 2 + 1.25, buffer_size=0, fused=True).process(t, ang, w)
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))


def test_plan_reports_the_last_call(dev):
    """Accumulating calls run on the vector kernel, and the plan says so."""
    from imagingsuite_amd.recon import BackProjector
    nu, nv, n_p = 512, 32, 200
    bp = BackProjector("MultiProjBPparallel", nu, nv, nu / 2, buffer_size=0, fused=True)
    t = torch.ones((n_p, nv, nu), dtype=torch.float32, device=dev)
    ang, w = np.arange(n_p, dtype=np.float32), np.ones(n_p, np.float32)
    vol = bp.process(t, ang, w)
    assert bp.kernel.startswith("bp_mfma_kernel")
    bp.process(t, ang, w, volume=vol, accumulate=True)
    assert bp.kernel.startswith("bp_lds_kernel")
    bp.process(t, ang, w, volume=vol)
    assert bp.kernel.startswith("bp_mfma_kernel")
