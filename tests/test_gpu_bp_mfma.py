"""GPU: the matrix-core form of the fused back-projection (mr_bp_mfma.hip).

Fused plans with more than 16 slices and at least 1.5e9 voxel-projection
updates run it.  Its sums differ from the float kernel's by rounding only:
relRMSE <= 1e-6 of the range against the oracle, the bound of the fused mode
(a product of two 22-bit operands is off by at most 2^-21, and that times
the sums of positive weights stays below the float sums' own rounding,
sqrt(n_proj) 2^-24).  Sizes sit at the edges of its tiles: widths that are
no multiple of 4, 16 or 32, slice counts around multiples of 16 and 64 and
not multiples of 4, projection counts that are no multiple of 4, 16 x 16 and
32 x 32 voxel tiles, centres that put part of the volume outside the detector.
"""
import numpy as np
import pytest
import torch

from conftest import rel_err

pytestmark = pytest.mark.gpu

# width, slices, projections, centre offset, direction, tile
CASES = [(701, 17, 241, 1.25, 0, 16),
         (514, 33, 202, -37.5, 1, 16),
         (512, 64, 101, 0.0, 0, 16),
         (403, 65, 163, 61.0, 1, 16),
         (640, 98, 47, -3.75, 0, 16),
         (1041, 19, 801, 2.5, 0, 32),
         (770, 66, 803, -55.25, 1, 32)]


def _case(seed, nu, nv, n_p):
    rng = np.random.default_rng(seed)
    proj = rng.normal(size=(n_p, nv, nu)).astype(np.float32)
    ang = (np.arange(n_p, dtype=np.float32) * np.float32(180.0 / n_p)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n_p).astype(np.float32)
    return proj, ang, w


def _plan(nu, nv, center, direction=0, fused=True):
    from imagingsuite_amd.recon import BackProjector
    return BackProjector("MultiProjBPparallel", nu, nv, center, direction=direction, buffer_size=0, fused=fused)


@pytest.mark.parametrize("nu,nv,n_p,off,direction,tile", CASES)
def test_mfma_matches_oracle(orc, dev, nu, nv, n_p, off, direction, tile):
    proj, ang, w = _case(nu + nv, nu, nv, n_p)
    bp = _plan(nu, nv, nu / 2 + off, direction)
    t = torch.from_numpy(proj).to(dev)
    vol = bp.process(t, ang, w)
    assert bp.kernel == f"bp_mfma_kernel tile={tile}"
    ref = orc.bp_parallel_f32(proj, ang, w, nu / 2 + off, direction, "linear", 0, False)
    got = vol.cpu().numpy()
    err = rel_err(got, ref)[0]
    print(f"{bp.kernel} {nu}x{nv}x{n_p}: relRMSE vs oracle {err:.2e}")
    assert err <= 1e-6
    # outside the circle and above the last group of four slices nothing is written but zeros
    first, second = bp.mask
    inside = (np.arange(nu)[None, :] >= first[:, None]) & (np.arange(nu)[None, :] < second[:, None])
    assert float(np.abs(got[~inside]).max()) == 0.0
    if nv % 4:
        assert float(np.abs(got[:, :, nv // 4 * 4:]).max()) == 0.0
    # the same bits on a second call
    assert torch.equal(bp.process(t, ang, w), vol)


def test_mfma_slices_scaled_apart(orc, dev):
    """Each slice has a scale of its own: slices 2^-60 to 2^60 apart keep the
    relative bound, slices of zeros stay zero."""
    nu, nv, n_p = 520, 20, 300
    proj, ang, w = _case(5, nu, nv, n_p)
    factor = np.float32(2.0) ** np.linspace(-55, 60, nv).astype(np.int32)
    factor[7] = 0.0
    scaled = proj * factor[None, :, None].astype(np.float32)
    bp = _plan(nu, nv, nu / 2 + 0.5)
    base = bp.process(torch.from_numpy(proj).to(dev), ang, w).cpu().numpy()
    got = bp.process(torch.from_numpy(scaled).to(dev), ang, w).cpu().numpy()
    assert bp.kernel.startswith("bp_mfma_kernel")
    # powers of two: the same bits, scaled
    assert np.array_equal(got, base * factor[None, None, :])


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 2.0 ** 90, 2.0 ** -80])
def test_mfma_unsplittable_samples(dev, monkeypatch, bad):
    """Samples that do not fit the split (not finite; a slice whose largest
    magnitude is far outside the exponent range) give the float kernel's
    bits: the plan with 64-bit staging, which never runs on the matrix cores."""
    nu, nv, n_p = 513, 18, 330
    proj, ang, w = _case(9, nu, nv, n_p)
    if np.isfinite(bad) and abs(bad) < 1:
        proj[:, 3, :] *= np.float32(bad)
    else:
        proj[11, 3, 200] = bad
        proj[300, 16, 0] = bad
    t = torch.from_numpy(proj).to(dev)
    bp = _plan(nu, nv, nu / 2 - 1.5)
    got = bp.process(t, ang, w)
    monkeypatch.setenv("MR_BP_STAGE64", "1")
    valu = _plan(nu, nv, nu / 2 - 1.5)
    ref = valu.process(t, ang, w)
    assert valu.kernel.startswith("bp_lds_kernel")
    assert torch.equal(got.view(torch.int32), ref.view(torch.int32))
    # and the plan goes on with ordinary samples afterwards
    monkeypatch.delenv("MR_BP_STAGE64")
    ok = torch.from_numpy(_case(9, nu, nv, n_p)[0]).to(dev)
    again = bp.process(ok, ang, w)
    assert float((again - valu.process(ok, ang, w)).abs().max()) <= 1e-5 * float(again.abs().max())


def test_mfma_batch_with_unsplittable_stack(dev):
    """A fused batch of matrix-core stacks, stacks below the rule and one
    stack with an infinity: every volume has the bits of its single-stack
    plan, in the persistent launch, its graph replays (eager work between
    them) and the sequential launches."""
    from imagingsuite_amd.recon import BatchReconstructor, ProjectionFilterSingle, fbp_parallel
    stacks = []
    for i, (nu, nv, n_p) in enumerate([(517, 35, 203), (96, 20, 61), (512, 17, 350), (401, 70, 161), (640, 8, 100)]):
        proj, ang, w = _case(40 + i, nu, nv, n_p)
        if i == 2:
            proj[5, 2, 100] = np.inf
        stacks.append(dict(proj=torch.from_numpy(proj).to(dev), angles=ang, weights=w, center=nu / 2 + i - 2.0,
                           filtertype="Hanning", buffer_size=0))
    singles = []
    for s in stacks:
        n_p, nv, nu = s["proj"].shape
        bp = _plan(nu, nv, s["center"])
        vol = torch.empty((nu, nu, nv), dtype=torch.float32, device=dev)
        singles.append(fbp_parallel(ProjectionFilterSingle(nu, "Hanning"), bp, s["proj"].clone(), s["angles"],
                                    s["weights"], vol))
    br = BatchReconstructor(stacks, tune=False, fused=True)

    def check(what):
        torch.cuda.synchronize()
        for i, v in enumerate(br.volumes):
            assert torch.equal(v.view(torch.int32), singles[i].view(torch.int32)), (what, i)
            v.fill_(-1.0)
        torch.cuda.synchronize()

    br.run()
    check("persistent")
    br.run_sequential()
    check("sequential")
    st = torch.cuda.Stream(device=dev)
    for rep in range(3):
        with torch.cuda.stream(st):
            br.run_graph(stream=st)
        check(f"graph {rep}")
    br.close()
