"""Small parallel-beam grids: 4- and 8-slice tiles.

With 32 projections or more, a grid of few blocks takes tiles of 4 or 8 slices
(unrolled, chunks of 16 projections).  Sizes on both sides of each line of the
rule, with remainders in slices, projections and tiles, against the oracle: bit
for bit in reference order (both interpolations), relRMSE <= 1e-6 in fused mode;
and the kernel that the plan reports before and after the tables.
"""
import numpy as np
import pytest
import torch

from conftest import rel_err

pytestmark = pytest.mark.gpu

# width, slices, projections, template arguments after the plan has its tables
SHAPES = [(64, 1, 32, "4,0,{},16,1"),
          (100, 18, 71, "4,0,{},16,1"),
          (64, 13, 31, "8,0,{},16,0"),
          (256, 8, 65, "4,0,{},16,1"),
          (256, 9, 65, "8,0,{},16,1"),
          (250, 21, 66, "8,0,{},16,1"),
          (300, 15, 129, "8,0,{},16,1"),
          (336, 17, 64, "8,0,{},16,1"),
          (500, 7, 70, "8,0,{},16,0"),
          (500, 8, 70, "8,0,{},16,1"),
          (513, 16, 66, "16,0,{},8,1")]


@pytest.mark.parametrize("mode", ["exact", "fused", "nearest"])
@pytest.mark.parametrize("nu,nv,n_p,kernel", SHAPES)
def test_small_grids(orc, dev, nu, nv, n_p, kernel, mode):
    from imagingsuite_amd.recon import BackProjector
    rng = np.random.default_rng(nu + nv + n_p)
    proj = rng.normal(size=(n_p, nv, nu)).astype(np.float32)
    ang = (np.arange(n_p, dtype=np.float32) * np.float32(180.0 / n_p)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n_p).astype(np.float32)
    c = nu / 2 - 1.25
    bp = BackProjector("NearestNeighborBP" if mode == "nearest" else "MultiProjBPparallel", nu, nv, c, buffer_size=0,
                       fused=mode == "fused")
    before = bp.kernel
    vol = bp.process(torch.from_numpy(proj).to(dev), ang, w).cpu().numpy()
    print(f"{nu}x{nv}x{n_p} {mode}: {before} -> {bp.kernel}", flush=True)
    assert before == BackProjector("NearestNeighborBP" if mode == "nearest" else "MultiProjBPparallel", nu, nv, c,
                                   fused=mode == "fused").kernel
    args = kernel.format("false" if mode == "fused" else "true")
    if mode == "nearest":
        args = args.replace(",0,", ",1,", 1)
    assert bp.kernel.startswith(f"bp_lds_kernel<{args}>")
    ref = orc.bp_parallel_f32(proj, ang, w, c, 0, "nearest" if mode == "nearest" else "linear", 0, False)
    if mode == "fused":
        assert rel_err(vol, ref)[0] <= 1e-6
    else:
        assert np.array_equal(vol, ref), int((vol != ref).sum())
