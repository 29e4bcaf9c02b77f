"""GPU: mr_bp_parallel_noalloc on tall fused stacks, which it takes in slabs of slices.

Where fewer than 32 projections fit the fixed scratch the matrix-core form runs
slab by slab; the volume equals mr_bp_parallel's bit for bit, whatever the
slabs' ends, and so does that of samples which do not fit the split (the vector
kernel, without slabs).
"""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# slabs of 448, of 448 (the last slice past the last group), of 576; one slab
@pytest.mark.parametrize("nu,nv,n_p", [(1024, 600, 41), (1030, 513, 36), (640, 1603, 33), (512, 200, 33)])
@pytest.mark.parametrize("bad", [False, True])
def test_slabs_equal_plan(dev, nu, nv, n_p, bad):
    import imagingsuite_amd._lib as L
    from imagingsuite_amd.recon import BackProjector
    lib = L.load()
    rng = np.random.default_rng(nv)
    t = torch.randn((n_p, nv, nu), device=dev, generator=torch.Generator(device=dev).manual_seed(nv))
    if bad:
        t[7, nv - 2, 100] = float("inf")
    ang = (np.arange(n_p) * (180.0 / n_p)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n_p).astype(np.float32)
    center = nu / 2 + 1.5
    bp = BackProjector("MultiProjBPparallel", nu, nv, center, buffer_size=0, fused=True)
    ref = bp.process(t, ang, w)
    assert bp.kernel.startswith("bp_mfma_kernel")
    p = L.BpParams()
    p.width, p.slices, p.center, p.fused = nu, nv, center, 1
    got = torch.full((nu, nu, nv), 5.0, dtype=torch.float32, device=dev)
    fp = ctypes.POINTER(ctypes.c_float)
    print(f"noalloc slabs {nu} {nv} {n_p} {bad}", flush=True)
    rc = lib.mr_bp_parallel_noalloc(ctypes.byref(p), t.data_ptr(), n_p, ang.ctypes.data_as(fp), w.ctypes.data_as(fp),
                                    got.data_ptr(), 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.mr_last_error()
    assert torch.equal(got.view(torch.int32), ref.view(torch.int32))
