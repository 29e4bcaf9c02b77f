"""GPU: the matrix-core back-projection when a slice's samples differ widely.

Its samples hold an absolute 2^-40 of their slice's largest, so one value far above
the others (a sentinel for a dead pixel) would take bits from every other sample
of the slice.  Slices with more than a sixteenth of their samples below 2^-17 of
the largest run on the vector kernel.

Voxels whose rays all miss the large samples do not depend on them: their values
are compared with 64-bit sums of the same float samples at the same float
positions, relative to the range of these voxels: at most 2e-6 (each kernel is
within 1e-6 of the oracle, test_gpu_bp_mfma.py, whose own sums are off by as much).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

NU, NV = 512, 20


def _process(monkeypatch, vector, t, ang, w, offset=0.0):
    from imagingsuite_amd.recon import BackProjector
    monkeypatch.setenv("MR_BP_STAGE64", "1" if vector else "0")
    bp = BackProjector("MultiProjBPparallel", NU, NV, NU / 2 + offset, buffer_size=0, fused=True)
    out = bp.process(t, ang, w)
    assert bp.kernel.startswith("bp_lds_kernel" if vector else "bp_mfma_kernel")
    return out


def _stack(seed, n_p, kind, dev):
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(n_p, NV, NU)) if kind == "normal" else rng.uniform(0.5, 1.5, (n_p, NV, NU))
    ang = (np.arange(n_p) * (180.0 / n_p)).astype(np.float32)
    return torch.from_numpy(x.astype(np.float32)).to(dev), ang, np.full(n_p, 1.0 / n_p, np.float32)


def _sums64(orc, t, ang, w):
    """Sums in 64 bits of the weighted float samples at the kernels' float positions."""
    dev = t.device
    sn, cs, su = (torch.from_numpy(np.asarray(a)) for a in orc.bp_tables_f32(ang, 0, NU / 2, NU))
    y = torch.arange(1, NU + 1, device=dev, dtype=torch.float32)[:, None]
    x = torch.arange(1, NU + 1, device=dev, dtype=torch.float32)[None, :]
    vol = torch.zeros((NU, NU, NV), device=dev, dtype=torch.float64)
    for k in range(len(ang)):
        u = (su[k].to(dev) + cs[k].to(dev) * y) - sn[k].to(dev) * x
        n = u.to(torch.int64)
        ok = (n >= 0) & (n <= NU - 2)
        n = n.clamp(0, NU - 2)
        f = (u.double() - n.double()).abs()
        f = torch.where(ok, f, torch.zeros_like(f))[..., None]
        row = (t[k] * float(w[k])).double().t().contiguous()   # [column][slice]
        vol += ok[..., None] * row[n] * (1.0 - f) + row[n + 1] * f
    return vol


def _inside(radius, dev):
    y, x = torch.meshgrid(torch.arange(NU, device=dev), torch.arange(NU, device=dev), indexing="ij")
    return (x - NU / 2) ** 2 + (y - NU / 2) ** 2 < radius ** 2


@pytest.mark.parametrize("kind", ["normal", "positive"])
@pytest.mark.parametrize("power", [8, 14, 17, 20, 24, 30, 40, 60])
@pytest.mark.parametrize("where", ["one", "column"])
def test_a_value_far_above_the_others(orc, dev, monkeypatch, kind, power, where):
    n_p = 320
    t, ang, w = _stack(power, n_p, kind, dev)
    # column 2 (slice 5): in one projection, or in every one as a dead pixel's marker
    if where == "one":
        t[100, 5, 2] = 2.0 ** power
    else:
        t[:, 5, 2] = 2.0 ** power
    got = _process(monkeypatch, False, t, ang, w)
    valu = _process(monkeypatch, True, t, ang, w)
    ref = _sums64(orc, t, ang, w)
    free = _inside(NU / 2 - 8, dev)   # column 2 is never within their reach
    b = ref[free]
    span = float(b.max() - b.min())
    err, err_v = (float((a[free].double() - b).pow(2).mean(0).sqrt().max()) / span for a in (got, valu))
    print(f"{kind} 2^{power} {where}: relative rms {err:.2e}, vector kernel {err_v:.2e}", flush=True)
    on_matrix_cores = not torch.equal(got, valu)
    if power >= 20:   # every ordinary sample of the slice is below 2^-17 of it: the vector kernel's bits
        assert not on_matrix_cores
    if power <= 8:
        assert on_matrix_cores
    if on_matrix_cores:
        assert err <= 2e-6 and err <= err_v


def test_one_heavy_projection(dev, monkeypatch):
    """A weight of 2^30 on one projection: all other samples times weights are small."""
    t, ang, w = _stack(1, 320, "normal", dev)
    w = w.copy()
    w[7] *= 2.0 ** 30
    assert torch.equal(_process(monkeypatch, False, t, ang, w), _process(monkeypatch, True, t, ang, w))


def test_a_tenth_far_below(dev, monkeypatch):
    """A band of columns at 2^-25 of the rest: more than a sixteenth, the vector kernel's bits."""
    t, ang, w = _stack(2, 320, "positive", dev)
    t[:, :, 200:255] *= 2.0 ** -25
    assert torch.equal(_process(monkeypatch, False, t, ang, w), _process(monkeypatch, True, t, ang, w))


@pytest.mark.parametrize("kind", ["normal", "positive", "sparse"])
def test_ordinary_samples_stay_on_the_matrix_cores(dev, monkeypatch, kind):
    t, ang, w = _stack(3, 320, "normal" if kind == "normal" else "positive", dev)
    if kind == "sparse":   # mostly exact zeros, a few values a thousand times the others
        t[:, :, :400] = 0.0
        t[::7, :, 405:407] *= 1000.0
    a, b = _process(monkeypatch, False, t, ang, w), _process(monkeypatch, True, t, ang, w)
    assert not torch.equal(a, b)
    span = float(b.max() - b.min())
    assert float((a - b).double().pow(2).mean().sqrt()) / span <= 2e-6
