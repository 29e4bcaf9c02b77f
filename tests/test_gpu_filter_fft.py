"""The radix-8 filter line against a double-precision convolution of the same row
with the same impulse response.

Every line length from 64 to 16384 points, in the short form (the row fills at
most half of the line) and as the full padded line, with odd row counts (the last
block holds one row), widths that leave most of the line empty and widths that
fill it.

Bound: one transform of L points rounds each value log2 L times, so the
difference from double is at most about eps (2 log2 L + twiddles 4) of the
line's 2-norm per point in the mean square: 32 eps of the largest value's row
norm covers it ten times over, an index or twiddle mistake exceeds it by orders
of magnitude.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


@pytest.mark.parametrize("rows", [1, 5])
@pytest.mark.parametrize("doubler", [2, 1])
@pytest.mark.parametrize("width", [32, 33, 64, 100, 128, 129, 256, 300, 512, 513, 1024, 1025, 2048, 2049, 4096, 5000,
                                   8192])
def test_filter_line_against_double(dev, width, doubler, rows):
    """paddingdoubler 2: the short form, 1: the full line (and the adjoint of each)."""
    from imagingsuite_amd.recon import ProjectionFilterSingle
    f = ProjectionFilterSingle(width, filtertype="Hamming", paddingdoubler=doubler)
    print(f"{f.kernel} width {width} rows {rows}", flush=True)
    assert f.kernel.endswith(" short") == (doubler == 2)
    rng = np.random.default_rng(width + rows)
    x = rng.standard_normal((rows, width)).astype(np.float32)
    x[:, 0] = x[:, -1] = 0.0                         # no tapers: a plain convolution
    P, ins = f.fft_size, f.n_insert
    h = np.zeros(P)
    h[:P // 2] = f.filter
    h[P // 2] = 1.0
    h[P // 2 + 1:] = f.filter[1:][::-1]
    line = np.zeros((rows, P))
    line[:, ins:ins + width] = x
    ref = np.fft.ifft(np.fft.fft(line, axis=1) * h, axis=1).real[:, ins:ins + width] * P * (np.pi / (2.0 * P))
    bound = 32 * EPS * np.linalg.norm(x, axis=1).max()
    y = f.process(torch.from_numpy(x.copy()).to(dev)).cpu().numpy()
    err = np.abs(y - ref).max()
    print(f"max error {err:.2e}, bound {bound:.2e}")
    assert err <= bound
    # the adjoint's interior is the same convolution (the tapers fold onto the ends)
    z = f.adjoint(torch.from_numpy(x.copy()).to(dev)).cpu().numpy()
    assert np.abs(z[:, 1:-1] - ref[:, 1:-1]).max() <= bound
