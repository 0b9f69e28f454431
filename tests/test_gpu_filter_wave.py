"""The ramp filter at 1024 points (a wave per row pair, the signal in registers) against the oracle's FP64 filter: the
smallest and largest widths of that length, one row and odd row counts (the last pair has one row), blocks with idle
waves, and a half-fan panel padded into it on either side.  Tolerance as for the other lengths: ~20 FP32 butterfly
levels of 6e-8 against the largest output, 2e-5 with the offset weighting's chain 5e-5."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as T
    if not T.cuda.is_available():
        pytest.skip("no GPU")
    return T


@pytest.mark.parametrize("W,H,n", [(321, 5, 1), (322, 1, 1), (400, 9, 3), (449, 7, 2), (512, 3, 5)])
def test_filter_1024_matches_fp64_oracle(torch, W, H, n):
    from virtualcbct_amd import fdk
    print(W, H, n, flush=True)
    assert fdk.filter_fft_length(W) == 1024
    rng = np.random.default_rng(W)
    proj = rng.uniform(0.02, 1.0, (n, H, W)).astype(np.float32)
    xs, ys = rng.uniform(-7.0, 7.0, n), rng.uniform(-1.0, 1.0, n)
    out = fdk.filter_sinogram_device(torch.from_numpy(proj).cuda(), xs, ys).cpu().numpy()
    ref = O.filter_sinogram(proj, xs, ys, acc64=True)
    err = np.abs(out - ref).max() / np.abs(ref).max()
    print(f"  vs FP64: {err:.3e}")
    assert err < 2e-5


@pytest.mark.parametrize("side", [1.0, -1.0])
def test_half_fan_filter_1024_matches_fp64_oracle(torch, side):
    from virtualcbct_amd import fdk
    rng = np.random.default_rng(8)
    n, H, W = 5, 7, 300
    proj = rng.uniform(0.1, 1.0, (n, H, W)).astype(np.float32)
    ang = np.deg2rad(np.arange(n) * 40.0 - 90.0)
    xs, ys = side * (45.0 + 0.5 * rng.standard_normal(n)) * 40.0 / W, np.full(n, 0.3)
    plan = fdk.FdkPlan(H, W, n, 16, 2, 0, 0.45, 0.4, 1000, ang, xs, ys, half_fan=True)
    print(plan.width, flush=True)
    assert fdk.filter_fft_length(plan.width) == 1024
    filt = plan.filter(torch.from_numpy(proj).cuda()).cpu().numpy()
    pw, xo, yo = O.offset_weight(proj, xs, ys)
    ref = O.filter_sinogram(pw, xo, yo, pitch_iso=0.032509752 * plan.width / W, acc64=True)
    err = np.abs(filt - ref).max() / np.abs(ref).max()
    print(f"  vs FP64: {err:.3e}")
    plan.close()
    assert err < 5e-5
