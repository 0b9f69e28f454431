"""The filter's cosine weight to FP32.  Rows of equal content, one in two so that they fill the same half of their pairs' packed
signals, have the same convolution bit for bit and differ by the weight alone: the ratio of two such outputs is that of
their weights, each product rounded once.  A correctly rounded weight and its product are 2.5e-8 rms each (an ulp over
the square root of 12, averaged over a binade), 5.0e-8 for a ratio; a weight an ulp off on top is 6.5e-8.  Held to
5.7e-8."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as T
    if not T.cuda.is_available():
        pytest.skip("no GPU")
    return T


@pytest.mark.parametrize("W", [300, 400, 512, 700])  # block filter, wave filter, block filter
def test_cosine_weight_is_rounded_about_once(torch, W):
    from virtualcbct_amd import fdk
    H, n = 512, 2
    rng = np.random.default_rng(W)
    row = rng.uniform(0.1, 1.0, W).astype(np.float32)
    proj = torch.from_numpy(np.broadcast_to(row, (n, H, W)).copy()).cuda()
    out = fdk.filter_sinogram_device(proj, np.zeros(n), np.zeros(n)).double().cpu().numpy()
    pitch = 0.032509752 * 800.0 / W
    # the tables' FP32 positions
    xc = yc = np.float32(-W / 2.0 - 1.0)  # (both centres by the width, F/filterSinogram.cpp:86-87)
    pos1 = np.abs(xc + np.arange(W, dtype=np.float32)) * np.float32(pitch)
    pos2 = np.abs(yc + np.arange(H, dtype=np.float32)) * np.float32(pitch)
    cm = 100.0 / np.sqrt(1e4 + pos1[None, :].astype(np.float64) ** 2 + pos2[:, None].astype(np.float64) ** 2)
    flat = out / cm[None]
    rows = flat[:, 0::2]
    ratio = rows[:, 1:] / rows[:, :1] - 1.0
    rms = float(np.sqrt((ratio ** 2).mean()))
    print(f"W {W}: ratio off by {rms:.2e} rms, {np.abs(ratio).max():.2e} at most", flush=True)
    assert rms < 5.7e-8
