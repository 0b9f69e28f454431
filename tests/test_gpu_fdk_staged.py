"""The LDS-staged backprojector against the plain one, bit for bit: angle counts off the stage of four, slice counts off
the blocks, footprints that fit the tiles, leave the panel, or are too tall or too wide for a tile.  Fixed at four
slices a thread (VCBCT_NO_AUTOTUNE) and as the autotuner picks them; the one-shot and allocation-free calls, which choose
the form by rule, equal both."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# R, Z, n, H, W, zstart, step, scale
CASES = [
    (96, 40, 7, 120, 130, -2, 0.1, 0.1),    # two or three pixels a slice, partial blocks of slices and columns
    (135, 64, 9, 200, 210, -3, 0.1, 0.1),
    (70, 33, 5, 60, 64, -4, 0.2, 0.2),      # rows and columns leave the panel
    (64, 32, 6, 400, 400, -6, 0.4, 0.1),    # slices too far apart for a tile
    (64, 16, 4, 128, 400, -1, 0.05, 0.4),   # columns too far apart for a tile
    (50, 3, 13, 90, 90, 0, 0.1, 0.15),      # fewer slices than a block
]


@pytest.fixture(scope="module")
def torch():
    import torch as T
    if not T.cuda.is_available():
        pytest.skip("no GPU")
    return T


@pytest.mark.parametrize("tune", ["0", "1"])
@pytest.mark.parametrize("case", CASES)
def test_staged_equals_plain_bit_for_bit(torch, monkeypatch, case, tune):
    from virtualcbct_amd import fdk
    R, Z, n, H, W, zstart, step, scale = case
    print(case, "autotuned" if tune == "1" else "four slices", flush=True)
    monkeypatch.setenv("VCBCT_NO_AUTOTUNE", "0" if tune == "1" else "1")
    rng = np.random.default_rng(17)
    ang = np.deg2rad(-180.0 + 360.0 / n * np.arange(n) + 1e-4)
    xs = rng.uniform(-1.5, 1.5, n)
    sino = torch.from_numpy(rng.standard_normal((n, H, W)).astype(np.float32)).cuda()
    recs = []
    for lds in ("0", "1"):
        monkeypatch.setenv("VCBCT_BP_LDS", lds)
        plan = fdk.FdkPlan(H, W, n, R, Z, zstart, step, scale, 1000, ang, xs, np.zeros(n))
        print("  staged", plan.bp_staged, "slices a thread", plan.slices_per_thread, flush=True)
        assert plan.bp_staged == (lds == "1")
        rec = torch.zeros(plan.shape_recon, device="cuda")
        plan.backproject(sino, rec)
        recs.append(rec)
        plan.close()
    rec = torch.zeros_like(recs[0])
    fdk.reconstruct_image_device(rec, sino, zstart, step, scale, 1000, ang, xs)
    recs.append(rec)
    torch.cuda.synchronize()
    assert float(recs[0].abs().max()) > 0
    for r in recs[1:]:
        assert torch.equal(recs[0], r)
