"""The tile scatter against the ray-ordered one (fixed by set_adjoint_tile) in what a sum in any order has in common: the
voxels that no ray charges hold exactly 0, and an infinite or undefined upstream gradient reaches the voxels that its
ray charges and no others.  One map without a basis, so that the gradient is the scattered channel itself; grids on and
off the plane grid, thin slices (a plane in most blocks), the circle's boundary in view.

The upstream gradient is positive, so a charged voxel's gradient is; the forms may differ in segments shorter than the
geometry's rounding (1e-12 of a voxel), hence voxels whose gradient is below 1e-7 of the largest are left out of the second
comparison and must be below that in both of the first."""
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


# N, s, Nz, t, H, W, angles, pixnum
CASES = [(64, 0.25, 33, 0.25, 100, 120, 60, 800.0), (61, 0.3, 20, 0.33, 130, 90, 60, 500.0),
         (96, 0.2, 70, 0.05, 200, 64, 40, 800.0), (64, 0.2, 40, 0.1, 128, 128, 60, 300.0)]


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-s{c[1]}-t{c[3]}" for c in CASES])
def test_tile_scatter_charges_the_same_voxels(torch, case):
    from virtualcbct_amd.projector import Projector
    N, s, Nz, t, H, W, nA, pixnum = case
    print(case, flush=True)
    rng = np.random.default_rng(17)
    ang = np.deg2rad(-180.0 + 360.0 / nA * np.arange(nA) + 1e-5)
    k = 10.0 / (0.05 * (pixnum / H))
    cs, sn, xc, yc = O.trig_table_proj(W, H, ang, np.full(nA, ((W - H) / 2.0 + 0.3) / k), np.zeros(nA),
                                       det_pixel_num=pixnum)
    P = Projector(N, s, Nz, t, H, W, nA, cs, sn, xc, yc, 0.0, 0.0, 0.1, 0.05, 0.032509752, 100.0, pixnum, 1, 0)
    P.set_spectrum(np.array([[0.2]], np.float32), np.array([1.0], np.float32))
    P.set_volume(torch.from_numpy(rng.uniform(0.1, 1.0, (1, Nz, N, N)).astype(np.float32)).cuda())
    _, L = P.logproj_save(1.0)

    def both(gp):
        P.set_adjoint_tile(1, 4, 0, 0)
        a = P.logproj_backward_saved(L, gp, 1.0).cpu().numpy()
        P.set_adjoint_tile(0)
        return a, P.logproj_backward_saved(L, gp, 1.0).cpu().numpy()

    gp = torch.from_numpy(rng.uniform(0.2, 1.0, P.shape_proj).astype(np.float32)).cuda()
    gp[:, :, 3::7] = 0.0
    gp[nA // 3:] = 0.0  # a few angles: many voxels of one or two rays
    ref, got = both(gp)
    tiny = 1e-7 * ref.max()
    off = (ref == 0.0) != (got == 0.0)
    print(f"  charged {int((ref != 0).sum())} of {ref.size}, in one form only {int(off.sum())}", flush=True)
    assert (got >= 0.0).all() and np.maximum(ref, got)[off].max(initial=0.0) < tiny
    for value in (float("inf"), float("nan")):
        bad = gp.clone()
        bad[1, ::9, 2::7] = value
        b_ref, b_got = both(bad)
        clear = (np.maximum(ref, got) > tiny) | ((ref == 0.0) & (got == 0.0))
        m = np.isfinite(b_ref) != np.isfinite(b_got)
        print(f"  {value}: reaches {int((~np.isfinite(b_ref)).sum())} voxels, differs at {int((m & clear).sum())}", flush=True)
        assert (~np.isfinite(b_ref)).any() and not (m & clear).any()
    P.close()
