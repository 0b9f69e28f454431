"""The adjoint's scatter by voxel tiles against the ray-ordered scatter (fixed by set_adjoint_tile), on the same
coefficients: voxel pitches on and off the whole-cm plane grid, odd sizes (partial tiles, partial slice chunks), rows
denser and sparser than the slices, blocks of several slice planes, an offset isocentre, one to five channels, and
the geometries below the tile form's range, which keep the ray-ordered form.

Tolerance: a voxel sums up to ~1e3 FP32 terms of one sign pattern in either form, each rounded to 6e-8 of the running
sum; the orders differ, so the forms differ by at most sqrt(1e3) * 6e-8 = 2e-6 of the largest gradient in the mean
case: 1e-5 as for the ray-ordered form's own tile shapes."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# N, s, Nz, t, H, W, angles, pixnum, channels, (x, y, z) offsets
CASES = [
    (64, 0.25, 33, 0.25, 100, 120, 60, 800.0, 2, (0.0, 0.0, 0.0)),     # planes on voxel boundaries, a chunk of one slice
    (61, 0.3, 20, 0.33, 130, 90, 60, 500.0, 2, (0.2, -0.1, 0.15)),     # planes inside voxels, odd N
    (39, 0.8, 10, 1.0, 100, 111, 110, 710.0, 1, (-0.22, -0.08, 0.1)),  # several slice planes' blocks in a tile
    (96, 0.2, 70, 0.05, 200, 64, 40, 800.0, 1, (0.0, 0.1, -0.3)),      # thin slices: rows three slices apart
    (80, 0.25, 9, 0.5, 150, 70, 60, 150.0, 5, (0.0, 0.0, 0.2)),        # dense rows: fifteen to a slice
    (45, 0.5, 40, 0.05, 128, 128, 64, 600.0, 2, (0.0, 0.0, 0.0)),      # two slice planes in a step: listed columns
    (128, 0.2, 64, 0.2, 65, 129, 48, 800.0, 2, (0.0, 0.0, 0.0)),       # columns through the box corners (45 degrees)
    (12, 0.5, 5, 0.4, 40, 30, 7, 300.0, 2, (0.0, 0.0, 0.1)),           # below the tile form's range
]


@pytest.fixture(scope="module")
def torch():
    import torch as T
    if not T.cuda.is_available():
        pytest.skip("no GPU")
    return T


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-s{c[1]}-t{c[3]}-nch{c[8]}" for c in CASES])
def test_tile_scatter_equals_ray_ordered_scatter(torch, case):
    from virtualcbct_amd.projector import Projector
    N, s, Nz, t, H, W, nA, pixnum, nch, (xr, yr, zr) = case
    print(case, flush=True)
    rng = np.random.default_rng(91)
    ang = np.deg2rad(-180.0 + 360.0 / nA * np.arange(nA) + 1e-5)  # (the diagonals among them)
    k = 10.0 / (0.05 * (pixnum / H))
    cs, sn, xc, yc = O.trig_table_proj(W, H, ang, np.full(nA, (W - H) / 2.0 / k), np.zeros(nA), det_pixel_num=pixnum)
    P = Projector(N, s, Nz, t, H, W, nA, cs, sn, xc, yc, xr, yr, zr, 0.05, 0.032509752, 100.0, pixnum, 6, 0)
    basis = rng.uniform(0.1, 0.5, (6, nch))
    atten = (basis @ rng.uniform(0.2, 1.0, (nch, 7))).astype(np.float32)
    P.set_spectrum(atten, rng.uniform(0.1, 1.0, 7).astype(np.float32))
    P.set_volume(torch.from_numpy(rng.uniform(0.0, 1.0, (6, Nz, N, N)).astype(np.float32)).cuda())
    assert P.adjoint_channels == nch
    _, L = P.logproj_save(1.0)
    gp = torch.from_numpy(rng.uniform(0.2, 1.0, P.shape_proj).astype(np.float32)).cuda()
    gp[:, ::7, ::5] = 0.0
    P.set_adjoint_tile(1, 4, 0, 0)
    ref = P.logproj_backward_saved(L, gp, 1.0).double()
    P.set_adjoint_tile(0)
    scale = float(ref.abs().max())
    assert scale > 0
    for _ in range(2):
        got = P.logproj_backward_saved(L, gp, 1.0).double()
        err = float((got - ref).abs().max()) / scale
        print(f"  max difference {err:.2e} of max |grad|", flush=True)
        assert err < 1e-5
    P.close()
