"""Infinite voxels in FP32 maps: a ray that charges one has an infinite line integral (not finite in the channel
volumes, where a basis weighs the infinity), every other ray the finite one that
the FP64 oracle gives it (1e-5 of the largest: FP32 sums of ~60 terms).  Grids on and off the plane grid, columns through
voxel edges (equal crossing distances), thin slices, rays that cross the circle's boundary beside such a voxel; the maps
themselves and their two- and four-channel volumes."""
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


# N, s, Nz, t, panel shift in pixels, z shift
CASES = [(32, 0.5, 24, 0.2, 0.3, 0.0), (32, 0.5, 24, 0.2, 0.0, 0.0), (30, 0.55, 24, 0.2, 0.3, 0.1),
         (30, 0.55, 24, 0.2, 0.0, 0.0), (32, 0.5, 60, 0.06, 0.3, 0.0)]


@pytest.mark.parametrize("nmat", [2, 4, 6])
@pytest.mark.parametrize("case", CASES, ids=[f"s{c[1]}-t{c[3]}-x{c[4]}" for c in CASES])
def test_infinite_voxels_reach_only_the_rays_that_charge_them(torch, case, nmat):
    from virtualcbct_amd.projector import Projector
    N, s, Nz, t, shift, z_reg = case
    print(case, nmat, flush=True)
    H, W, pixnum = 96, 40, 96.0
    ang = np.deg2rad(np.array([-170.0001, -135.00001, -45.00001, 9.99999, 30.0, 100.0, 157.0]))
    k = 10.0 / (0.05 * (pixnum / H))
    cs, sn, xc, yc = O.trig_table_proj(W, H, ang, np.full(len(ang), ((W - H) / 2.0 + shift) / k), np.zeros(len(ang)),
                                       det_pixel_num=pixnum)
    xc = xc * 12.0  # (columns twelve rows wide: the panel spans the volume)
    g = O.Geometry(N=N, s=s, Nz=Nz, t=t, H=H, W=W, cos_t=cs, sin_t=sn, xc=xc, yc=yc, z_reg=z_reg,
                   det_pixel_num=pixnum, nmat=nmat)
    rng = np.random.default_rng(N + Nz + nmat)
    maps = rng.uniform(0.1, 1.0, (nmat, Nz, N, N)).astype(np.float32)
    mark = np.zeros_like(maps)
    r, n = 0.46 * N, N // 2
    for i in range(14):  # voxels about the rim and the axis, in slices of the central rays
        x, y = (int(n + r * np.cos(0.7 * i)), int(n + r * np.sin(0.7 * i))) if i < 9 else rng.integers(n - 4, n + 4, 2)
        mark[:, int(rng.integers(1, Nz)), y, x] = 1.0
    zm = np.ascontiguousarray(maps.transpose(1, 0, 2, 3))
    charged = O.line_integrals(g, np.ascontiguousarray(mark.transpose(1, 0, 2, 3)))[0]
    assert (charged > 1e-6).any()
    finite = O.line_integrals(g, zm * (1.0 - mark.transpose(1, 0, 2, 3)))[0]
    scale = finite.max()
    P = Projector(N, s, Nz, t, H, W, len(ang), cs, sn, xc, yc, 0.0, 0.0, z_reg, 0.05, 0.032509752, 100.0, pixnum, nmat, 0)
    atten = (np.eye(nmat) + 0.01).astype(np.float32)  # full rank: up to four maps, the channels are the maps
    P.set_spectrum(atten, np.full(nmat, 1.0 / nmat, np.float32))
    maps[mark > 0] = np.inf
    P.set_volume(torch.from_numpy(maps).cuda())
    forms = {"line integrals": P.line_integrals().double().cpu().numpy()}
    if nmat <= 4:
        assert P.forward_channels > 0
        _, L = P.logproj_save(1.0)
        forms["channels"] = np.moveaxis(L.double().cpu().numpy().reshape((nmat, len(ang), H, W)), 0, -1)
    P.close()
    for name, L in forms.items():
        hit, clear = charged > 1e-6, charged == 0.0
        assert (np.isposinf(L[hit]) if name == "line integrals" else ~np.isfinite(L[hit])).all(), name
        assert np.isfinite(L[clear]).all(), name
        err = np.abs(L[clear] - finite[clear]).max() / scale
        print(f"  {name}: {int(hit.sum())} infinite, the others within {err:.1e}", flush=True)
        assert err < 1e-5
