"""Intensities of rays through ever thicker objects, to exponents past the FP32 exponential's range, for spectra of any
scale (photon counts as well as a normalised pdf): two bins whose terms leave that range one after the other.  Against the
FP64 oracle: an FP32 line integral's 3e-7 times an exponent of up to 100 is 3e-5, held to 1e-4 as other projections."""
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


@pytest.mark.parametrize("scale", [1e-9, 1.0, 1e6, 1e12])
@pytest.mark.parametrize("nmat", [1, 6])
def test_opaque_rays_of_any_spectrum_scale(torch, scale, nmat):
    from virtualcbct_amd.projector import Projector
    N, s, Nz, t, H, W = 32, 0.5, 4, 0.5, 24, 60
    pixnum = 0.9 * N * s / 0.032509752 * H / W  # (columns over nine tenths of the volume's width)
    ang = np.deg2rad(np.array([-170.0001, -100.0, -40.00001, 9.99999, 30.0, 77.0]))
    k = 10.0 / (0.05 * (pixnum / H))
    cs, sn, xc, yc = O.trig_table_proj(W, H, ang, np.full(len(ang), ((W - H) / 2.0 + 0.3) / k), np.zeros(len(ang)),
                                       det_pixel_num=pixnum)
    g = O.Geometry(N=N, s=s, Nz=Nz, t=t, H=H, W=W, cos_t=cs, sin_t=sn, xc=xc, yc=yc, det_pixel_num=pixnum, nmat=nmat)
    vol = np.full((Nz, nmat, N, N), 1000, np.uint16)
    # exponents up to ~97 in the first bin (2^-140) over a 16 cm chord, 2 % less in the second
    mu = 97.0 / (nmat * 16.0)
    atten = np.tile(np.array([[mu, 0.98 * mu]], np.float32), (nmat, 1))
    pdf = np.array([scale, scale], np.float32)
    ref = O.forward_collapsed(g, vol, atten, pdf, 1000.0).astype(np.float64)
    P = Projector(N, s, Nz, t, H, W, len(ang), cs, sn, xc, yc, 0.0, 0.0, 0.0, 0.05, 0.032509752, 100.0, pixnum, nmat, 0)
    P.set_volume(vol)
    P.set_spectrum(atten, pdf)
    out = P.forward(1000.0).double().cpu().numpy()
    P.close()
    seen = ref > 1e-36  # (normal FP32 values)
    err = np.abs(out - ref)[seen] / ref[seen]
    print(f"{int(seen.sum())} of {ref.size} rays, down to {ref[seen].min():.1e}, error {err.max():.2e}", flush=True)
    assert ref[seen].min() < 1e-34 * max(scale, 0.1) and err.max() < 1e-4
