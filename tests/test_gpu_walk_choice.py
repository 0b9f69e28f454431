"""Geometries whose rays the run walk leaves to the step walk, wholly or in part: volumes past the 2 GiB that a buffer
load reaches, and slices thin against the rise of a plane step.

Past 2 GiB there is no oracle in reasonable time: a few slices of random voxels around the axis in otherwise empty
volumes of 8103 slices (the run walk) and 8105 (the step walk) are compared with the same slices alone.  The three sum the
same ~300 FP32 terms of one sign in different orders, 6e-8 of the running sum each: sqrt(300) * 6e-8 = 1e-6, held to 5e-6 of
the largest.  The thin slices are compared with the FP64 oracle at the tolerances of the other geometries: 1e-4 relative
for projections, 1e-4 of the largest gradient."""
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


def geometry(N, s, Nz, t, H, W, pixnum, nmat, angles, z_reg=0.0):
    ang = np.deg2rad(np.asarray(angles, float))
    k = 10.0 / (0.05 * (pixnum / H))
    cs, sn, xc, yc = O.trig_table_proj(W, H, ang, np.full(len(ang), ((W - H) / 2.0 + 0.3) / k), np.zeros(len(ang)),
                                       det_pixel_num=pixnum)
    return O.Geometry(N=N, s=s, Nz=Nz, t=t, H=H, W=W, cos_t=cs, sin_t=sn, xc=xc, yc=yc, z_reg=z_reg,
                      det_pixel_num=pixnum, nmat=nmat)


def projector(g):
    from virtualcbct_amd.projector import Projector
    return Projector(g.N, g.s, g.Nz, g.t, g.H, g.W, g.n_ang, g.cos_t, g.sin_t, g.xc, g.yc, g.x_reg, g.y_reg, g.z_reg,
                     g.det_pitch, g.det_pitch_iso, g.sad, g.det_pixel_num, g.nmat, 0)


def test_projections_on_either_side_of_the_run_walks_reach(torch):
    N, few = 182, 12  # 182^2 x 8103 records of 8 bytes are within 2^31 bytes, x 8105 past it
    assert N * N * 8103 <= 2 ** 28 < N * N * 8105
    rng = np.random.default_rng(3)
    core = rng.integers(0, 2000, (few, 1, N, N)).astype(np.uint16)
    core[0] = 0  # (slice 0 of a volume is thicker than the others: left empty)
    atten, pdf = np.array([[0.2, 0.3]], np.float32), np.array([0.4, 0.6], np.float32)
    out = {}
    for Nz in (few, 8103, 8105):
        print(Nz, flush=True)
        g = geometry(N, 0.1, Nz, 0.2, 70, 40, 65.0, 1, [-170.0001, -45.0, 9.99999, 100.0])
        P = projector(g)
        vol = torch.zeros((Nz, 1, N, N), dtype=torch.int16, device="cuda")
        z0 = Nz // 2 - few // 2
        vol[z0:z0 + few] = torch.from_numpy(core.view(np.int16)).cuda()
        P.set_volume(vol)
        P.set_spectrum(atten, pdf)
        assert P.forward_channels > 0  # (the channel volume: 8 bytes a voxel)
        out[Nz] = (P.logproj(1000.0).double(), P.forward(1000.0).double())
        P.close()
        del vol
        torch.cuda.empty_cache()
    for Nz in (8103, 8105):
        for a, b in zip(out[Nz], out[few]):
            err = float((a - b).abs().max() / b.abs().max())
            print(f"  {Nz}: {err:.2e}", flush=True)
            assert float(b.abs().max()) > 0 and err < 5e-6


# N, s, Nz, t, H, W, pixnum, z shift
THIN = [
    (32, 0.5, 200, 0.01, 80, 20, 80.0, 0.0),     # on the plane grid, several slice planes in a step
    (30, 0.55, 200, 0.01, 80, 20, 80.0, 0.1),    # off it
    (32, 0.5, 60, 0.045, 130, 16, 120.0, 0.05),  # blocks of one step and of several
    (30, 0.55, 60, 0.045, 130, 16, 120.0, 0.0),
]


@pytest.mark.parametrize("case", THIN, ids=[f"s{c[1]}-t{c[3]}" for c in THIN])
def test_thin_slices_match_fp64_oracle(torch, case):
    print(case, flush=True)
    g = geometry(*case[:7], 2, [-170.0001, -45.0, 9.99999, 100.0], case[7])
    rng = np.random.default_rng(g.N + g.Nz)
    maps = rng.uniform(0.0, 1.0, (2, g.Nz, g.N, g.N)).astype(np.float32)
    atten, pdf = rng.uniform(0.05, 0.4, (2, 5)).astype(np.float32), rng.uniform(0.1, 1.0, 5).astype(np.float32)
    vz = np.ascontiguousarray(maps.transpose(1, 0, 2, 3))
    ref = O.logproj(g, vz, atten, pdf, 1.0)
    target = (0.8 * ref).astype(np.float32)
    rgrad, rloss = O.adjoint(g, vz, atten, pdf, 1.0, target)
    rgrad = rgrad.transpose(1, 0, 2, 3)
    P = projector(g)
    P.set_volume(torch.from_numpy(maps).cuda())
    P.set_spectrum(atten, pdf)
    p = P.logproj(1.0).cpu().numpy()
    grad, loss = P.adjoint(torch.from_numpy(target).cuda(), 1.0)
    gu = P.logproj_backward(torch.from_numpy((2.0 * (ref - target)).astype(np.float32)).cuda(), 1.0)
    P.close()
    scale = np.abs(rgrad).max()
    e = (np.abs(p - ref).max() / np.abs(ref).max(), abs(float(loss) - rloss) / rloss,
         np.abs(grad.cpu().numpy() - rgrad).max() / scale, np.abs(gu.cpu().numpy() - rgrad).max() / scale)
    print("  projection, loss, gradient, backward: " + " ".join(f"{x:.2e}" for x in e), flush=True)
    assert max(e) < 1e-4
