"""The slice-run walk (virtualcbct_amd/csrc/runs.h), compiled for the host, against the per-lane step walk of the same
build over the forms it accepts: pitches on and off the plane grid, thin and thick slices (blocks of 1 to 64 steps,
and slices thinner than a step's rise, which keep the step walk), z shifts (rays that cross z = 0), panel shifts
(central rays through voxel edges: equal crossing distances), odd sizes, near-axis and diagonal angles.  (On an axis
exactly, where many rays run along lattice edges, either walk's voxels are decided by the last rounding.)"""
import ctypes as C
import os

import numpy as np
import pytest

from oracle import oracle as O

HERE = os.path.join(os.path.dirname(__file__), "host_traverse")
LIBS = {"plain": os.path.join(HERE, "libhostruns.so"), "fma": os.path.join(HERE, "libhostruns_fma.so")}
D = C.POINTER(C.c_double)
# both walks charge the same cells; a length is rounded to FP32 once in each (6e-8), the sums are FP64
TOL = 2.5e-7


def line_integrals(lib, g, vol, runs):
    if not os.path.exists(lib):
        pytest.skip(f"host run-walk harness not built: {lib}")
    f = C.CDLL(lib).hr_line_integrals
    f.restype = C.c_long
    tab = np.ascontiguousarray(np.concatenate(g.tables()))
    L = np.zeros((g.n_ang, g.H, g.W, g.nmat))
    v = np.ascontiguousarray(vol, np.uint16)
    n = f(g.N, C.c_double(g.s), g.Nz, C.c_double(g.t), g.H, g.W, g.n_ang, C.c_double(g.x_reg), C.c_double(g.y_reg),
          C.c_double(g.z_reg), C.c_double(g.det_pitch), C.c_double(g.det_pitch_iso), C.c_double(g.sad),
          C.c_double(g.det_pixel_num), g.nmat, tab.ctypes.data_as(D), v.ctypes.data_as(C.POINTER(C.c_uint16)),
          L.ctypes.data_as(D), int(runs))
    return L, n


def geom(N, Nz, s, t, H, W, angles_deg, xs=0.0, z_reg=0.0, x_reg=0.0):
    ang = np.deg2rad(np.asarray(angles_deg, float))
    xs = xs - (H - W) / 2.0 * (0.05 * 800.0 / H) / 10.0  # a panel that is not square stays centred on the axis
    cs, sn, xc, yc = O.trig_table_proj(W, H, ang, np.full(len(ang), xs), np.zeros(len(ang)))
    return O.Geometry(N=N, s=s, Nz=Nz, t=t, H=H, W=W, cos_t=cs, sin_t=sn, xc=xc, yc=yc, z_reg=z_reg, x_reg=x_reg)


def compare(lib, g, seed, expect_runs=None):
    """Largest relative error per ray of the run walk and of its two ordered forms; the run walk's waves."""
    vol = np.random.default_rng(seed).integers(0, 2000, (g.Nz, g.nmat, g.N, g.N)).astype(np.uint16)
    Lb, _ = line_integrals(lib, g, vol, 0)
    err, taken = 0.0, 0
    for form in (1, 2, 3):
        La, n = line_integrals(lib, g, vol, form)
        if form == 1:
            taken = n
            if expect_runs is not None:
                assert (n > 0) == expect_runs
        err = np.maximum(err, np.abs(La - Lb).sum(-1) / np.maximum(np.abs(Lb).sum(-1), 1e-9))
    return err, taken


ANGLES = [-170.0001, -90.00001, -40.00001, 9.99999, 45.0, 59.99999, 133.3, 179.99999, 0.00001, 90.0001]


@pytest.mark.parametrize("build", ["plain", "fma"])
@pytest.mark.parametrize("case", [
    (32, 8, 0.5, 0.5, 24, 24, 0.3, 0.0123, True),
    (32, 8, 0.5, 0.5, 24, 24, 0.0, 0.0, True),        # columns through voxel edges
    (64, 16, 0.25, 0.3, 80, 70, -0.7, 0.3, True),
    (48, 100, 0.2, 0.05, 130, 20, 0.0, 0.0, True),  # thin slices: blocks of one or two steps
    (24, 320, 1.0, 0.01, 64, 20, 0.0, 0.0, False),    # several planes within one step: the step walk everywhere
    (41, 9, 0.37, 0.21, 33, 29, 0.11, -0.2, True),    # planes off the voxel grid
    (16, 4, 0.8, 1.2, 14, 14, 0.0, 0.01, True),       # every midpoint of a whole step a tie
    (128, 40, 0.1, 0.1, 200, 9, 0.45, 0.0, True),     # full 64-step tables, several blocks each
    (300, 2, 0.09765625, 5.0, 65, 7, 0.0, 0.4, True),  # one slice plane (z = 0) only
])
def test_run_walk_equals_step_walk(case, build):
    N, Nz, s, t, H, W, zr, xs, runs = case
    err, _ = compare(LIBS[build], geom(N, Nz, s, t, H, W, ANGLES, xs, zr), N + Nz, runs)
    assert err.max() < TOL, np.unravel_index(err.argmax(), err.shape)


@pytest.mark.parametrize("build", ["plain", "fma"])
def test_run_walk_random_geometries(build):
    rng = np.random.default_rng(4242)
    took = 0
    for it in range(150):
        N = int(rng.integers(8, 72))
        s = float(rng.choice([0.05, 0.1, 0.2, 0.25, 0.3, 0.4, 0.5, 0.8, 1.0, 0.37, 0.09765625]))
        Nz = int(rng.integers(1, 40))
        t = float(rng.choice([0.05, 0.1, 0.125, 0.2, 0.5, 1.0, 0.33]))
        H, W = int(rng.integers(2, 140)), int(rng.integers(2, 24))
        ang = list(rng.uniform(-180, 180, 5)) + [-90.00001, 45.0, 179.99999]
        g = geom(N, Nz, s, t, H, W, ang, float(rng.choice([0.0, 0.013, -0.2, 1.15])),
                 float(rng.choice([0.0, 0.3, -0.45, 0.1])), float(rng.choice([0.0, 0.25])))
        err, n = compare(LIBS[build], g, it)
        took += n > 0
        assert err.max() < TOL, (it, N, s, Nz, t, H, W, np.unravel_index(err.argmax(), err.shape), err.max())
    assert took > 100
