"""The walks with a wave's 64 lanes stepped together on the host.

The ordered run walk (the fused losses' line integrals) is the step table's walk with its additions in the same order: the
FP32 sums must be equal bit for bit, so nothing is tolerated.  Waves whose lanes cross slices in different steps, hand held
pieces over for one another, cross again within a block, run along voxel edges (equal crossing distances, where the block
is cut for one lane's sake), pass the circle's boundary, miss the volume, or stand beyond the panel's last row.

rows_miss may only turn row groups away that charge nothing; it is asked about panels whose row groups end just above,
at and below the volume's slices as its rays see them."""
import ctypes as C
import os

import numpy as np
import pytest

from oracle import oracle as O

HERE = os.path.join(os.path.dirname(__file__), "host_traverse")
LIBS = {"plain": os.path.join(HERE, "libhostwave.so"), "fma": os.path.join(HERE, "libhostwave_fma.so")}
D = C.POINTER(C.c_double)


def load(build):
    if not os.path.exists(LIBS[build]):
        pytest.skip(f"host wave harness not built: {LIBS[build]}")
    lib = C.CDLL(LIBS[build])
    lib.hw_ordered_differences.restype = C.c_long
    lib.hw_rows_miss_charged.restype = C.c_long
    return lib


def geom(N, Nz, s, t, H, W, angles_deg, xs=0.0, z_reg=0.0, x_reg=0.0, ys=0.0, pixnum=800.0):
    ang = np.deg2rad(np.asarray(angles_deg, float))
    k = 10.0 / (0.05 * (pixnum / H))
    cs, sn, xc, yc = O.trig_table_proj(W, H, ang, np.full(len(ang), (W - H) / 2.0 / k + xs), np.full(len(ang), ys),
                                       det_pixel_num=pixnum)
    return O.Geometry(N=N, s=s, Nz=Nz, t=t, H=H, W=W, cos_t=cs, sin_t=sn, xc=xc, yc=yc, z_reg=z_reg, x_reg=x_reg,
                      det_pixel_num=pixnum)


def args(g):
    return [g.N, C.c_double(g.s), g.Nz, C.c_double(g.t), g.H, g.W, g.n_ang, C.c_double(g.x_reg), C.c_double(g.y_reg),
            C.c_double(g.z_reg), C.c_double(g.det_pitch), C.c_double(g.det_pitch_iso), C.c_double(g.sad),
            C.c_double(g.det_pixel_num)]


ANGLES = [-170.0001, -90.00001, 45.0, 59.99999, 133.3, 0.00001]


@pytest.mark.parametrize("build", ["plain", "fma"])
@pytest.mark.parametrize("case", [
    (32, 8, 0.5, 0.5, 24, 12, 0.3, 0.0123, 800.0),
    (32, 8, 0.5, 0.5, 24, 12, 0.0, 0.0, 800.0),        # columns through voxel edges
    (64, 16, 0.25, 0.3, 80, 6, -0.7, 0.3, 300.0),
    (48, 100, 0.2, 0.05, 130, 4, 0.0, 0.0, 260.0),     # thin slices: blocks of one or two steps
    (128, 40, 0.1, 0.1, 100, 3, 0.45, 0.0, 150.0),     # full 64-step tables, several blocks each
    (40, 12, 0.5, 0.25, 64, 8, 0.0, 0.0, 100.0),       # a lattice of equal distances near the axis
    (100, 2, 0.1, 5.0, 65, 3, 0.0, 0.4, 800.0),        # one slice plane (z = 0) only
])
def test_ordered_walk_sums_equal_the_step_walks_bit_for_bit(case, build):
    N, Nz, s, t, H, W, zr, xs, pixnum = case
    lib = load(build)
    g = geom(N, Nz, s, t, H, W, ANGLES, xs, zr, pixnum=pixnum)
    rng = np.random.default_rng(N + Nz)
    tab = np.ascontiguousarray(np.concatenate(g.tables()))
    for vol in (rng.integers(0, 2000, (Nz, 2, N, N)), np.full((Nz, 2, N, N), 1047)):
        v = np.ascontiguousarray(vol, np.uint16)
        for second_first in (0, 1):
            counts = (C.c_long * 2)()
            n = lib.hw_ordered_differences(*args(g), 2, tab.ctypes.data_as(D), v.ctypes.data_as(C.POINTER(C.c_uint16)),
                                           second_first, counts)
            assert counts[0] > 100 and n == 0, (second_first, n, counts[0])


@pytest.mark.parametrize("build", ["plain", "fma"])
def test_ordered_walk_sums_on_random_geometries(build):
    lib = load(build)
    rng = np.random.default_rng(7)
    rays = 0
    for it in range(40):
        N = int(rng.integers(8, 64))
        s = float(rng.choice([0.1, 0.2, 0.25, 0.5, 1.0]))
        Nz = int(rng.integers(1, 40))
        t = float(rng.choice([0.05, 0.1, 0.125, 0.2, 0.5]))
        g = geom(N, Nz, s, t, int(rng.integers(2, 140)), 3, [float(rng.uniform(-180, 180)), 45.0, -90.00001],
                 float(rng.choice([0.0, 0.013, -0.2])), float(rng.choice([0.0, 0.3, -0.45])),
                 float(rng.choice([0.0, 0.25])), pixnum=float(rng.choice([800.0, 200.0, 90.0])))
        v = np.ascontiguousarray(rng.integers(0, 2000, (Nz, 1, N, N)), np.uint16)
        tab = np.ascontiguousarray(np.concatenate(g.tables()))
        counts = (C.c_long * 2)()
        n = lib.hw_ordered_differences(*args(g), 1, tab.ctypes.data_as(D), v.ctypes.data_as(C.POINTER(C.c_uint16)),
                                       it & 1, counts)
        rays += counts[0]
        assert n == 0, (it, N, s, Nz, t, g.H, n, counts[0])
    assert rays > 5000


def test_rows_miss_turns_only_empty_row_groups_away():
    lib = load("plain")
    rng = np.random.default_rng(11)
    told = groups = 0
    for it in range(150):
        N, s = int(rng.integers(8, 80)), float(rng.choice([0.1, 0.25, 0.37, 0.5]))
        Nz, t = int(rng.integers(1, 30)), float(rng.choice([0.05, 0.1, 0.3, 1.0]))
        H = int(rng.choice([65, 130, 200, 400]))
        # the boundary of a row group near the top or bottom slice's projection, a few rows about it
        pixnum = float(rng.choice([100.0, 250.0, 800.0]))
        row = 0.032509752 * pixnum / H
        edge = rng.choice([-1.0, 1.0]) * 0.5 * Nz * t * 100.0 / (100.0 + rng.choice([-0.5, 0.0, 0.5]) * N * s)
        k = 10.0 / (0.05 * (pixnum / H))
        at = edge / row + 64.0 * rng.integers(-1, 2) + rng.uniform(-3.0, 3.0)  # rows from the panel's centre
        g = geom(N, Nz, s, t, H, 3, [float(rng.uniform(-180, 180)), 45.0], 0.1, float(rng.choice([0.0, 0.4, -2.0])),
                 float(rng.choice([0.0, 0.3])), float((at % 64) / k), pixnum)
        tab = np.ascontiguousarray(np.concatenate(g.tables()))
        counts = (C.c_long * 2)()
        bad = lib.hw_rows_miss_charged(*args(g), tab.ctypes.data_as(D), counts)
        told, groups = told + counts[0], groups + counts[1]
        assert bad == 0, (it, bad, N, s, Nz, t, H)
    assert 0.05 * groups < told < 0.95 * groups
