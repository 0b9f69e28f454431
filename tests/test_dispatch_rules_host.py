"""The host-side rules that choose the adjoint's scatter and the projections' kernels, at the geometries measured beside
them, on either side of each line."""
import ctypes as C
import os

import pytest

LIB = os.path.join(os.path.dirname(__file__), "host_traverse", "libhostwave.so")


def harness():
    if not os.path.exists(LIB):
        pytest.skip(f"host wave harness not built: {LIB}")
    return C.CDLL(LIB)


def test_tile_scatter_rule():
    lib = harness()

    def tiles(N, s, Nz, t, H, nA, nch):
        return bool(lib.hw_scatter_by_tiles(N, C.c_double(s), Nz, C.c_double(t), H, H, nA, nch))
    for nch in (1, 2):
        assert tiles(128, 0.2, 32, 0.2, 128, 24, nch) and tiles(256, 0.1, 64, 0.1, 256, 4, nch)
    for nch in (3, 4, 5, 6):  # one angle a block
        assert not tiles(128, 0.2, 32, 0.2, 128, 24, nch) and not tiles(512, 0.05, 256, 0.1, 400, 1, nch)
        assert tiles(64, 0.4, 20, 0.4, 60, 360, nch) and tiles(512, 0.05, 256, 0.1, 400, 8, nch)
    assert not tiles(64, 0.4, 20, 0.4, 60, 24, 1)  # few ray steps
    assert tiles(128, 0.2, 256, 0.025, 128, 48, 2) and not tiles(128, 0.2, 355, 0.018, 128, 48, 2)  # thin slices
    assert tiles(100, 0.26, 128, 0.05, 128, 48, 2) and not tiles(100, 0.26, 213, 0.03, 128, 48, 2)


def test_thin_slice_rule():
    lib = harness()

    def thin(N, s, Nz, t, H):
        return bool(lib.hw_thin(N, C.c_double(s), Nz, C.c_double(t), H, H))
    assert thin(128, 0.2, 533, 0.012, 128) and thin(256, 0.1, 1280, 0.01, 256)
    assert not thin(512, 0.05, 128, 0.1, 400) and not thin(64, 0.3, 12, 0.4, 72) and not thin(24, 0.5, 6, 0.4, 24)
