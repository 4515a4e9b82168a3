"""The plan of the Lorenzo inverse by tiles (lorenzo_inverse_scratch in
mans_amd/csrc/lorenzo.hip), on the CPU: its scratch never exceeds the 4 bytes
an element that the route through q takes (so a workspace sized by one serves
the other), a column has at most 4096 bands whatever the field's shape (the
prefixes walk them one after another), and every launch fits a grid."""
import ctypes

import numpy as np
import pytest

import mans_amd


class Scratch(ctypes.Structure):
    _fields_ = [("fits", ctypes.c_bool), ("ty", ctypes.c_uint32), ("band", ctypes.c_uint64),
                ("corner", ctypes.c_uint64), ("words", ctypes.c_uint64)]


def plan(nz, ny, nx, cu=256):
    f = mans_amd.lib()._ZN4mans23lorenzo_inverse_scratchEjjji
    f.restype = Scratch
    f.argtypes = [ctypes.c_uint32] * 3 + [ctypes.c_int]
    return f(nz, ny, nx, cu)


def shapes():
    rng = np.random.default_rng(5)
    out = [(1, 1, 1), (1, 2, 1), (2, 2, 2), (5, 3, 8192), (1, 500, 1000), (1, 512, 8192), (24, 500, 900),
           (512, 24, 1024), (64, 512, 1024), (500, 499, 900), (1, 1_000_000, 1000), (1, 4_000_000, 1000),
           (17, 100_000, 64), (1, (1 << 32) - 1, 1), (1, 1 << 31, 1), (2, 1 << 30, 1), ((1 << 32) - 1, 1, 1),
           (1_000_000, 64, 64)]
    for _ in range(2000):
        nx = int(np.exp(rng.uniform(0, np.log(8193))))
        ny = int(np.exp(rng.uniform(0, np.log((1 << 32) / nx))))
        nz = int(np.exp(rng.uniform(0, np.log((1 << 32) / nx / ny))))
        out.append((max(nz, 1), max(ny, 1), max(nx, 1)))
    return out


@pytest.mark.parametrize("cu", [64, 256, 304])
def test_plan_is_bounded(cu):
    for nz, ny, nx in shapes():
        n = nz * ny * nx
        if n >= 1 << 32:
            continue
        s = plan(nz, ny, nx, cu)
        bands = -(-ny // s.ty)
        assert s.words <= n, (nz, ny, nx, s.words / n)
        assert bands <= 4096, (nz, ny, nx, s.ty)
        assert bands * -(-nx // 1024) * 1024 < 1 << 32, (nz, ny, nx, s.ty)


# (shapes on which the two routes' times differ by a tenth and more)
@pytest.mark.parametrize("shape,tiles", [((4, 4, 4), False), ((16, 16, 16), False), ((24, 24, 32), False),
                                         ((1, 16, 1024), False), ((16, 16, 1500), False), ((64, 8, 512), False),
                                         ((33, 1, 1024), False), ((24, 2, 1024), False), ((160, 8, 1024), False),
                                         ((1, 1, 8192), True), ((16, 1, 512), True), ((16, 2, 100), True),
                                         ((1, 64, 64), True), ((256, 8, 64), True), ((128, 16, 33), True),
                                         ((16, 24, 247), True), ((60, 26, 643), True), ((256, 48, 1024), True),
                                         ((64, 64, 64), True), ((1024, 3, 32), True), ((500, 499, 900), True)])
def test_the_shorter_route_is_taken(shape, tiles):
    assert plan(*shape).fits == tiles


# (shapes on which the rows of a tile make a difference of a fifth and more)
@pytest.mark.parametrize("shape,rows", [((256, 48, 1024), 4), ((500, 100, 900), 16), ((64, 512, 1024), 8),
                                        ((128, 512, 300), 8), ((24, 500, 900), 4), ((768, 32, 1024), 8),
                                        ((500, 499, 900), 32), ((200, 300, 1500), 32), ((1, 1_000_000, 1000), 256)])
def test_tiles_fill_the_chip_in_whole_rounds(shape, rows):
    assert plan(*shape).ty == rows
