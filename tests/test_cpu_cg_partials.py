"""The CG sweeps' partial sums fit their buffer (no GPU).

A sweep launches ceil(nx / 256) workgroups per row and component, each of
which leaves two partial sums; sizing the buffer by ceil(nx ny / 256) writes
past it wherever nx is not a multiple of 256."""
import ctypes

import pytest

import wumingpic2d_amd as wm


@pytest.mark.parametrize("nx", [16, 64, 128, 250, 256, 257, 301, 512, 517, 2048, 2049])
@pytest.mark.parametrize("ny", [1, 7, 16, 128, 203])
def test_partial_sums_fit(nx, ny):
    f = wm.load_library()["_Z14wm_cg_partialsii"]
    f.argtypes, f.restype = [ctypes.c_int, ctypes.c_int], ctypes.c_size_t
    assert f(nx, ny) >= 3 * 2 * (-(-nx // 256)) * ny
