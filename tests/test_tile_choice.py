"""Which GEMM tile and which form of the GEMM and CRT a call takes (os2-xe_amd/csrc/planner.cpp, host build).

The GPU tests compare the fused kernel with the separate ones at sizes that are meant to reach it; here it is pinned
that they do."""
import ctypes

import pytest

from test_gpu_fused import EDGES
from test_planner import _emu, shape, vp
from test_planner_limits import tile

_emu.emu_fused_tile.argtypes = [vp, ctypes.c_int64, ctypes.c_int64]


def fused(m, n, k, s, mb=None, nb=None, **kw):
    sh = shape(m, n, k, s, **kw)
    return _emu.emu_fused_tile(sh.ctypes.data_as(vp), mb or m, nb or n)


@pytest.mark.parametrize("s", EDGES)
def test_sizes_of_the_fused_tests(s):
    assert fused(2047, 2041, 300, s) == 128
    # with the longest moduli sets the 128 x 128 tiles spill: 64 x 64 up to k = 128
    assert fused(1921, 2048, 129, s) == 128
    assert fused(1348, 1409, 1, s) == 64
    assert fused(2177, 1153, 128, s) == 64


@pytest.mark.parametrize("s", [7, 14, 19, 23])
def test_long_k(s):
    assert fused(2048, 2048, 512, s) == 128
    assert fused(4096, 1000, 1024, s) == (0 if s in (7, 23) else 128)


@pytest.mark.parametrize("s", [8, 16, 22])
def test_zeros_and_non_finite(s):
    assert fused(2048, 1985, 96, s) == (64 if s == 22 else 128)


def test_separate_kernels():
    assert fused(64, 64, 64, 16) == 0                      # a few tiles
    assert fused(4096, 4096, 2048, 16) == 0                # a long k
    assert fused(4096, 4096, 256, 16, cplx=True) == 0
    assert fused(4096, 4096, 256, 16, tile=128) == 0       # a tile was asked for
    assert fused(4096, 4096, 256, 16, per_plane=1) == 0
    assert fused(4096, 4096, 256, 16) == 128
    assert fused(4096, 4096, 256, 16, 4096, 704) == 64     # a panel of it


# the call's own tile and the one of panels and batches
@pytest.mark.parametrize("m,n,k,s,cplx,own,small", [
    (64, 64, 64, 16, False, 64, 64), (100, 40, 5000, 16, False, 64, 64), (1024, 1024, 1024, 14, False, 256128, 128),
    (1537, 771, 3001, 15, False, 128, 128), (4096, 4096, 4096, 8, False, 256, 256), (8192, 8192, 8192, 16, False, 256, 256),
    (777, 1023, 515, 16, True, 256128, 256128), (163, 180, 414, 20, True, 128, 64), (8192, 8192, 256, 16, False, 256128, 256128),
    (130, 8000, 1000, 16, False, 256128, 256128)])
def test_gemm_tile(m, n, k, s, cplx, own, small):
    sh = shape(m, n, k, s, cplx)
    assert (tile(sh, 1), tile(sh, 0)) == (own, small)


def test_forced_tile():
    for code in (64, 128, 256, 256128):
        sh = shape(1000, 1000, 1000, 16, tile=code)
        assert tile(sh, 1) == tile(sh, 0) == code
