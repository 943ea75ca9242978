"""A call whose workspace is limited takes the GEMM tile that lets it run whole, if one of the two rules' does.

The call's own tile (fastest with the chip to itself) may pad its operands further than the tile of the simpler rule.
A limit that holds the call with the latter, but not with the former, must not cut C into panels."""
import ctypes
import random

import numpy as np
import pytest

from test_planner import _emu, ceil_div, plan, shape, total, vp

_emu.emu_tile_code.argtypes = [vp, ctypes.c_int64, ctypes.c_int64, ctypes.c_int]


def tile(sh, alone):
    return _emu.emu_tile_code(sh.ctypes.data_as(vp), int(sh[0]), int(sh[1]), alone)


def forced(sh, code):
    f = sh.copy()
    f[11] = code
    return f


@pytest.mark.parametrize("seed", range(4))
def test_fits_whole_with_either_tile(seed):
    rnd = random.Random(seed)
    between = 0
    for _ in range(400):
        m, n = (int(np.exp(rnd.uniform(0, 8.5))) for _ in range(2))
        sh = shape(m, n, rnd.choice((1, 60, 200, 700, 5000)), rnd.choice((2, 8, 16, 24)), rnd.random() < 0.3)
        own, small = (total(forced(sh, tile(sh, a)), m, n) for a in (1, 0))
        assert total(sh, m, n) == own
        p = plan(sh, 1 << 50)
        if p["pm"] * p["pn"] > 1:  # panels are priced lower, whatever fits
            continue
        assert p["ws"] == own
        p = plan(sh, small)
        assert (p["pm"], p["pn"], p["ws"]) == (1, 1, min(own, small)), (sh, own, small, p)
        between += own > small
        p = plan(sh, min(own, small) - 1)  # holds neither
        if p is not None:
            assert p["ws"] < min(own, small) and p["pm"] * p["pn"] > 1
            assert (p["pm"], p["pn"]) == (ceil_div(m, p["mb"]), ceil_div(n, p["nb"]))
    assert between > 4
