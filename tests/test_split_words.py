"""The split's words in base 2^31 (to_limbs in os2-xe_amd/csrc/math.hpp), compiled for the host, against Python's
integers at the values where a rounding to a word can go wrong: ties, word borders, the largest magnitudes,
subnormals.  All residues are exact."""
import ctypes
import math
import os
from fractions import Fraction

import numpy as np
import pytest

from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_emu = ctypes.CDLL(os.path.join(ROOT, "os2-xe_amd", "lib", "liboz2_emu.so"))


def values(tk):
    """(v, e) with |v 2^e| < 2^tk"""
    out = [(0.0, 0), (-0.0, 7), (5e-324, 1074), (-5e-324, 1073), (5e-324, 1074 + tk - 1), (2.2250738585072009e-308, 1022 + tk)]
    for b in range(0, tk):
        for d in (0.0, 0.5, -0.5, 1.0, -1.0, 1.5, 2.5):
            x = math.ldexp(1.0, b) + d
            out += [(x, 0), (-x, 0), (math.ldexp(x, -40), 40)]
    for w in range(31, tk, 31):  # halfway between two multiples of a word's unit
        for j in (-3, -1, 1, 3):
            for low in (0.0, 1.0, -1.0):
                out.append(((2 * j * 2.0 ** (w - 1) + 2.0 ** (w - 1) if w < tk - 3 else 2.0 ** (w - 1)) + low, 0))
    top = math.nextafter(1.0, 0.0)
    out += [(top, tk), (-top, tk), (-1.0 / 3.0, tk), (math.ldexp(top, -1000), tk + 1000)]
    return [(v, e) for v, e in out if abs(Fraction(v)) * Fraction(2) ** e < Fraction(2) ** tk]


@pytest.mark.parametrize("s,tk", [(5, 20), (16, 52), (16, 55), (18, 61), (18, 62), (24, 86), (24, 92), (24, 93), (24, 100)])
def test_split_words(s, tk):
    pairs = values(tk)
    v = np.array([p[0] for p in pairs])
    e = np.array([p[1] for p in pairs], dtype=np.int32)
    got = np.zeros((s, v.size), dtype=np.int8)
    p = ctypes.c_void_p
    _emu.emu_split(v.ctypes.data_as(p), e.ctypes.data_as(p), ctypes.c_int64(v.size), s, tk, got.ctypes.data_as(p))
    want = np.zeros_like(got)
    for i, (x, q) in enumerate(pairs):
        r = round(Fraction(x) * Fraction(2) ** q)  # to nearest even
        for t, m in enumerate(O.moduli(s)):
            h = (int(m) - 1) // 2
            want[t, i] = np.uint8(((r + h) % int(m) - h) & 0xFF).astype(np.int8)
    assert np.array_equal(got, want)
