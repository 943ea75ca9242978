"""The CRT's two forms (16-bit dot products; int8 matrix product) against the oracle at the edges of
their dispatch: every number of moduli next to a change of the limb count, row counts that leave 1 to 4
rows in a column's last quad, C aligned and not, one k-chunk, several, and more than 128 (the chunk
sums fold there).  All results are exact, so every comparison is bit for bit."""
import pytest

import oz2
from gpu_cases import complex_case, real_case

pytestmark = pytest.mark.gpu

EDGES = [2, 8, 9, 12, 13, 16, 17, 20, 21, 24]


@pytest.fixture(scope="module")
def oz():
    h = oz2.Ozaki2()
    yield h
    h.close()


@pytest.mark.parametrize("s", EDGES)
def test_real_quads(oz, s):
    for m, n, pad, beta in ((1, 1, 0, 0.0), (66, 7, 1, -0.5), (131, 5, 0, 2.0), (260, 3, 2, 0.0)):
        real_case(oz, "N", "N", m, n, 48, s, "phi", alpha=1.5, beta=beta, ldc_extra=pad, check_bound=False)


@pytest.mark.parametrize("s", EDGES[1:])
def test_complex_quads(oz, s):
    for m, n, pad, beta in ((2, 1, 0, 0j), (67, 6, 1, 0.5 - 1j), (129, 2, 0, 0j)):
        complex_case(oz, "N", "C", m, n, 40, s, "phi", alpha=1 + 0.5j, beta=beta, ld_extra=pad, check_bound=False)


@pytest.mark.parametrize("s", EDGES[2:])
def test_far_below_the_bound(oz, s):
    # small integers: |C'| is tiny next to M / 4, so the rounding takes its general window; results
    # are exact
    real_case(oz, "N", "T", 70, 9, 33, s, "ints", check_bound=False)
    complex_case(oz, "T", "N", 37, 5, 21, s, "ints", check_bound=False)


@pytest.mark.parametrize("s", [8, 12, 16, 18, 24])
def test_chunks(oz, s):
    real_case(oz, "T", "N", 7, 5, 70001, s, "phi", beta=1.0, check_bound=False)
    complex_case(oz, "C", "N", 3, 6, 66000, s, "uniform", check_bound=False)


def test_many_chunks(oz):
    real_case(oz, "T", "N", 3, 2, 130 * 65408 - 77, 6, "uniform", check_bound=False)
    assert oz.last_tiling().k_chunks == 130
