"""Scale and split in one kernel (k <= 256): rows of subnormals, whose products with columns of order 2^1000
come out normal, and of large values, bit for bit against the oracle.  Forms of two words (16 moduli) and of three (24)."""
import numpy as np
import pytest
import torch

import oz2
from gpu_cases import bits, flat, to_dev
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("s", [16, 24])
@pytest.mark.parametrize("ta,tb", [("N", "T"), ("T", "N")])
@pytest.mark.parametrize("k", [3, 128, 200, 256])
def test_finite_extremes(ta, tb, k, s):
    m, n = 130, 70
    rng = np.random.default_rng(k)
    A, B = rng.standard_normal((m, k)), rng.standard_normal((k, n)) * 2.0**1000
    A *= 2.0**-1000
    # the smallest subnormals; with 24 moduli larger ones (the oracle shifts a mantissa by less than 75 bits)
    tiny = 5e-324 if s == 16 else 5e-324 * 2**17
    A[3] = 0.0
    A[64] = tiny
    A[65] = rng.integers(-9, 10, k) * tiny
    A[66] = 0.0
    A[66, k - 1] = -tiny                                # one among zeros
    A[129] = (2.0**-1022 - 5e-324) * np.sign(A[129])    # the largest
    A[100] = rng.standard_normal(k) * np.exp2(rng.integers(-1074, -990, k).astype(float))
    A[101] *= 2.0**1014                                 # entries of C near the largest double
    B[:, 5] = 0.0
    B[:, 6] = tiny
    B[:, 69] = rng.standard_normal(k) * np.exp2(rng.integers(-60, 1000, k).astype(float))
    a, b = flat(A if ta == "N" else A.T), flat(B if tb == "N" else B.T)
    lda, ldb = (m if ta == "N" else k), (k if tb == "N" else n)
    C0 = rng.uniform(-1, 1, m * n)
    C, ref = to_dev(C0.copy()), C0.copy()
    with oz2.Ozaki2() as oz:
        oz.gemm(ta, tb, m, n, k, 1.0, to_dev(a), lda, to_dev(b), ldb, 0.0, C, m, s)
        torch.cuda.synchronize()
    O.dgemm(ta, tb, m, n, k, 1.0, a, lda, b, ldb, 0.0, ref, m, s)
    got = C.cpu().numpy()
    assert np.array_equal(bits(got), bits(ref))
    # the rows of subnormals are there: 2^-1074 times 2^1000 is a normal number
    rows = np.abs(got.reshape(n, m)[[0, 1, 2]])
    assert (rows[:, 64] > 0).all() and (rows[:, 129] > 0).all()
