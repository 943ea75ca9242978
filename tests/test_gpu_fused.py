"""The fused GEMM + CRT kernel against the separate kernels (which a forced GEMM tile selects, and whose
results other tests compare with the oracle): every limb count, both tile sizes, sizes at the edges of
the tiles, and each form of C.  All results are exact, so every comparison is bit for bit."""
import pytest
import torch

import oz2

pytestmark = pytest.mark.gpu

EDGES = [2, 8, 9, 12, 13, 16, 17, 20, 21, 24]


@pytest.fixture(scope="module")
def oz():
    h = oz2.Ozaki2()
    yield h
    h.close()


def rnd(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(n, dtype=torch.float64, device="cuda", generator=g)
    return x * torch.exp2(torch.randint(-20, 20, (n,), device="cuda", generator=g).double())


def bits(x):
    return x.view(torch.int64)


def both(oz, ta, tb, m, n, k, s, alpha, beta, pad=0, tile=128, spoil=None):
    lda, ldb, ldc = (m if ta == "N" else k), (k if tb == "N" else n), m + pad
    A, B, C = rnd(lda * (k if ta == "N" else m), 1), rnd(ldb * (n if tb == "N" else k), 2), rnd(ldc * n, 3)
    if spoil is not None:
        spoil(A, B, C)
    D = C.clone()
    oz.gemm(ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s)
    oz.set_tuning(gemm_tile=tile)
    try:
        oz.gemm(ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, D, ldc, s)
    finally:
        oz.set_tuning()
    assert torch.equal(bits(C), bits(D))


@pytest.mark.parametrize("s", EDGES)
def test_tiles_and_edges(oz, s):
    # 128 x 128 tiles in one full round (k = 300: 64 x 64 is too long for every limb count), the last ones cut
    both(oz, "T", "N", 2047, 2041, 300, s, 1.5, 0.5)
    both(oz, "N", "T", 1921, 2048, 129, s, -1.0, 0.0, pad=1)
    # 64 x 64 tiles: 121 tiles of 128 would leave half the chip idle; k below one stage, rows past the tile
    both(oz, "N", "N", 1348, 1409, 1, s, 1.0, 1.0, pad=3)
    both(oz, "N", "N", 2177, 1153, 128, s, 0.25, -2.0)


@pytest.mark.parametrize("s", [7, 14, 19, 23])
def test_long_k(oz, s):
    both(oz, "N", "N", 2048, 2048, 512, s, 1.0, 0.0)
    both(oz, "T", "T", 4096, 1000, 1024, s, 1.0, 0.0, pad=2)


@pytest.mark.parametrize("s", [8, 16, 22])
def test_zeros_and_non_finite(oz, s):
    m, n, k = 2048, 1985, 96

    def spoil(A, B, C):
        A[5 :: m] = 0.0            # a zero row
        A[77] = float("inf")
        B[k * 3 + 2] = float("nan")
        B[k * 64 : k * 65] = 0.0   # a zero column
        C[m * 9 : m * 9 + 20] = float("nan")
        C[m * 10 + 1] = float("-inf")

    both(oz, "N", "N", m, n, k, s, 1.0, 0.0, spoil=spoil)
    both(oz, "N", "N", m, n, k, s, 2.0, -1.0, spoil=spoil)


@pytest.mark.parametrize("s", EDGES)
def test_batch(oz, s):
    shapes = [(1, 1, 1), (64, 63, 128), (65, 130, 127), (128, 128, 512), (129, 257, 513), (300, 40, 1024), (90, 200, 1100),
              (2048, 1985, 300), (1921, 2047, 100)]  # these fill a round of the fused launch
    probs, want = [], []
    for i, (m, n, k) in enumerate(shapes):
        A, B, C = rnd(m * k, 10 + i), rnd(k * n, 20 + i), rnd((m + i % 3) * n, 30 + i)
        beta = (0.0, 0.5)[i % 2]
        probs.append(dict(ta="N", tb="N", m=m, n=n, k=k, alpha=1.5, A=A, lda=m, B=B, ldb=k, beta=beta, C=C, ldc=m + i % 3,
                          num_moduli=s))
        want.append(C.clone())
    oz.set_tuning(gemm_tile=128)
    try:
        for p, w in zip(probs, want):
            oz.gemm(p["ta"], p["tb"], p["m"], p["n"], p["k"], p["alpha"], p["A"], p["lda"], p["B"], p["ldb"], p["beta"], w,
                    p["ldc"], s)
    finally:
        oz.set_tuning()
    for tiles in ([64] * len(probs), [128] * len(probs), None):
        start = [p["C"].clone() for p in probs]
        b = oz2.Batch(oz, probs, tiles=tiles)
        b.run()
        torch.cuda.synchronize()
        for p, w, c in zip(probs, want, start):
            assert torch.equal(bits(p["C"]), bits(w)), (tiles, p["m"], p["n"], p["k"])
            p["C"].copy_(c)
        b.close()
