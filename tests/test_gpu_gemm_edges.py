"""The half tiles at the edges of 128 x 128 and 256 x 128 tiles, bit for bit against 64 x 64 tiles (which have
none): every remainder on either side of a half, in single calls, k-chunk sums and both batch schedules."""
import pytest
import torch

import oz2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    h = oz2.Ozaki2()
    yield h
    h.close()


def rnd(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(n, dtype=torch.float64, device="cuda", generator=g)


def forced(oz, tile, m, n, k, s, A, B):
    C = torch.zeros(m * n, dtype=torch.float64, device="cuda")
    oz.set_tuning(gemm_tile=tile)
    try:
        oz.gemm("N", "N", m, n, k, 1.0, A, m, B, k, 0.0, C, m, s)
    finally:
        oz.set_tuning()
    return C.view(torch.int64)


SIZES = [(1, 1), (64, 128), (65, 64), (128, 65), (129, 129), (192, 191), (193, 256), (256, 193), (257, 320), (384, 385), (385, 63)]


@pytest.mark.parametrize("tile", [128, 256128])
@pytest.mark.parametrize("k,s", [(1, 5), (200, 16), (1100, 21)])
def test_edges(oz, tile, k, s):
    for m, n in SIZES:
        A, B = rnd(m * k, 1), rnd(k * n, 2)
        assert torch.equal(forced(oz, tile, m, n, k, s, A, B), forced(oz, 64, m, n, k, s, A, B)), (m, n)


def test_edges_of_chunks(oz):
    m, n, k = 193, 65, 66000
    A, B = rnd(m * k, 3), rnd(k * n, 4)
    for tile in (128, 256128):
        assert torch.equal(forced(oz, tile, m, n, k, 16, A, B), forced(oz, 64, m, n, k, 16, A, B))


@pytest.mark.parametrize("persistent", [False, True])
@pytest.mark.parametrize("tile", [128, 256128])
def test_edges_of_batches(oz, tile, persistent):
    def run(t):
        probs = []
        for i, (m, n) in enumerate(SIZES):
            k = 1030 + 64 * i
            probs.append(dict(ta="N", tb="N", m=m, n=n, k=k, alpha=1.0, beta=0.0, A=rnd(m * k, i), lda=m, B=rnd(k * n, 50 + i),
                              ldb=k, C=torch.zeros(m * n, dtype=torch.float64, device="cuda"), ldc=m, num_moduli=16))
        b = oz2.Batch(oz, probs, tiles=[t] * len(probs), persistent=persistent, graph=False)
        b.run()
        torch.cuda.synchronize()
        return [p["C"].view(torch.int64) for p in probs]

    for x, y in zip(run(tile), run(64)):
        assert torch.equal(x, y)


@pytest.mark.parametrize("s", [8, 12, 16, 20, 24])
def test_edges_of_fused_tiles(oz, s):
    for m, n in ((1985, 2048), (2048, 1985), (1921, 1921), (1984, 1983)):
        A, B, C = rnd(m * 200, 1), rnd(200 * n, 2), torch.zeros(m * n, dtype=torch.float64, device="cuda")
        oz.gemm("N", "N", m, n, 200, 1.0, A, m, B, 200, 0.0, C, m, s)
        assert torch.equal(C.view(torch.int64), forced(oz, 64, m, n, 200, s, A, B)), (m, n)
