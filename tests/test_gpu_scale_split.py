"""Scale and split of both operands in one launch, bit for bit against the oracle, at the sizes where its forms
change: one partial maximum a row or several, read by the split or reduced by a launch; moduli of a block dealt to
several blocks; rows strided or contiguous on either side, odd sizes and leading dimensions."""
import pytest

import oz2
from gpu_cases import complex_case, real_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oz():
    h = oz2.Ozaki2()
    yield h
    h.close()


# k: scale and split in one kernel up to 256 (two and four 64-k blocks); two partials at 257, sixteen up to 4096, then the reducing launch
@pytest.mark.parametrize("k", [1, 65, 128, 129, 256, 257, 515, 4096, 4097])
@pytest.mark.parametrize("ta,tb", [("N", "T"), ("N", "N"), ("T", "N"), ("T", "T")])
def test_partials(oz, ta, tb, k):
    real_case(oz, ta, tb, 67, 33, k, 16, "wide", -1.0, 1.0, lda_extra=1, ldc_extra=1, check_bound=False)
    real_case(oz, ta, tb, 65, 129, k, 21, "u11", check_bound=False)


# 64 blocks of the two splits and fewer go to parts of the moduli: rows / 64 times k / 64, both operands padded
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (64, 64, 64), (512, 512, 256), (512, 576, 256), (640, 512, 256), (1000, 24, 500)])
@pytest.mark.parametrize("s", [2, 3, 9, 24])
def test_parts(oz, m, n, k, s):
    real_case(oz, "N", "N", m, n, k, max(s, 4) if k > 64 else s, "uniform", check_bound=False)


@pytest.mark.parametrize("ta,tb", [("N", "C"), ("C", "N"), ("T", "C"), ("N", "N")])
@pytest.mark.parametrize("k,s", [(130, 16), (300, 24), (1200, 9)])
def test_complex(oz, ta, tb, k, s):
    complex_case(oz, ta, tb, 70, 130, k, s, "uniform", 1.5 - 0.5j, 0.5j, ld_extra=1, check_bound=False)


@pytest.mark.parametrize("ta,tb", [("N", "T"), ("T", "N")])
@pytest.mark.parametrize("k", [3, 200])
def test_special_rows_of_short_k(oz, ta, tb, k):
    # zero rows, subnormals, infinities and NaN among ordinary rows, against the product with k past 256 (padded by
    # zeros), whose exponents come from the scale kernel
    import torch

    def case(kk):
        g = torch.Generator(device="cuda").manual_seed(5)
        A = torch.zeros(130, kk, dtype=torch.float64, device="cuda")
        B = torch.zeros(kk, 70, dtype=torch.float64, device="cuda")
        A[:, :k] = torch.randn(130, k, dtype=torch.float64, device="cuda", generator=g)
        B[:k] = torch.randn(k, 70, dtype=torch.float64, device="cuda", generator=g)
        A[3] = 0.0
        A[64, 1] = float("inf")
        A[65, k - 1] = float("nan")
        A[129, :k] = 5e-324
        B[:, 69] = 0.0
        B[2, 11] = float("-inf")
        a = (A.T if ta == "N" else A).contiguous().reshape(-1)  # column-major op
        b = (B.T if tb == "N" else B).contiguous().reshape(-1)
        C = torch.zeros(130 * 70, dtype=torch.float64, device="cuda")
        oz.gemm(ta, tb, 130, 70, kk, 1.0, a, 130 if ta == "N" else kk, b, kk if tb == "N" else 70, 0.0, C, 130, 24)
        return C

    x, y = case(k), case(300)
    assert torch.equal(torch.isnan(x), torch.isnan(y)) and torch.isnan(x).any()
    # the two take other widths tk (k enters it), so values agree to the accuracy of 24 moduli only
    assert torch.allclose(x.nan_to_num(0.0), y.nan_to_num(0.0), rtol=1e-13, atol=1e-13)


@pytest.mark.parametrize("k", [200, 515])
@pytest.mark.parametrize("ta,tb", [("N", "T"), ("T", "N")])
def test_column_blocks_and_panels(oz, ta, tb, k):
    # exponents written by splits on two streams and panel by panel, against one stream and one panel
    import torch

    g = torch.Generator(device="cuda").manual_seed(9)
    m, n, s = 700, 900, 16
    A = torch.randn(m * k, dtype=torch.float64, device="cuda", generator=g)
    B = torch.randn(k * n, dtype=torch.float64, device="cuda", generator=g)

    def run():
        C = torch.zeros(m * n, dtype=torch.float64, device="cuda")
        oz.gemm(ta, tb, m, n, k, 1.0, A, m if ta == "N" else k, B, k if tb == "N" else n, 0.0, C, m, s)
        torch.cuda.synchronize()
        return C.view(torch.int64)

    want = run()
    whole = oz.workspace_query(ta, tb, m, n, k, s)
    try:
        oz.set_tuning(overlap_blocks=3)
        assert torch.equal(run(), want)
        oz.set_workspace_limit(whole // 3)
        assert torch.equal(run(), want)
        oz.set_tuning()
        assert torch.equal(run(), want)
        assert oz.last_tiling().pm * oz.last_tiling().pn > 1
    finally:
        oz.set_tuning()
        oz.set_workspace_limit(0)
