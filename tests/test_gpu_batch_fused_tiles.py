"""A batch whose products take the fused kernel: it runs its own tiles, whatever GEMM tile the problems ask for."""
import pytest
import torch

import oz2

pytestmark = pytest.mark.gpu


# 3 x 3 and 5 x 1 tiles of 128 x 128, where 256 rows or columns a tile would pad to 4 x 4 and 6 x 2; 40 and 60 products fill
# more than one round of the fused launch
@pytest.mark.parametrize("m,n,count", [(300, 300, 40), (520, 100, 60)])
@pytest.mark.parametrize("code", [256, 256128])
def test_only_tiles_of_c(m, n, count, code):
    k, s = 200, 16
    g = torch.Generator(device="cuda").manual_seed(1)
    A, B, C0 = (torch.randn(count, x, dtype=torch.float64, device="cuda", generator=g) for x in (m * k, k * n, m * n))
    out, ws = [], []
    with oz2.Ozaki2() as oz:
        for tile in (128, code):
            C = C0.clone()
            b = oz2.Batch(oz, [dict(m=m, n=n, k=k, alpha=1.5, A=A[i], lda=m, B=B[i], ldb=k, beta=0.5, C=C[i], ldc=m, num_moduli=s)
                               for i in range(count)], tiles=[tile] * count)
            b.run()
            torch.cuda.synchronize()
            assert b.info()["launches"] <= 4  # scale, its reduction, split, fused
            ws.append(b.info()["workspace_bytes"])
            out.append(C)
            b.close()
        one = C0[0].clone()
        oz.gemm("N", "N", m, n, k, 1.5, A[0], m, B[0], k, 0.5, one, m, s)
        torch.cuda.synchronize()
    assert ws[0] == ws[1]
    assert torch.equal(out[0], out[1]) and torch.equal(out[0][0], one)
