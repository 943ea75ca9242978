"""A workspace limit that holds the call with the smaller of two GEMM tiles only: one panel pair, the same bits."""
import pytest
import torch

import oz2

pytestmark = pytest.mark.gpu


# sizes whose own tile (256 x 128, 128 x 128) pads further than that of the simpler rule: short k, a longer one, complex
@pytest.mark.parametrize("m,n,k,s,cplx,tile", [(294, 525, 87, 16, False, 64), (783, 507, 73, 24, False, 128),
                                               (2404, 655, 10945, 8, False, 128), (163, 180, 414, 20, True, 64)])
def test_same_bits(m, n, k, s, cplx, tile):
    w = 2 if cplx else 1
    A, B = (torch.randn(w * x * k, dtype=torch.float64, device="cuda") for x in (m, n))
    C = [torch.randn(w * m * n, dtype=torch.float64, device="cuda")]
    C.append(C[0].clone())
    with oz2.Ozaki2() as oz:
        call = oz.zgemm if cplx else oz.gemm
        own = oz.workspace_query("N", "T", m, n, k, s, cplx)
        call("N", "T", m, n, k, 1.5, A, m, B, n, 0.5, C[0], m, s)
        oz.set_tuning(gemm_tile=tile)
        small = oz.workspace_query("N", "T", m, n, k, s, cplx)
        oz.set_tuning()
        assert small < own
        for limit in (small, own - 1):
            oz.set_workspace_limit(limit)
            assert oz.workspace_query("N", "T", m, n, k, s, cplx) == small
        call("N", "T", m, n, k, 1.5, A, m, B, n, 0.5, C[1], m, s)
        ti = oz.last_tiling()
    assert (ti.pm, ti.pn) == (1, 1)
    assert torch.equal(C[0], C[1])
