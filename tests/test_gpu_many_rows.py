"""Products whose operands have so many rows that one launch cannot hold the blocks of both (a launch takes fewer
than 2^32 threads, a scale block 256 threads for 4 contiguous rows): each operand alone fits, and the calls were
always accepted.  Small integers (four moduli hold 14 bits of each), so the products are exact."""
import pytest
import torch

import oz2

pytestmark = pytest.mark.gpu

M = 67108856  # contiguous rows: 2^24 - 2 scale blocks


def ints(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-100, 101, (n,), device="cuda", generator=g, dtype=torch.int32).double()


def outer_matches(C, A, B):
    """C column-major (len(A) x len(B)) equals A B^T, column by column (the whole of it would double the memory)"""
    return all(torch.equal(C[j * A.numel():(j + 1) * A.numel()], A * B[j]) for j in range(B.numel()))


def test_zgemm():
    n = 8  # two blocks more
    A, B = ints(2 * M, 1), ints(2 * n, 2)
    C = torch.zeros(2 * M * n, dtype=torch.float64, device="cuda")
    with oz2.Ozaki2() as oz:
        oz.set_workspace_limit(4 << 30)
        oz.zgemm("T", "N", M, n, 1, 1.0, A, 1, B, 1, 0.0, C, M, 4)
    assert outer_matches(torch.view_as_complex(C.view(-1, 2)), torch.view_as_complex(A.view(-1, 2)),
                         torch.view_as_complex(B.view(-1, 2)))


def test_batch():
    n = 65  # op(B) strided: two blocks more
    A, B = ints(M, 3), ints(n, 4)
    C = torch.zeros(M * n, dtype=torch.float64, device="cuda")
    with oz2.Ozaki2() as oz:
        b = oz2.Batch(oz, [dict(ta="T", tb="T", m=M, n=n, k=1, alpha=1.0, A=A, lda=1, B=B, ldb=n, beta=0.0, C=C, ldc=M,
                                num_moduli=4)], graph=False)
        b.run()
        torch.cuda.synchronize()
        b.close()
    assert outer_matches(C, A, B)
