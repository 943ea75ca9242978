"""Stage times of regions of more launches than a handle has stamps (256): the calls neither wait for the GPU nor lose
a launch."""
import pytest
import torch

import oz2

pytestmark = pytest.mark.gpu


def rnd(n):
    return torch.randn(n, dtype=torch.float64, device="cuda")


def call(oz, x, size, s):
    oz.gemm("N", "N", size, size, size, 1.0, x[0], size, x[1], size, 0.0, x[2], size, s)


@pytest.mark.parametrize("per_plane", [False, True])
def test_calls_do_not_wait(per_plane):
    # 300 launches of small calls, or two calls with a launch for each plane of their 9 panel pairs
    size, s, calls = (64, 16, 100) if not per_plane else (384, 16, 2)
    x = [rnd(size * size) for _ in range(3)]
    done = torch.cuda.Event()
    with oz2.Ozaki2() as oz:
        if per_plane:
            oz.set_tuning(batched_gemm=False)
            oz.set_workspace_limit(2 << 20)
        call(oz, x, size, s)
        if per_plane:
            assert oz.last_tiling().pm * oz.last_tiling().pn >= 9
        oz.profile_begin()
        torch.cuda.synchronize()
        torch.cuda._sleep(1000000000)  # about 0.4 s
        done.record()
        for _ in range(calls):
            call(oz, x, size, s)
        waited = done.query()
        st, n = oz.profile_end()
    assert n == calls and st.gemm_ms > 0 and not waited


# Sums over 100 calls (300 launches and more) and over 20: per call alike.  1024^3 with 14 moduli takes about 42 us of
# kernels; a GPU's clock and the gaps' share move that by a few percent, a lost block of 256 launches by 60 % and more.
@pytest.mark.parametrize("overlap", [1, 4])
def test_long_region_adds_up(overlap):
    size, s = 1024, 14
    x = [rnd(size * size) for _ in range(3)]
    with oz2.Ozaki2() as oz:
        oz.set_tuning(overlap_blocks=overlap)
        for _ in range(20):
            call(oz, x, size, s)
        per = []
        for calls in (20, 100, 20, 100):
            oz.profile_begin()
            for _ in range(calls):
                call(oz, x, size, s)
            st, n = oz.profile_end()
            assert n == calls
            per.append([st.scale_ms / n, st.split_ms / n, st.gemm_ms / n, st.crt_ms / n])
        call(oz, x, size, s)
        one = oz.stage_times()
    assert 0.5 * min(map(sum, per)) <= one.total_ms() <= 2 * max(map(sum, per)), (one.as_dict(), per)
    for short, long in ((per[0], per[1]), (per[2], per[3])):
        for a, b in zip(short, long):
            assert abs(a - b) <= 0.2 * a, per
