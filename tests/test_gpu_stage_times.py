"""Stage times against events around the call, and what asking for them waits for."""
import ctypes

import pytest
import torch

import oz2

pytestmark = pytest.mark.gpu


def rnd(n):
    return torch.randn(n, dtype=torch.float64, device="cuda")


# Launches whose workgroups are far from alike: one operand has a few blocks that read 1.6 MB rows, the other many
# short ones, behind them (T,T) or before (N,N).  The stages are 1.2 to 1.4 ms in eight launches; the gaps between
# those, a few microseconds each, and the events' own share stay below 60 us, 5 %.
@pytest.mark.parametrize("ta,tb", [("T", "T"), ("N", "N"), ("T", "N")])
def test_sum_of_uneven_launches(ta, tb):
    m, n, k = 64, 64, 200000
    A, B, C = rnd(m * k), rnd(k * n), rnd(m * n)
    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    with oz2.Ozaki2() as oz:
        runs = []
        for _ in range(6):
            torch.cuda._sleep(2000000)  # the launches queue up behind it
            begin.record()
            oz.gemm(ta, tb, m, n, k, 1.0, A, m if ta == "N" else k, B, k if tb == "N" else n, 0.0, C, m, 16)
            end.record()
            st = oz.stage_times()
            torch.cuda.synchronize()
            runs.append((begin.elapsed_time(end), st.total_ms(), st.as_dict()))
    call, stages, parts = min(runs)
    assert 0.95 * call <= stages <= call, (call, stages, parts)


def test_waits_for_the_calls_stream_only():
    # a blocking stream (one that the legacy default stream waits for) is busy with other work
    hip = ctypes.CDLL("libamdhip64.so")
    s = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    A, B, C = rnd(64 * 64), rnd(64 * 64), rnd(64 * 64)
    other, done = torch.cuda.ExternalStream(s.value), torch.cuda.Event()
    with oz2.Ozaki2(torch.cuda.Stream()) as oz:
        torch.cuda.synchronize()
        with torch.cuda.stream(other):
            torch.cuda._sleep(1000000000)  # about 0.4 s
            done.record()
        oz.gemm("N", "N", 64, 64, 64, 1.0, A, 64, B, 64, 0.0, C, 64, 16)
        st = oz.stage_times()
        waited = done.query()
        torch.cuda.synchronize()
    del other
    assert hip.hipStreamDestroy(s) == 0
    assert st.gemm_ms > 0 and not waited
