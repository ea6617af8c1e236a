"""Durations, correlation ids and "External id"s that have no column are taken from the records again: documents and counters against the
oracle for every clock of runtime and device rows and every kind of row, in passes that keep all columns and passes that do not, and the
columns that ktj_debug_fetch gives."""
import numpy as np
import pytest

import oracle_glue as og
from kineto_amd import abi
from kineto_amd.engine import TraceEngine
from stream_builder import B, StreamBuilder

pytestmark = pytest.mark.gpu

IDENTITY, CONVERT, OFFSET = 0, 1, 2


def stream(runtime_mode, device_mode, spans, n=1500, seed=3):
    rng = np.random.default_rng(seed)
    b = StreamBuilder(window=(B + 10**6, B + 10**9), host_name="columns")
    b.api(["hipLaunchKernel", "hipMemcpyAsync", "hipMalloc", "hipDeviceSynchronize"], flow_start=[0, 1], malloc_cid=2)
    b.clock = abi.ClockModel(10**9 + 7, B - 7777, 0.99999871, -987654321, runtime_mode, device_mode)

    def raw(mode, t):
        return t if mode == IDENTITY else t + 987654321 if mode == OFFSET else 10**9 + 7 + int((t - (B - 7777)) / 0.99999871)

    for k in range(n):
        begin = B + int(rng.integers(0, 1002 * 10**6))   # some rows in front of the window, some across its end
        long = int(rng.choice([0, 1, 2, 700, 2 * 10**6, 11 * 10**9]))
        if k % 5 == 0:
            b.add_generic("op%d" % (k % 7), 0, begin - 50, begin + long, 4242, 5, id=k + 1)
        b.add_extcorr(k + 1, k // 5 * 5 + 1)
        if spans and k % 3:
            b.add_usercorr(k + 1, k // 5 * 5 + 1)
        b.add_runtime(k + 1, raw(runtime_mode, begin), raw(runtime_mode, begin + long), k % 5, 4242, 5 + k % 3, kind=k % 4,
                      grid=(k, 2, 1), workgroup=(64, 1, 1), stream=k % 3, size=k * 8)
        at = raw(device_mode, begin + 900)
        if k % 4 == 3:
            b.add_memset(k + 1, at, at + long, device=k % 2, context=1, stream=k % 3, nbytes=k)
        else:
            b.add_device(k + 1, at, at + long, domain=int(k % 4 == 2), op=1 + k % 4, device=k % 2, name="kernel%d" % (k % 9), stream=k % 3, queue=7 + k % 2)
    return b.build()


@pytest.mark.parametrize("spans", (False, True))
@pytest.mark.parametrize("device_mode", (IDENTITY, CONVERT, OFFSET))
@pytest.mark.parametrize("runtime_mode", (IDENTITY, CONVERT, OFFSET))
def test_clocks(runtime_mode, device_mode, spans):
    print(runtime_mode, device_mode, spans, flush=True)
    sp = stream(runtime_mode, device_mode, spans)
    ora = og.OracleRun(sp)
    want = ora.output()
    acts, n = ora.activities()
    with TraceEngine(sp.contents.trace_name.decode()) as eng:
        eng.submit_stream(sp)
        eng.process()
        assert eng.output() == want
        dur, ts = eng.debug("dur"), eng.debug("ts")
        rows = [(acts[i].arrival, acts[i].dur, acts[i].ts) for i in range(n)]
        assert len(rows) > 1000
        for arrival, d, t in rows:
            assert (dur[arrival], ts[arrival]) == (d, t), arrival
        assert len(eng.debug("ext")) == len(dur)
        eng.process()
        assert eng.output() == want
    ora.close()


@pytest.mark.parametrize("rows", (140000, 524288, 524289))
def test_joined_rows_in_one_launch_and_in_two(rows):
    """Generic and device records together: one launch makes both, however many (behind a million there were two)."""
    print(rows, flush=True)
    sp, release = abi.synth_stream(2, rows, host_name="columns")
    ora = og.OracleRun(sp)
    with TraceEngine(sp.contents.trace_name.decode()) as eng:
        eng.submit_stream(sp)
        eng.process()
        assert eng.output() == ora.output()
    ora.close()
    release()
