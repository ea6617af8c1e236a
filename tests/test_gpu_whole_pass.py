"""GPU: a pass that is put into the stream in one go, where it hands over to the stepwise one, and the sizes
at which its launches change, against the oracle: same document, same counters."""
import ctypes as C

import pytest

from kineto_amd import abi
from kineto_amd.engine import TraceEngine

pytestmark = pytest.mark.gpu


def oracle(sp):
    import oracle_glue as og
    ora = og.OracleRun(sp)
    want, cnt = ora.output(), ora.counters()
    ora.close()
    return want, (cnt["out_of_range"], cnt["out_of_order"], cnt["n_flow_events"], cnt["n_linked"])


def check(eng, want, counters, passes=2):
    for _ in range(passes):
        eng.process()
        st = eng.stats()
        assert eng.output() == want
        assert (st.out_of_range_events, st.gpu_and_cpu_op_out_of_order, st.n_flow_events, st.n_linked) == counters


# one sort tile, one more; both classes of joined rows in one launch, in two; rows of one class only
@pytest.mark.parametrize("config,rows", [(5, 4096), (5, 4097), (1, 1400), (3, 9000), (4, 5000), (5, 262143), (5, 262146), (5, 700001)])
def test_sizes(config, rows):
    sp, release = abi.synth_stream(config, rows, host_name="whole")
    want, counters = oracle(sp)
    with TraceEngine(sp.contents.trace_name.decode()) as eng:
        eng.submit_stream(sp)
        check(eng, want, counters)
    release()


def ops(spans, sync_at=None):
    """CPU ops at base + offset for the offsets of each span, some of them on other rows."""
    from stream_builder import B, StreamBuilder
    b = StreamBuilder()
    for k, off in enumerate(spans):
        b.add_generic("op %d" % (k % 50), 0, B + off, B + off + 5, 1, k % 7, id=k + 1)
    if sync_at is not None:
        b.add_generic("Stream Sync", 15, B + sync_at, B + sync_at + 5, 0, 5, id=len(spans) + 1)
    return b.build()


@pytest.mark.parametrize("bits", [8, 44, 45, 52, 53, 60, 62])
def test_timestamps_far_apart(bits):
    """The sort's passes: fewer than launched, as many, more than launched, keys too wide for a word with the
    index, for one key at all."""
    sp = ops([(k * 2654435761) % (1 << bits) for k in range(4999)] + [0, (1 << bits) - 1])
    want, counters = oracle(sp)
    with TraceEngine(sp.contents.trace_name.decode(), base_time_ns=sp.contents.base_time_ns) as eng:
        eng.submit_stream(sp)
        check(eng, want, counters)


@pytest.mark.parametrize("late,sync", [(1 << 20, None), (1 << 50, None), (2000, 1000)])
def test_later_records_need_more(late, sync):
    """The engine has seen records that sort in two passes; what is submitted afterwards needs more, or a row
    for its Stream Sync activities."""
    sp = ops([k % 3000 for k in range(5000)] + [late + k for k in range(100)], sync)
    want, counters = oracle(sp)
    s = sp.contents
    whole = s.n_generic
    with TraceEngine(s.trace_name.decode(), base_time_ns=s.base_time_ns) as eng:
        s.n_generic = 5000
        eng.submit_stream(sp)
        eng.process()
        eng.process()
        rest = C.addressof(s.generic.contents) + 5000 * C.sizeof(s.generic.contents)
        eng._chk(eng.lib.ktj_submit_records(eng.h, abi.REC_GENERIC, C.c_void_p(rest), whole - 5000), "ktj_submit_records")
        s.n_generic = whole
        check(eng, want, counters)


# sorts with one launch a pass: a last tile of one key, the most keys and one more; a digit that all keys share
@pytest.mark.parametrize("rows,bits", [(5121, 30), (5121, 55), (98304, 30), (98305, 30), (98304, 55), (131072, 30), (131073, 30), (131072, 55), (20000, 1)])
def test_sort_of_one_launch_a_pass(rows, bits):
    sp = ops([(k * 0x9E3779B97F4A7C15) % (1 << 64) >> (64 - bits) for k in range(rows)])
    want, counters = oracle(sp)
    with TraceEngine(sp.contents.trace_name.decode(), base_time_ns=sp.contents.base_time_ns) as eng:
        eng.submit_stream(sp)
        check(eng, want, counters)


def test_document_longer_than_the_first_buffer():
    from stream_builder import B, StreamBuilder
    b = StreamBuilder()
    names = ["n%d" % k for k in range(4000)] + ["long" * 3000]
    for n in names:
        b.s(n)
    for k in range(3000):
        b.add_generic(names[-1], 5, B + k, B + k + 10, 0, 1, id=k + 1)
    sp = b.build()
    want, counters = oracle(sp)
    with TraceEngine(sp.contents.trace_name.decode(), base_time_ns=sp.contents.base_time_ns) as eng:
        eng.submit_stream(sp)
        check(eng, want, counters)


@pytest.mark.parametrize("rows", [300, 2047, 5000, 140000])
def test_sessions_that_fall_back(rows):
    """One engine per trace, as a profiler's session has it: the first pass over the records is the only one.  Stream
    Sync activities and timestamps too far apart send it from three launches to one go and on to step by step; what
    that leaves for the next engine must not show."""
    near = [k * 3 % 5000 for k in range(rows)]
    apart = [(k * 0x9E3779B97F4A7C15) % (1 << 61) for k in range(rows)]
    cases = [(sp,) + oracle(sp) for sp in (ops(near), ops(near, 100), ops(apart), ops(apart, 1 << 60))]
    for k in (0, 1, 0, 2, 1, 3, 0, 3):
        sp, want, counters = cases[k]
        with TraceEngine(sp.contents.trace_name.decode(), base_time_ns=sp.contents.base_time_ns, no_stage_times=k % 2 == 1) as eng:
            eng.submit_stream(sp)
            check(eng, want, counters, passes=1)
            assert eng.stats().stage_ms[abi.STAGE_NAMES.index("total_gpu")] > 0
