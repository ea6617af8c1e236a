"""GPU: the three-launch pass of small traces at the edges of its range and where it hands over to the
launches of a large trace, against the oracle: same document, same counters."""
import pytest

from kineto_amd import abi
from kineto_amd.engine import TraceEngine

pytestmark = pytest.mark.gpu


def check(sp, passes=2, **flags):
    import oracle_glue as og
    ora = og.OracleRun(sp)
    want, cnt = ora.output(), ora.counters()
    ora.close()
    with TraceEngine(sp.contents.trace_name.decode(), base_time_ns=sp.contents.base_time_ns, device=0,
                     cuda12_args=bool(sp.contents.create_flags & abi.KTJ_CREATE_CUDA12_ARGS), **flags) as eng:
        eng.submit_stream(sp)
        for _ in range(passes):
            eng.process()
            st = eng.stats()
            assert eng.output() == want
        assert (st.out_of_range_events, st.gpu_and_cpu_op_out_of_order, st.n_flow_events, st.n_linked) == (
            cnt["out_of_range"], cnt["out_of_order"], cnt["n_flow_events"], cnt["n_linked"])
        # the launches of a large trace make the same document from the same records
        eng.debug("perm")
        assert eng.output() == want


# records: 3, 6, 2046, 2049; 2045 and 2048 of strings; with CPU ops per five launches; one wavefront more or less
@pytest.mark.parametrize("config,rows", [(1, 1), (1, 2), (1, 21), (1, 22), (1, 85), (1, 86), (1, 682), (1, 683), (2, 170), (2, 682), (3, 50),
                                         (3, 930), (3, 931), (4, 1100), (5, 1), (5, 255), (5, 257), (5, 2047), (5, 2048), (5, 2049)])
def test_sizes(config, rows):
    sp, release = abi.synth_stream(config, rows, host_name="small")
    check(sp)
    check(sp, no_stage_times=True)
    release()


@pytest.mark.parametrize("seed", range(12))
def test_random_streams(seed):
    """All record classes and edge values: ids that repeat, orphans, ambiguous queues, activities with more
    pieces than a wavefront has lanes, timestamps too far apart for a sort key, Stream Sync activities."""
    import random_streams
    scale = (1, 3, 8)[seed % 3]
    sp = random_streams.random_stream(100 + seed, 40 * scale, 40 * scale, 60 * scale, wide_ids=seed % 2 == 1,
                                      unique_runtime_ids=seed % 4 == 2).build()
    check(sp)


@pytest.mark.parametrize("elements", [1, 20, 30, 31, 60, 400])
def test_activities_with_many_pieces(elements):
    """Arrays around the number of pieces that one wavefront takes at once."""
    from stream_builder import B, StreamBuilder
    b = StreamBuilder()
    schema = b.schema([("values", abi.F_I64_ARRAY, elements), ("x", abi.F_F64, 1)])
    for k in range(9):
        b.add_generic("op %d" % k, 0, B + 1000 * k, B + 1000 * k + 500, 1, 2, id=k + 1, schema=schema,
                      values=[(k * 7919 + j) * (-1) ** j for j in range(elements)] + [0.1 * k])
    check(b.build())


def test_document_longer_than_the_first_buffer():
    """Every record prints the longest string: the buffer that is guessed from the average is too short."""
    from stream_builder import B, StreamBuilder
    b = StreamBuilder()
    names = ["n%d" % k for k in range(400)] + ["long" * 3000]
    for n in names:
        b.s(n)
    for k in range(60):
        b.add_generic(names[-1], 5, B + k, B + k + 10, 0, 1, id=k + 1)
    check(b.build())


@pytest.mark.parametrize("elements,dropped", [(1, False), (400, False), (400, True)])
def test_pass_has_a_time(elements, dropped):
    """Also where one wavefront after the other writes all of its activities, and where none is printed."""
    from stream_builder import B, StreamBuilder
    b = StreamBuilder(window=(B + 10**6, None) if dropped else (None, None))
    schema = b.schema([("values", abi.F_I64_ARRAY, elements)])
    for k in range(9):
        if dropped:
            b.add_device(k + 1, B + 10 * k, B + 10 * k + 5, name="kernel")
        else:
            b.add_generic("op %d" % k, 0, B + 1000 * k, B + 1000 * k + 500, 1, 2, id=k + 1, schema=schema, values=list(range(elements)))
    sp = b.build()
    with TraceEngine("t.json") as eng:
        eng.submit_stream(sp)
        for _ in range(2):
            eng.process()
            ms = eng.stats().stage_ms
            assert 0 < ms[abi.STAGE_NAMES.index("emit")] <= ms[abi.STAGE_NAMES.index("total_gpu")] < 60000
        assert eng.stats().n_emitted == (0 if dropped else 9)
