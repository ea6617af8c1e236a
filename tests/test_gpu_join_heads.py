"""What the external-correlation records leave for the runtime and device rows has a place of its own where all ids fit 31 bits
(NarrowHead): documents and counters against the oracle, in memory that a pass over other records has just left, for ids that only
some classes of records have, rows that hand nothing over, ids that several rows have, and ids beyond 31 bits that coincide after narrowing."""
import pytest

import oracle_glue as og
from kineto_amd import abi
from kineto_amd.engine import TraceEngine
from stream_builder import B, StreamBuilder

pytestmark = pytest.mark.gpu
N = 1200


def narrowed(id):
    """What an id is looked up by: its low 32 bits with their sign."""
    return id & 0xFFFFFFFF if id & 0x80000000 == 0 else id & 0xFFFFFFFF | 0xFFFFFFFF00000000


def stream(first_id, step, full, beyond, repeated):
    """full: every id has a record of each class, and all of it is handed over.  Otherwise ids lack one class or two, rows lie outside the
    capture window or are of no kind, and (repeated) share ids.  beyond: three ids each coincide after narrowing; external-correlation
    records name the narrowed ids, and with "both" what they were as well, which nothing is looked up by."""
    b = StreamBuilder(window=(B + 10**6, B + 10**9), host_name="heads")
    b.api(["hipLaunchKernel", "hipMemcpyAsync", "hipMalloc", "hipDeviceSynchronize"], flow_start=[0, 1], malloc_cid=2)
    for k in range(0, N, 4):
        b.add_generic("op%d" % (k % 7), 0, B + 2 * 10**6 + k, B + 2 * 10**6 + k + 9, 4242, 5, id=k + 1)
    for k in range(N):
        group = k // 3
        id = first_id + group * step + ((k % 3) << 32) if beyond else first_id + k * step
        of = lambda m: full or k % m != m - 1   # noqa: E731
        if not beyond and of(3):
            b.add_extcorr(id, k // 4 * 4 + 1 if full or k % 7 else 10**6)   # (some name no CPU op)
            if repeated and k % 11 == 0:
                b.add_extcorr(id, k // 8 * 8 + 1)
        if beyond and group % 4 != 3:
            if repeated or k % 3 == group % 3:
                b.add_extcorr(narrowed(id), k // 4 * 4 + 1 if group % 7 else 10**6)
            if beyond == "both" and k % 3:
                b.add_extcorr(id, k // 8 * 8 + 1)
        at = B + 2 * 10**6 + 10 * k if full or k % (7 if beyond else 6) else B + 100   # (some in front of the window)
        kind = 1 if full else k % 4
        if of(5):
            for again in range(2 if repeated and k % 9 == 0 else 1):
                b.add_runtime(id, at + again, at + 5, kind, 4242, 5 + k % 3, kind=(kind + again) % 4, grid=(k + 1, 2, again + 1), workgroup=(64, 1, 1), stream=k % 3, size=k * 8)
        if of(4):
            b.add_device(id, at + 900, at + 950, domain=0 if kind == 1 else 1, op=1 + k % 4, device=k % 2, name="kernel%d" % (k % 9), stream=k % 3, queue=7 + k % 2)
    return b.build()


def ids_that_coincide(s):
    """Slots that rows of different ids share, with rows of different kinds, in and out of the window; and whether the ids lie close enough
    together for slots of their own."""
    rows = {}
    for k in range(s.n_runtime):
        r = s.runtime[k]
        rows.setdefault(narrowed(r.id), []).append((r.id, r.kind, r.begin >= s.window_start_ns))
    shared = [x for x in rows.values() if len({id for id, _, _ in x}) > 1]
    assert len(shared) > N // 3 * 0.8 and max(len({id for id, _, _ in x}) for x in shared) == 3
    assert {len({kind for _, kind, _ in x}) for x in shared} >= {2, 3} and {len({inside for _, _, inside in x}) for x in shared} == {1, 2}
    looked_up = [*rows, *(s.extcorr[k].correlation for k in range(s.n_extcorr))]
    return max(looked_up) - min(looked_up) < s.n_extcorr + s.n_runtime


@pytest.mark.parametrize("hashed", (False, True))
@pytest.mark.parametrize("beyond, repeated, step, first_id", (
    ("", False, 1, 5), ("", True, 3, 5), ("", False, 977, 5), ("narrowed", False, 1, 5), ("narrowed", True, 2, 5), ("both", False, 1, 5),
    ("both", True, 2, 5), ("narrowed", False, 3, 2**31 - 600), ("both", True, 1, 2**31 - 200)))
def test_rows_that_lack_one_class_or_another(beyond, repeated, step, first_id, hashed):
    print(beyond, repeated, step, first_id, hashed, flush=True)
    lib = abi.load_engine()
    lib.ktj_debug_force_sort_passes(1)
    try:
        # the first leaves its rows' values in the memory that the second then takes
        for sp in (stream(5, step, True, "", False), stream(first_id, step, False, beyond, repeated)):
            o = og.OracleRun(sp)
            want, counters = o.output(), o.counters()
            o.close()
            with TraceEngine(sp.contents.trace_name.decode(), base_time_ns=sp.contents.base_time_ns, hash_join=hashed) as e:
                e.submit_stream(sp)
                for _ in range(2):
                    e.process()
                    assert e.output() == want
                    got = e.stats()
                    assert [got.n_linked, got.gpu_and_cpu_op_out_of_order, got.out_of_range_events] == [counters[k] for k in ("n_linked", "out_of_order", "out_of_range")]
        if beyond:  # (of the second)
            assert ids_that_coincide(sp.contents) == (beyond == "narrowed" and first_id == 5)
    finally:
        lib.ktj_debug_force_sort_passes(0)


@pytest.mark.parametrize("ops", (349525, 349526, 420001))
def test_tables_of_a_prime_number_of_runs(ops):
    """Ids too far apart for slots of their own, some without a runtime row: the last table of a power of two runs, and tables of as many
    as the records ask for."""
    print(ops, flush=True)
    sp, release = abi.synth_stream(2, ops, host_name="heads")
    s = sp.contents
    assert (s.n_runtime, s.n_device) == (ops, ops)
    for k in range(ops):
        s.runtime[k].id = s.runtime[k].id * 977 + (k % 5 == 4)
        s.device[k].id *= 977
    for k in range(s.n_extcorr):
        s.extcorr[k].correlation *= 977
    o = og.OracleRun(sp)
    want, counters = o.output(), o.counters()
    o.close()
    with TraceEngine(s.trace_name.decode(), base_time_ns=s.base_time_ns) as e:
        e.submit_stream(sp)
        for _ in range(2):
            e.process()
            assert e.output() == want
            assert e.stats().n_linked == counters["n_linked"]
    release()
