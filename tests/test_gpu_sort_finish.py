"""The sort leaves the key's lowest bits out of its passes and puts rows that differ in these only, a group, into order behind them
(k_sortp_finish): documents against the oracle with groups at the edges of a tile and of the longest that is put into order, in order
of arrival and not, and with groups beyond it, whose order is made with passes over all bits."""
import ctypes as C

import numpy as np
import pytest

import oracle_glue as og
from kineto_amd import abi
from kineto_amd.engine import TraceEngine
from stream_builder import B, StreamBuilder

pytestmark = pytest.mark.gpu


def ops(ts, tid, window=None):
    """CPU ops in this order of arrival; with a window: launches, of which it drops some."""
    n = len(ts)
    b = StreamBuilder(window=window or (B, B + 10**15), host_name="sort")
    b.api(["hipLaunchKernel"], flow_start=[0])
    names = [b.s("op%d" % k) for k in range(7)]
    sp = b.build()
    if window is None:
        rec = np.zeros(n, dtype=np.dtype(abi.GenericRec))
        rec["start_ns"], rec["end_ns"] = ts, ts + 5 + np.arange(n) % 900
        rec["resource"], rec["device"], rec["id"] = tid, 4242, np.arange(n) + 1
        rec["name_id"], rec["schema_id"] = np.array(names)[np.arange(n) % 7], abi.KTJ_NONE
        held = (abi.GenericRec * n).from_buffer_copy(rec.tobytes())
        sp.contents.generic, sp.contents.n_generic = C.cast(held, type(sp.contents.generic)), n
    else:
        rec = np.zeros(n, dtype=np.dtype(abi.RuntimeRec))
        rec["begin"], rec["end"], rec["tid"], rec["pid"], rec["id"] = ts, ts + 5, tid, 4242, np.arange(n) + 1
        held = (abi.RuntimeRec * n).from_buffer_copy(rec.tobytes())
        sp.contents.runtime, sp.contents.n_runtime = C.cast(held, type(sp.contents.runtime)), n
    sp._held = (held, b)
    return sp


def same_as_oracle(sp):
    """What the passes say of the sort: bits left to the launch behind its passes, and whether these were made again (KTJ_DBG_SORT)."""
    ora = og.OracleRun(sp)
    want = ora.output()
    info = []
    with TraceEngine(sp.contents.trace_name.decode()) as eng:
        eng.submit_stream(sp)
        for turn in range(2):   # the second one knows how many passes there are
            eng.process()
            assert eng.output() == want, turn
            info.append([int(x) for x in eng.debug("sort_info")])
    ora.close()
    return info


def left_to_the_last_launch(info):
    assert info[0][0] > 0 and info == 2 * [[info[0][0], 0]]


ALL_BITS = [[0, 1], [0, 0]]   # in the second turn from the start


def groups(n, size, order, threads=3, seed=1):
    """Rows in groups of `size` neighbours within 500 ns, groups a millisecond apart, each thread's rows of a group in this order."""
    rng = np.random.default_rng(seed)
    k = np.arange(n)
    group, inside = k // (size * threads), k % (size * threads)
    place = inside // threads
    if order == "backwards":
        place = size - 1 - place
    elif order == "shuffled":
        place = rng.permutation(size)[place]
    elif order == "halves":   # one row only is smaller than the one before it
        place = (place + size // 2) % size
    ts = B + 10**6 + group * 2**20 + place * 500 // size   # (some at the same time: these stay as they came)
    return ts, 5 + inside % threads


@pytest.mark.parametrize("order", ("forwards", "backwards", "shuffled", "halves"))
@pytest.mark.parametrize("size", (1, 2, 63, 64, 65, 255, 256, 257, 400, 700))
def test_groups(size, order):
    """257 rows and more, not in order: all bits by passes."""
    print(size, order, flush=True)
    info = same_as_oracle(ops(*groups(9001, size, order)))
    if size > 256 and order != "forwards":
        assert info == ALL_BITS
    else:
        left_to_the_last_launch(info)


@pytest.mark.parametrize("n", (4097, 8191, 98304, 98305, 262144 + 7))
def test_sizes(n):
    """One launch a pass, tiles of 512 and tiles behind them, whole and with a few rows."""
    print(n, flush=True)
    left_to_the_last_launch(same_as_oracle(ops(*groups(n, 256, "backwards", threads=2))))


def test_large_tiles():
    ts, tid = groups(1200001, 97, "shuffled", threads=5)
    left_to_the_last_launch(same_as_oracle(ops(ts, tid)))


@pytest.mark.parametrize("size, order", ((255, "backwards"), (256, "shuffled"), (256, "halves"), (257, "forwards"), (257, "halves"), (257, "backwards")))
@pytest.mark.parametrize("n", (98305, 1200001))
def test_longest_groups_in_large_tiles(n, size, order):
    """The longest groups that are put into order, and the shortest that are not, with tiles of 1024 rows and of 4096."""
    print(n, size, order, flush=True)
    info = same_as_oracle(ops(*groups(n, size, order)))
    if size > 256 and order != "forwards":
        assert info == ALL_BITS
    else:
        left_to_the_last_launch(info)


def test_dropped_rows_and_random_order():
    rng = np.random.default_rng(5)
    for n in (5000, 20001):
        ts = B + rng.integers(0, 10**9, n)
        same_as_oracle(ops(ts, 5 + rng.integers(0, 4, n)))                                # any order
        same_as_oracle(ops(ts, 5 + rng.integers(0, 4, n), (B + 10**8, B + 6 * 10**8)))    # half of them outside the window
        same_as_oracle(ops(ts, 5 + rng.integers(0, 4, n), (B + 10**10, B + 10**11)))      # all of them
        same_as_oracle(ops(np.full(n, B + 77), 5 + rng.integers(0, 4, n)))                # one time
        far = np.where(np.arange(n) == n // 2, 1000, ts)                                  # a row at the clock's beginning
        same_as_oracle(ops(far, 5 + rng.integers(0, 4, n)))


@pytest.mark.parametrize("n", (90001, 600011, 2400001))
def test_long_groups_in_many_workgroups(n):
    """Workgroups that start when others have found a group that is too long and not in order: tiles of every size."""
    print(n, flush=True)
    assert same_as_oracle(ops(*groups(n, 400, "shuffled"))) == ALL_BITS


def test_long_groups_are_remembered_for_the_next_records():
    """The passes are made twice for the first records of a producer, over all bits for the next fifteen, and the sixteenth are tried again."""
    import torch
    lib = abi.load_engine()
    kinds = []
    for order, size in (("shuffled", 400), ("forwards", 400), ("backwards", 300)):
        for n in (9001, 30011):
            sp = ops(*groups(n, size, order))
            ora = og.OracleRun(sp)
            records = torch.frombuffer(bytearray(C.string_at(sp.contents.generic, n * C.sizeof(abi.GenericRec))), dtype=torch.uint8).cuda()
            kinds.append((sp, n, records, ora.output()))
            ora.close()
    torch.cuda.synchronize()
    sp = kinds[0][0]
    sp.contents.n_generic = 0
    with TraceEngine(sp.contents.trace_name.decode()) as eng:
        eng.submit_stream(sp)

        def served(kind):
            _, n, records, want = kinds[kind]
            eng._chk(lib.ktj_submit_records_device(eng.h, abi.REC_GENERIC, records.data_ptr(), n), "ktj_submit_records_device")
            eng.process()
            assert eng.output() == want, kind
            return [int(x) for x in eng.debug("sort_info")]

        for kind in (3, 2):
            low, again = served(kind)
            assert low > 0 and again == 0
        for bad, good in ((0, 3), (5, 2)):
            assert served(bad) == [0, 1]
            for turn in range(15):
                assert served(turn % 6) == [0, 0], turn
            low, again = served(good)
            assert low > 0 and again == 0
        assert served(1) == [0, 1]
        served(2)


def test_long_groups_and_rows_that_are_not_woven():
    """The list of these is made with the order, the rows are made once: counters and list as if the first order had held."""
    n = 300007
    sp = ops(*groups(n, 400, "shuffled"))
    rec = (abi.GenericRec * n).from_address(C.addressof(sp.contents.generic.contents))
    for k in range(0, n, 5003):
        rec[k].end_ns = rec[k].start_ns + 10**10
    assert same_as_oracle(sp) == ALL_BITS
    ts, tid = groups(20011, 400, "shuffled")
    assert same_as_oracle(ops(ts, tid, (B + 10**6 + 2**20, B + 10**6 + 9 * 2**20))) == ALL_BITS   # launches, some of them dropped


def test_long_groups_in_a_buffer_of_the_callers():
    """The second sort of ktj_process_noalloc, without room for the document and with it."""
    import torch
    for n in (9001, 40013):
        sp = ops(*groups(n, 400, "shuffled"))
        ora = og.OracleRun(sp)
        want = ora.output()
        ora.close()
        for room in (len(want) // 2, len(want) + 64):
            out = torch.full((len(want) + 4096,), 0xEE, dtype=torch.uint8, device="cuda:0")
            torch.cuda.synchronize()
            with TraceEngine(sp.contents.trace_name.decode()) as eng:
                eng.submit_stream(sp)
                for again in (1, 0):
                    size = C.c_uint64()
                    rc = eng.lib.ktj_process_noalloc(eng.h, eng.end_time_ns, out.data_ptr(), room, C.byref(size))
                    got = bytes(out.cpu().numpy())
                    if room < len(want):
                        assert rc != 0 and size.value >= len(want) and got == b"\xEE" * len(got)
                    else:
                        assert rc == 0 and size.value == len(want) and got[:len(want)] == want and got[room:] == b"\xEE" * (len(got) - room)
                        assert [int(x) for x in eng.debug("sort_info")] == [0, again]
