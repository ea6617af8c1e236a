"""Activities put together from segments (weave_core.h, weave.hip): the rows' texts, lengths and tail kinds and the schemas'
texts against the oracle's documents, on the CPU for every kind of row and at the edges of what a row has room for, and on the
GPU at the edges of a turn, of the strings that wait in LDS and of the activities that are left to the other kernel."""
import ctypes as C
import os
import struct

import pytest

import oracle_glue as og
from kineto_amd import abi
from stream_builder import B, StreamBuilder

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NAME_LENGTHS = (0, 1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, 257, 259, 300, 383, 384, 385, 500, 511, 512, 513, 1200, 2600, 12800, 12801)
PIDS = (0, 1, 4194303, 4194304, (1 << 31) - 1, -3)                       # 22 bits, and beyond
TIDS = (0, 5, (1 << 42) - 1, 1 << 42, (1 << 47) - 1, 1 << 47, -5, (1 << 63) - 1)
NUMBERS = (0, 9, 10, 99999999, 100000000, 10**10, 10**11 - 1, 10**11, 10**15 - 1, 10**15, (1 << 63) - 1, -1, -(10**9), -(10**10), -(1 << 63))


def _text(n, salt=0):
    return "".join(chr(97 + (k * 7 + salt) % 26) for k in range(n))


def edge_stream(n, other_types=True):
    """n activities: ordinary kernels and launches, and among them one after the other what a text row has just room for and what
    it has not.  other_types: also what is never a text row, by its type or schema."""
    b = StreamBuilder(window=(B, B + 10**13), host_name="edge")
    b.api(["hipLaunchKernel", "hipMemcpyAsync", "hipMalloc", None, "hipFree"], flow_start=[0, 1], malloc_cid=2)
    names = [b.s(_text(k, k)) for k in NAME_LENGTHS] + [b.s('"quoted"\\'), b.s("kernel"), b.s("Stream Sync")]
    fields = [
        [("Sequence number", abi.F_I64, 1)],
        [("Trace name", abi.F_STR, 1)],
        [("Value", abi.F_F64, 1)],
        [(None, abi.F_RAW, 1)],
        [("A", abi.F_I64, 1), ("B", abi.F_U64, 1), ("C", abi.F_BOOL, 1), ("D", abi.F_I64, 1)],
        [("A", abi.F_I64, 1), ("B", abi.F_U64, 1), ("C", abi.F_BOOL, 1), ("D", abi.F_I64, 1), ("E", abi.F_I64, 1)],
        [("grid", abi.F_I64_ARRAY, 3), ("block", abi.F_I64_ARRAY, 2), ("n", abi.F_U64, 1), ("m", abi.F_I64, 1)],
        [("none", abi.F_I64_ARRAY, 0), ("one", abi.F_I64_ARRAY, 1)],
        [("four", abi.F_I64_ARRAY, 4)],
        [("d", abi.F_DICT_BEGIN, 0), ("x", abi.F_I64, 1), (None, abi.F_DICT_END, 0), ("s", abi.F_STR, 1), ("y", abi.F_I64, 1)],
        [(_text(48), abi.F_I64, 1), (_text(40, 3), abi.F_STR, 1)],
        [(_text(49), abi.F_I64, 1)],
        [("s", abi.F_STR, 1), ("t", abi.F_STR, 1)],
        [],
    ]
    if other_types:   # the last lie behind the sixteenth
        fields += [[("late %d" % k, abi.F_I64, 1)] for k in range(5)]
    schemas = [b.schema(f) for f in fields]
    types = (0, 1, 2, 10, 17, 9, 0, 0) if other_types else (0, 1, 2, 10, 3, 5, 0, 0)

    def number(k):
        return NUMBERS[k % len(NUMBERS)]

    def op_id(j):
        return (j, -j, 2**31 - 1 - j, j - 2**31)[j % 4]

    def rare(k, ts):
        kind, j = k % 4, k // 4
        if kind == 0:                                # generic
            values = []
            f = fields[j % len(fields)]
            for i, (_key, typ, count) in enumerate(f):
                if typ == abi.F_F64:
                    values.append((0.5, 1e22, 123456.789, -2.2250738585072014e-308, float("inf"), float("nan"))[(j // 3 + i) % 6])
                elif typ in (abi.F_STR, abi.F_RAW):
                    values.append((names + [abi.KTJ_NONE - 1])[(j + i) % (len(names) + 1)])
                elif typ == abi.F_BOOL:
                    values.append(j & 1)
                else:
                    values += [number(j + i + c) if j & 1 else (j + c) % 1200000 for c in range(count)]
            r = b.add_generic(None, types[j % 8], ts, ts + (0, 999, 1000, 10**10 - 1, 10**10, -4)[j % 6], PIDS[j % 6], TIDS[j % 8] if j % 3 else 5,
                              id=op_id(j), schema=schemas[j % len(fields)], values=values, flow_id=number(j) if j % 2 else 0, flow_type=1 + j % 2, flow_start=j % 4 < 2)
            r.name_id = names[j % len(names)]
        elif kind == 1:                              # launches
            dim = ((1, 1, 1), (99999, 999, 999), (999999, 999, 999), (4294967295, 1, 1), (1, 999999, 1), (1, 1000000, 1))[j % 6]
            r = b.add_runtime(number(j) & 0xFFFFFFFFFFFFFFFF if j % 2 else 1 << 20 | j, ts, ts + 1500, 0, 1, TIDS[j % 5], kind=1, grid=dim, workgroup=dim if j % 2 else (256, 1, 1),
                              lds=(0, 4294967295)[j % 2], stream=j % 3)
            r.u.kernel.kernel_name_id = (names + [abi.KTJ_NONE])[j % (len(names) + 1)]
        elif kind == 2:                              # copies and allocations
            size = (0, 10**11 - 1, 10**11, 1 << 40, 4096)[j % 5]
            if j % 2:
                b.add_runtime(1 << 21 | j, ts, ts + 999, 1, 1, 5, kind=2, src=(1 << 60) - 1 if j % 3 else 1 << 60, dst=j, size=size, copy_kind=(0, 4, -1, 9999, -1000)[j % 5])
            else:
                b.add_runtime(1 << 21 | j, ts, ts + 999, (2, 3, 4)[j % 3], 1, 5, kind=(3, 0)[j // 2 % 2], ptr=(0, 0x7F0000000000, (1 << 64) - 1)[j % 3], size=size)
        else:                                        # device rows
            domain, op = ((0, 0), (1, 2), (1, 4), (2, 0), (3, 0))[j % 5]
            if domain == abi.KTJ_DOM_MEMSET:
                b.add_memset(1 << 22 | j, ts, ts + (1, 0, 77)[j % 3], device=j % 2, context=(1, 9999999, 10000000)[j % 3], stream=j % 4, nbytes=number(j) & 0xFFFFFFFFFF,
                             memory_kind=j % 10)
            else:
                b.add_device(number(j) & 0xFFFFFFFFFFFFFFFF if j % 2 else 1 << 20 | (j - 1), ts, ts + (0, 1, 12345678, 10**10)[j % 4], domain=domain, op=op, device=j % 3, name=None,
                             queue=(1, 9999999, 10000000)[j % 3], nbytes=number(j) & 0xFFFFFFFFFFFF).name_id = names[j % len(names)]

    for k in range(n):
        ts = B + 1000 + 2001 * k
        if k % 5 < 2:
            if k % 2:
                b.add_extcorr(k + 1, op_id(k // 40))
            b.add_device(k + 1, ts, ts + 1234, device=0, name="gemm_%d" % (k % 7), queue=1 + k // 97 % 2)
        elif k % 5 == 2:
            b.add_runtime(k, ts, ts + 1234, 0, 1, 5, kind=1, grid=(k, 1, 1), workgroup=(256, 1, 1))
        else:
            rare(k // 5 * 2 + k % 5 - 3, ts)
    return b.build()


@pytest.fixture(scope="module")
def sim():
    lib = C.CDLL(os.path.join(ROOT, "tests", "host_sim", "libktjsim.so"))
    lib.ktjsim_render.argtypes = [C.POINTER(abi.Stream), C.c_uint32, C.POINTER(C.c_void_p), C.POINTER(C.c_uint64)]
    lib.ktjsim_free.argtypes = [C.c_void_p]
    return lib


def _woven_vs_oracle(sim, sp):
    o = og.OracleRun(sp)
    want = o.output()
    o.close()
    p, nb, woven, left = C.c_void_p(), C.c_uint64(), C.c_uint64(), C.c_uint64()
    assert sim.ktjsim_render(sp, 1, C.byref(p), C.byref(nb)) == 0   # 1: from segments; it fails where a length or tail kind differs
    sim.ktjsim_woven(C.byref(woven), C.byref(left))
    got = C.string_at(p, nb.value)
    sim.ktjsim_free(p)
    if got != want:
        i = next((k for k in range(min(len(got), len(want))) if got[k] != want[k]), min(len(got), len(want)))
        raise AssertionError(f"byte {i}: got {got[max(0, i - 80):i + 60]!r} want {want[max(0, i - 80):i + 60]!r}")
    return woven.value, left.value


def test_segments_of_every_kind_of_row(sim):
    import kat_cases
    import random_streams
    for cfg in range(1, 6):
        sp, release = abi.synth_stream(cfg, 2000, host_name="box")
        assert _woven_vs_oracle(sim, sp)[1] == 0, cfg        # ordinary records are text rows, all of them
        release()
    for case in kat_cases.SUBSTRING_CASES + [kat_cases.case_rocm_sync_trace]:
        _woven_vs_oracle(sim, case()[0].build())
    for seed in range(60):
        _woven_vs_oracle(sim, random_streams.random_stream(seed, wide_ids=seed % 2 == 1).build())
    assert _woven_vs_oracle(sim, edge_stream(3000, False))[1] > 200
    woven, left = _woven_vs_oracle(sim, edge_stream(3000))
    assert woven > 1800 and left > 300, (woven, left)


HOUR, DAY, LEAD = 3600 * 10**9, 86400 * 10**9, 10**14   # ns; a time's lead counts the last


def _base_back(sp, ns):
    """The same records ns further behind the base of the times."""
    sp.contents.base_time_ns -= ns
    return sp


@pytest.mark.parametrize("back", (27 * HOUR, 28 * HOUR, LEAD - 10**9, LEAD - 1, LEAD, 62 * DAY, 91 * DAY, 10 * LEAD - 10**9, B))
def test_times_long_behind_the_base(sim, back):
    """libkineto's base is the clock floored to 91 days; B: a base of 0.  Times of twelve digits and more are text rows as any, the
    carry into another lead inside the trace too."""
    for cfg in range(1, 6):
        sp, release = abi.synth_stream(cfg, 2000, host_name="box")
        assert _woven_vs_oracle(sim, _base_back(sp, back))[1] == 0, cfg
        release()
    at_base = _woven_vs_oracle(sim, edge_stream(3000, False))
    left = _woven_vs_oracle(sim, _base_back(edge_stream(3000, False), back))[1]
    assert left <= at_base[1] + 60, (left, at_base)   # a track of 22 digits has no room for five more


def test_leads_with_no_room_are_left(sim):
    """Process, thread and lead share the room that the segment of their text has; a lead has sixteen bits."""
    def stream(base, pid, tid):
        b = StreamBuilder(base=base, window=(B, B + 10**13), host_name="edge")
        for k in range(3):
            b.add_generic("op", 0, B + 1000 + 2000 * k, B + 2000 + 2000 * k, pid, tid, id=k + 1)
        return b.build()
    pid, tid = 4194303, (1 << 47) - 1
    assert _woven_vs_oracle(sim, stream(B, pid, tid)) == (3, 0)
    assert _woven_vs_oracle(sim, stream(B - 999 * LEAD, pid, tid)) == (3, 0)
    assert _woven_vs_oracle(sim, stream(B - 1000 * LEAD, pid, tid)) == (0, 3)
    assert _woven_vs_oracle(sim, stream(B - 1000 * LEAD, pid // 10, tid)) == (3, 0)
    assert _woven_vs_oracle(sim, stream(B - 65535 * LEAD, pid, tid // 100)) == (3, 0)
    assert _woven_vs_oracle(sim, stream(B - 65536 * LEAD, 1, 1)) == (0, 3)


def _odd_streams():
    """Streams of three ordinary CPU ops, a launch, a copy, an allocation and a kernel, each with one row that is no text row, as its record says."""
    def base():
        b = StreamBuilder(window=(B, B + 10**13), host_name="odd")
        b.api(["hipLaunchKernel", "hipMemcpyAsync", "hipMalloc"], flow_start=[0], malloc_cid=2)
        for k in range(3):
            b.add_generic("op", 0, B + 1000 + k, B + 2000 + k, 1, 5, id=k + 1)
        b.add_runtime(1, B + 3000, B + 4000, 0, 1, 5, kind=1, grid=(99999, 999, 999), workgroup=(256, 1, 1))
        b.add_runtime(2, B + 5000, B + 6000, 1, 1, 5, kind=2, src=1, dst=2, size=10**11 - 1, copy_kind=-999)
        b.add_runtime(3, B + 7000, B + 8000, 2, 1, 5, kind=3, ptr=(1 << 60) - 1, size=5)
        b.add_device(1, B + 9000, B + 9500, name="k", queue=9999999)
        return b
    t = B + 20000
    def generic(b, typ=0, end=t + 5, dev=1, res=5, **kw):
        b.add_generic(kw.pop("name", "op"), typ, t, end, dev, res, **kw)
    def runtime(b, **kw):
        b.add_runtime(kw.pop("id", 9), t, kw.pop("end", t + 5), kw.pop("cid", 0), kw.pop("pid", 1), kw.pop("tid", 5), **kw)
    def device(b, **kw):
        b.add_device(kw.pop("id", 9), t, kw.pop("end", t + 5), **kw)
    def two_strings(b):
        generic(b, schema=b.schema([("Input type", abi.F_STR, 1), ("Input Dims", abi.F_STR, 1)]), values=[b.s("x"), b.s("y")])
    def five_numbers(b):
        generic(b, schema=b.schema([("n%d" % k, abi.F_I64, 1) for k in range(5)]), values=[1] * 5)
    def late_schema(b):
        ids = [b.schema([("k%d" % k, abi.F_I64, 1)]) for k in range(17)]
        generic(b, schema=ids[16], values=[1])
    def many_schemas(b):   # more descriptors than there is room for
        ids = [b.schema([("k%d_%d" % (k, j), abi.F_I64, 1) for j in range(4)]) for k in range(16)]
        generic(b, schema=ids[15], values=[1] * 4)
    edits = dict(
        instant=lambda b: generic(b, 17), counter=lambda b: generic(b, 9, schema=b.schema([("v", abi.F_F64, 1)]), values=[0.5]), two_strings=two_strings, five_numbers=five_numbers,
        late_schema=late_schema, many_schemas=many_schemas, stream_sync=lambda b: generic(b, 15, name="Stream Sync"),
        annotation_flow=lambda b: generic(b, 2, flow_id=3, flow_type=1), flow=lambda b: generic(b, flow_id=10**11, flow_type=1), external=lambda b: generic(b, id=-10**9, schema=b.schema([("n", abi.F_I64, 1)]), values=[1]),
        process=lambda b: generic(b, dev=1 << 22), negative_process=lambda b: generic(b, dev=-1), thread=lambda b: generic(b, res=1 << 47),
        duration=lambda b: generic(b, end=t + 10**10), annotation_duration=lambda b: generic(b, 2, end=t + 10**10 - 2),
        runtime_duration=lambda b: runtime(b, end=t + 10**10), correlation=lambda b: runtime(b, id=10**11),
        grid=lambda b: runtime(b, kind=1, grid=(999999, 999, 999)), block=lambda b: runtime(b, kind=1, grid=(1, 1, 1), workgroup=(1, 1000000, 1)),
        address=lambda b: runtime(b, cid=1, kind=2, src=1 << 60), size=lambda b: runtime(b, cid=1, kind=2, size=10**11), copy_kind=lambda b: runtime(b, cid=1, kind=2, copy_kind=-1000),
        pointer=lambda b: runtime(b, cid=2, kind=3, ptr=1 << 60), device_duration=lambda b: device(b, end=t + 1 + 10**10, name="k"), queue=lambda b: device(b, queue=10**11, name="k"),
        device_correlation=lambda b: device(b, id=10**11, name="k"), api=lambda b: runtime(b, cid=3), kernel_without_name=device)
    for name, edit in edits.items():
        b = base()
        edit(b)
        yield name, b.build()
    b = base()
    b.create_flags = abi.KTJ_CREATE_CUDA12_ARGS
    b.add_memset(9, t, t + 5)
    yield "cuda12", b.build()


def test_rows_left_are_known_when_decoded(sim):
    """Whether too many rows are left is decided before any is made: what a record says by itself is counted (and nothing that is
    a text row after all: ktjsim_render fails there)."""
    sim.ktjsim_left_known.restype = C.c_uint64
    for name, sp in _odd_streams():
        assert (_woven_vs_oracle(sim, sp)[1], sim.ktjsim_left_known()) == (1, 1), name
    _woven, left = _woven_vs_oracle(sim, edge_stream(3000))
    assert left * 0.6 < sim.ktjsim_left_known() < left


def test_long_jobs(sim):
    """What grows with a job is text however long it has run: the fourth number of its operators' schema (the sequence number), and
    the queues."""
    def stream(n):
        b = StreamBuilder(window=(B, B + 10**13), host_name="long")
        op = b.schema([("Ev Idx", abi.F_I64, 1), ("Record function id", abi.F_U64, 1), ("Fwd thread id", abi.F_U64, 1), ("Sequence number", abi.F_I64, 1)])
        string = b.schema([("a", abi.F_I64, 1), ("b", abi.F_I64, 1), ("c", abi.F_I64, 1), ("d", abi.F_I64, 1), ("s", abi.F_STR, 1)])
        t = B + 1000
        b.add_generic("op", 0, t, t + 5, 1, 5, id=1, schema=op, values=[1, 2, 3, n])
        b.add_generic("op", 0, t + 10, t + 15, 1, 5, id=2, schema=op, values=[1, 2, 3, -(n // 10)])
        b.add_generic("op", 0, t + 20, t + 25, 1, 5, id=3, schema=string, values=[1, 2, 3, n, b.s("text")])
        b.add_device(4, t + 70, t + 75, name="k", queue=n)
        b.add_device(6, t + 80, t + 85, domain=1, op=2, queue=n)
        b.add_memset(8, t + 90, t + 95, context=n & 0xFFFFFFFF, nbytes=5)
        return b.build()
    for digits in range(1, 12):   # (beside a string there is room for seven)
        assert _woven_vs_oracle(sim, stream(10**digits - 1)) == ((6, 0) if digits < 8 else (5, 1)), digits
    assert _woven_vs_oracle(sim, stream(10**11)) == (1, 5)   # (a minus is a character)


def test_bytes_without_a_bandwidth(sim):
    """A copy of no duration has bytes and no bandwidth, and so has a kernel with a copy's id: text rows as any."""
    b = StreamBuilder(window=(B, B + 10**13), host_name="copies")
    b.api(["hipLaunchKernel", "hipMemcpyAsync"], flow_start=[0, 1])
    for k in range(14):   # directions 0 to 6, the last two unknown ones
        t = B + 10000 * (k + 1)
        b.add_runtime(k + 1, t, t + 10, 1, 1, 5, kind=2, src=1, dst=2, size=(0, 7, 10**10)[k % 3], copy_kind=1, stream=k % 2)
        b.add_device(k + 1, t + 50, t + 50 + k // 7, domain=1, op=k % 7, queue=k)
    for k in range(20, 23):
        b.add_runtime(k, B + k, B + k + 5, 1, 1, 5, kind=2, size=4096, copy_kind=1)
        b.add_device(k, B + k + 50, B + k + 50 + k % 2, name="kernel with bytes", queue=1)
    assert _woven_vs_oracle(sim, b.build()) == (34, 0)
    sp, release = abi.synth_stream(2, 60000, host_name="box")
    assert _woven_vs_oracle(sim, sp)[1] == 0
    release()


def test_doubles_as_text(sim):
    """Shifted together, against the formatter's characters one by one: zeros behind the text, too."""
    import random
    import struct
    rng = random.Random(11)
    values = [0.0, -0.0, float("inf"), float("-inf"), float("nan"), 5e-324, 1.7976931348623157e308, -2.2250738585072014e-308, 0.1, 1e-4, 9.999e-5, 1e-5, 1e15, 1e16,
              123456789012345680.0, 9999999999999998.0, 1.0, 10.0, 12.5, -0.001234]
    values += [m * 10.0**e for e in range(-8, 20) for m in (1, 1.5, 12.25, 0.6666666666666666)]
    values += [struct.unpack("<d", struct.pack("<Q", rng.getrandbits(64)))[0] for _ in range(20000)]
    values += [rng.choice((-1, 1)) * rng.uniform(0, 1) * 10.0**rng.randrange(-7, 20) for _ in range(20000)]
    sim.ktjsim_fmt_double.argtypes = sim.ktjsim_real_text.argtypes = [C.c_double, C.c_char_p]
    got, want = C.create_string_buffer(64), C.create_string_buffer(64)
    for v in values:
        n, m = sim.ktjsim_real_text(v, got), sim.ktjsim_fmt_double(v, want)
        if v != v or v in (float("inf"), float("-inf")):   # (quoted where the formatter prints an argument)
            assert got.raw[:n].strip(b'"') == want.raw[:m].strip(b'"'), v
            assert got.raw[:n].startswith(b'"') and got.raw[:n].endswith(b'"')
        else:
            assert got.raw[:n] == want.raw[:m], v
        assert got.raw[n:24] == bytes(24 - n), v


def large_stream(n, left_known, long_names=False):
    """n CPU ops on five threads, so many that a wavefront takes several turns of sixteen: every 800 activities some at the edges of
    turns that are left (left_known: their records say so; the others have a typed number with no room), flow events, names that
    wait in LDS and names that do not, doubles beside their rows.  long_names: and most of them far longer than the dictionary's
    average, so that the first guess of the document's size is too small."""
    import numpy as np
    rng = np.random.default_rng(n)
    b = StreamBuilder(window=(B, B + 10**15), host_name="large")
    names = [b.s(_text(k, k)) for k in (1, 16, 17, 40, 127, 128, 129, 300, 700)]
    plain = b.schema([("Sequence number", abi.F_I64, 1)])
    wide = b.schema([("A", abi.F_I64, 1), ("B", abi.F_U64, 1), ("C", abi.F_BOOL, 1), ("x", abi.F_F64, 1)])
    text = b.schema([("s", abi.F_STR, 1), ("y", abi.F_I64, 1)])
    if long_names:
        for k in range(200):
            b.s("s%d" % k)
    values = [7, 12, 34567, 1, struct.unpack("<Q", struct.pack("<d", -1.2345678901234567e-300))[0], names[7], 3, 1 << 62]
    b.arg_slots(values)
    sp = b.build()
    rec = np.zeros(n, dtype=np.dtype(abi.GenericRec))
    k = np.arange(n)
    rec["start_ns"] = B + 1000 + 777 * k
    rec["end_ns"] = rec["start_ns"] + rng.integers(0, 100000, n)
    rec["resource"] = 5 + k // 37 % 5
    rec["device"] = 4242
    rec["id"] = k + 1
    rec["name_id"] = np.array(names)[rng.integers(0, len(names), n)]
    if long_names:
        rec["name_id"] = np.where(k % 8 != 0, names[8], rec["name_id"])
    kind = rng.integers(0, 4, n)
    rec["schema_id"] = np.array([abi.KTJ_NONE, plain, wide, text], dtype=np.uint32)[kind]
    rec["args_off"] = np.array([0, 0, 1, 5])[kind]
    flow = rng.integers(0, 3, n)
    rec["flow_id"], rec["flow_type"], rec["flags"] = np.where(flow, k + 1, 0), 1, flow == 1
    place = np.empty(n, dtype=np.int64)
    place[np.lexsort((rec["start_ns"], rec["resource"]))] = k   # of each in the document
    left = np.isin(place % 800, (0, 15, 16, 17, 399)) | (place == n - 1) | (rng.integers(0, 200, n) == 0)
    if left_known:
        rec["end_ns"] = np.where(left, rec["start_ns"] + 10**10, rec["end_ns"])
    else:
        rec["schema_id"] = np.where(left, plain, rec["schema_id"])
        rec["args_off"] = np.where(left, 7, rec["args_off"])
    assert 0 < left.sum() * 32 < n
    held = (abi.GenericRec * n).from_buffer_copy(rec.tobytes())
    sp.contents.generic, sp.contents.n_generic = C.cast(held, type(sp.contents.generic)), n
    sp.held = held
    return sp, int(left.sum())


def _gpu_vs_oracle(sp, passes=3):
    """Through the large passes whatever the size, several times from one engine; what each says of itself (KTJ_DBG_PASS)."""
    from kineto_amd.engine import TraceEngine
    lib = abi.load_engine()
    o = og.OracleRun(sp)
    want = o.output()
    o.close()
    lib.ktj_debug_force_sort_passes(1)
    try:
        with TraceEngine(sp.contents.trace_name.decode(), base_time_ns=sp.contents.base_time_ns, cuda12_args=sp.contents.create_flags != 0) as e:
            e.submit_stream(sp)
            info = []
            for _ in range(passes):
                e.process()
                assert e.output() == want
                info.append([int(x) for x in e.debug("pass_info")])
            return info
    finally:
        lib.ktj_debug_force_sort_passes(0)


@pytest.mark.gpu
@pytest.mark.parametrize("back", (28 * HOUR, LEAD - 10**9, LEAD - 2001 * 1000, 62 * DAY, B))
def test_woven_documents_long_behind_the_base(back):
    """Times with a lead, and (the second and third) its carry between activities of one track and one turn."""
    _gpu_vs_oracle(_base_back(edge_stream(2053, False), back))
    for cfg in (2, 3):
        sp, release = abi.synth_stream(cfg, 3001, host_name="box")
        _gpu_vs_oracle(_base_back(sp, back), passes=2)
        release()


@pytest.mark.gpu
@pytest.mark.parametrize("other_types", (False, True))
@pytest.mark.parametrize("n", (1, 3, 15, 16, 17, 40, 255, 257, 2053, 9001))
def test_woven_documents_at_the_edges(n, other_types):
    """Through the large passes whatever the size; the document three times from one engine, so that later passes meet used buffers.
    With other types the first pass leaves all activities to the other kernel, without them it leaves those with no room; the
    second makes no text rows where too many had none."""
    _gpu_vs_oracle(edge_stream(n, other_types))


@pytest.mark.gpu
def test_documents_with_one_row_left():
    """Known when decoded: the first pass of an engine makes no text row and does not wait for a second launch, the next are the shorter pass."""
    for name, sp in _odd_streams():
        print(name, flush=True)
        n = sp.contents.n_generic + sp.contents.n_runtime + sp.contents.n_device
        assert _gpu_vs_oracle(sp) == [[1, 1, n, 0]] + 2 * [[0, 0, 0, 0]], name


@pytest.mark.gpu
@pytest.mark.parametrize("n", (65537, 70000, 262144))
def test_several_turns_with_rows_left(n):
    """Few enough activities that any left make the next pass one without text rows; woven in the first.  (Whether that waited for
    those that are left depends on what the host knew of them by then.)"""
    sp, left = large_stream(n, False)
    first, second = _gpu_vs_oracle(sp, passes=2)
    assert first[:3] == [1, 0, left] and second == [0, 0, 0, 0]


@pytest.mark.gpu
@pytest.mark.parametrize("n, left_known, long_names", ((262145, True, False), (300007, False, False), (300007, True, True)))
def test_many_turns_with_few_rows_left(n, left_known, long_names):
    """Woven in every pass, the others behind; with long names the list of these is made twice in the first pass."""
    sp, left = large_stream(n, left_known, long_names)
    first, *later = _gpu_vs_oracle(sp)
    assert first[:3] == [1, 0, left] and later == 2 * [[1, 0, left, 0]]
    assert first[3] == 0 or not left_known


def short_stream(n):
    """n CPU ops whose texts are laid out in segments of a few bytes (names and strings of 0 to 9, of 58 to 70 and of 120 to 136
    characters, one word and less among them), at every alignment."""
    import numpy as np
    rng = np.random.default_rng(n)
    b = StreamBuilder(window=(B, B + 10**15), host_name="short")
    lengths = [*range(10), *range(58, 71), *range(120, 137)]
    names = np.array([b.s(_text(k, k)) for k in lengths])
    text = b.schema([("s", abi.F_STR, 1), ("y", abi.F_I64, 1)])
    raw = b.schema([(None, abi.F_RAW, 1)])
    values = rng.integers(0, 10**6, 512)
    values[::2] = names[rng.integers(0, len(names), 256)]
    b.arg_slots([int(v) for v in values])
    sp = b.build()
    rec = np.zeros(n, dtype=np.dtype(abi.GenericRec))
    k = np.arange(n)
    rec["start_ns"] = B + 10 * k
    rec["end_ns"] = rec["start_ns"] + rng.integers(0, 10**rng.integers(0, 7, n))
    rec["resource"], rec["device"], rec["id"] = 5 + k // 41 % 3, 42, k + 1
    rec["name_id"] = names[np.where(rng.integers(0, 3, n), rng.integers(0, 10, n), rng.integers(0, len(names), n))]
    rec["schema_id"] = np.array([abi.KTJ_NONE, text, raw], dtype=np.uint32)[rng.integers(0, 3, n)]
    rec["args_off"] = 2 * rng.integers(0, 256, n)
    held = (abi.GenericRec * n).from_buffer_copy(rec.tobytes())
    sp.contents.generic, sp.contents.n_generic = C.cast(held, type(sp.contents.generic)), n
    sp.held = held
    return sp


@pytest.mark.gpu
@pytest.mark.parametrize("n", (1, 2, 17, 1000, 30007, 524321))
def test_segments_of_a_few_bytes(n):
    """Several in one word of the document, and (the last) lines stored past the caches."""
    assert _gpu_vs_oracle(short_stream(n), passes=2)[1][0] == 1


@pytest.mark.gpu
def test_rows_left_that_no_pass_before_had():
    """Behind a wait of their own: the engine's last pass had none."""
    from kineto_amd.engine import TraceEngine
    sp, left = large_stream(300007, False)
    n, few = sp.contents.n_generic, 3000
    o = og.OracleRun(sp)
    want = o.output()
    o.close()
    size = C.sizeof(abi.GenericRec)
    records = C.string_at(sp.contents.generic, n * size)
    first = [k for k in range(few) if abi.GenericRec.from_buffer_copy(records, k * size).args_off != 7]
    then = sorted(set(range(n)) - set(first))
    halves = [(abi.GenericRec * len(x)).from_buffer_copy(b"".join(records[k * size:(k + 1) * size] for k in x)) for x in (first, then)]
    sp.contents.generic, sp.contents.n_generic = C.cast(halves[0], type(sp.contents.generic)), len(first)
    with TraceEngine(sp.contents.trace_name.decode()) as e:
        e.submit_stream(sp)
        e.process()
        assert [int(x) for x in e.debug("pass_info")] == [1, 0, 0, 0]
        e._chk(abi.load_engine().ktj_submit_records(e.h, abi.REC_GENERIC, halves[1], len(then)), "ktj_submit_records")
        e.process()
        assert [int(x) for x in e.debug("pass_info")] == [1, 0, left, 1]   # (no record says so)
        assert e.output() == want


@pytest.mark.gpu
def test_times_with_a_lead_each_are_not_woven():
    """Nearly every activity would end the run of its neighbours; a few that do (a row at time 0) do not matter to many."""
    b = StreamBuilder(base=0, window=(0, 1 << 62), host_name="apart")
    for k in range(700):
        b.add_generic("op", 0, (k << 61) // 700, ((k << 61) // 700) + 5, 1, 5, id=k + 1)
    assert _gpu_vs_oracle(b.build(), passes=2) == [[1, 1, 700, 0], [0, 0, 0, 0]]
    sp, left = large_stream(300007, False)
    rec = (abi.GenericRec * sp.contents.n_generic).from_address(C.addressof(sp.contents.generic.contents))
    for k in (1, 2, 999, 200001):
        rec[k].start_ns, rec[k].end_ns = 0, 17
    assert [x[:3] for x in _gpu_vs_oracle(_base_back(sp, B), passes=2)] == 2 * [[1, 0, left, ]]


@pytest.mark.gpu
def test_other_records_are_woven_again():
    """That a pass left too many is known of its records and not of others that are as many."""
    import torch
    from kineto_amd.engine import TraceEngine
    lib = abi.load_engine()
    lib.ktj_debug_force_sort_passes(1)
    try:
        b = StreamBuilder(window=(B, B + 10**13), host_name="odd")
        b.s("op")
        sp = b.build()
        with TraceEngine(sp.contents.trace_name.decode()) as e:
            e.submit_stream(sp)
            for typ, want in ((17, ([1, 1, 99], [0, 0, 0], [0, 0, 0])), (0, ([1, 0, 0], [1, 0, 0])), (17, ([1, 1, 99], [0, 0, 0]))):
                rec = (abi.GenericRec * 99)()
                for k, r in enumerate(rec):
                    r.start_ns, r.end_ns, r.resource, r.device, r.id, r.name_id, r.type, r.schema_id = B + k, B + k + 5, 5, 1, k + 1, 0, typ, abi.KTJ_NONE
                on_gpu = torch.frombuffer(bytearray(rec), dtype=torch.uint8).cuda()
                torch.cuda.synchronize()
                e._chk(lib.ktj_submit_records_device(e.h, abi.REC_GENERIC, on_gpu.data_ptr(), 99), "ktj_submit_records_device")
                for info in want:
                    e.process()
                    assert [int(x) for x in e.debug("pass_info")][:3] == info, typ
                    assert e.output().count(b'"cat": "cpu_op"') == (99 if typ == 0 else 0)
    finally:
        lib.ktj_debug_force_sort_passes(0)


@pytest.mark.gpu
def test_pass_without_room_for_text_rows():
    """It is made again with the shorter rows, and the next passes over these records do not try."""
    from kineto_amd.engine import EngineError, TraceEngine
    lib = abi.load_engine()
    sp = edge_stream(4001, False)
    o = og.OracleRun(sp)
    want = o.output()
    o.close()

    def process(e, failing):
        """How many of that many failing allocations the pass met."""
        lib.ktj_debug_fail_allocations(failing)
        try:
            e.process()
        finally:
            left = lib.ktj_debug_fail_allocations(0)
        return failing - left, int(e.debug("pass_info")[0])

    lib.ktj_trim(0)   # (a new engine would take the memory of the one before)
    with TraceEngine(sp.contents.trace_name.decode()) as e:
        e.submit_stream(sp)
        assert process(e, 1) == (1, 0)
        assert e.output() == want
        for _ in range(2):
            assert process(e, 1) == (0, 0)
            assert e.output() == want
        one = (abi.GenericRec * 1).from_buffer_copy(C.string_at(sp.contents.generic, C.sizeof(abi.GenericRec)))
        e._chk(lib.ktj_submit_records(e.h, abi.REC_GENERIC, one, 1), "ktj_submit_records")
        assert process(e, 0) == (0, 1)   # other records are tried again
    lib.ktj_trim(0)
    with TraceEngine(sp.contents.trace_name.decode()) as e:   # no room either way
        e.submit_stream(sp)
        with pytest.raises(EngineError):
            process(e, 2)
        e.process()
        assert e.output() == want and int(e.debug("pass_info")[0]) == 1


