"""GPU: where a pass may put its document.  A caller's buffer belongs to the call it was given to: a later pass
leaves it alone, whichever way that pass goes, and a buffer in use as working memory never holds a document."""
import ctypes as C

import pytest

from kineto_amd import abi
from kineto_amd.engine import TraceEngine

pytestmark = pytest.mark.gpu


def oracle_document(sp):
    import oracle_glue as og
    ora = og.OracleRun(sp)
    want = ora.output()
    ora.close()
    return want


def same(got, want):
    """(not a plain assert on megabytes, whose report would take minutes)"""
    if got != want:
        at = next((k for k, (x, y) in enumerate(zip(got, want)) if x != y), min(len(got), len(want)))
        pytest.fail("%d bytes, expected %d; they differ at %d: %r instead of %r" % (
            len(got), len(want), at, got[max(0, at - 80):at + 80], want[max(0, at - 80):at + 80]))


def device_document(eng):
    p, n = C.c_void_p(), C.c_uint64()
    eng._chk(eng.lib.ktj_output_device(eng.h, C.byref(p), C.byref(n)), "ktj_output_device")
    return p.value, n.value


def with_stream_sync(n):
    from stream_builder import B, StreamBuilder
    b = StreamBuilder()
    for k in range(n):
        b.add_generic("op %d" % (k % 50), 0, B + k, B + k + 5, 1, k % 7, id=k + 1)
    b.add_generic("Stream Sync", 15, B + 100, B + 105, 0, 5, id=n + 1)
    return b.build()


# three launches; in one go; step by step; and the debug read-back, which processes a small trace once more
@pytest.mark.parametrize("way", ["small", "one_go", "stepwise", "debug"])
def test_process_leaves_the_buffer_of_an_earlier_call_alone(way):
    import torch
    release = lambda: None
    if way == "stepwise":
        sp = with_stream_sync(5000)
    else:
        sp, release = abi.synth_stream(1, 3000 if way == "one_go" else 200, host_name="owner")
    want = oracle_document(sp)
    with TraceEngine(sp.contents.trace_name.decode(), base_time_ns=sp.contents.base_time_ns) as eng:
        eng.submit_stream(sp)
        out = torch.full((len(want) + 4096,), 0xEE, dtype=torch.uint8, device="cuda:0")
        n = C.c_uint64()
        rc = eng.lib.ktj_process_noalloc(eng.h, eng.end_time_ns, out.data_ptr(), out.numel(), C.byref(n))
        assert rc == 0, eng.lib.ktj_last_error(eng.h)
        assert device_document(eng) == (out.data_ptr(), len(want))
        same(bytes(out[:n.value].cpu().numpy()), want)
        out.fill_(0xA5)                       # the caller uses its memory for something else
        torch.cuda.synchronize()
        eng.debug("perm") if way == "debug" else eng.process()
        torch.cuda.synchronize()
        assert bool((out == 0xA5).all()), "a later pass wrote into the buffer of an earlier call"
        at, length = device_document(eng)
        assert length == len(want) and not out.data_ptr() <= at < out.data_ptr() + out.numel()
        same(eng.output(), want)
    release()


# three launches; in one go; in one go as far as that goes, then step by step
@pytest.mark.parametrize("way", ["small", "one_go", "stepwise"])
def test_a_buffer_that_is_too_short_stays_as_it_was(way):
    import torch
    release = lambda: None
    if way == "stepwise":
        sp = with_stream_sync(5000)
    else:
        sp, release = abi.synth_stream(1, 3000 if way == "one_go" else 200, host_name="owner")
    want = oracle_document(sp)
    with TraceEngine(sp.contents.trace_name.decode(), base_time_ns=sp.contents.base_time_ns) as eng:
        eng.submit_stream(sp)
        out = torch.full((len(want) + 4096,), 0xA5, dtype=torch.uint8, device="cuda:0")
        n = C.c_uint64()
        for cap in (len(want) // 2, len(want) + 63, 16):
            for _ in range(2):
                rc = eng.lib.ktj_process_noalloc(eng.h, eng.end_time_ns, out.data_ptr(), cap, C.byref(n))
                assert rc == abi.KTJ_ERR_LIMIT and n.value == len(want) and b"output buffer" in eng.lib.ktj_last_error(eng.h)
            assert bool((out == 0xA5).all()), "a part of the document in a buffer of %d bytes" % cap
        rc = eng.lib.ktj_process_noalloc(eng.h, eng.end_time_ns, out.data_ptr(), len(want) + 64, C.byref(n))
        assert rc == 0 and n.value == len(want)
        same(bytes(out[:n.value].cpu().numpy()), want)
        assert bool((out[n.value + 64:] == 0xA5).all())
    release()


def test_document_of_a_stepwise_pass_is_not_working_memory_of_the_next():
    """A few records with long names go step by step behind a pass that left much working memory; then many
    records with short names, whose document fits where the first one was."""
    import torch
    from stream_builder import B, StreamBuilder
    b = StreamBuilder()
    many, few = 100000, 2500
    b.s("long " * 700)
    b.s("short")
    b.s("Stream Sync")
    for k in range(many + few):
        r = b.add_generic(None, 0 if k != many else 15, B + k, B + k + 5, 0, k % 7, id=k + 1)
        r.name_id = 1 if k < many else 0 if k > many else 2
    sp = b.build()
    s = sp.contents
    records, size = C.addressof(s.generic.contents), C.sizeof(abi.GenericRec)
    host = (C.c_char * ((many + few) * size)).from_address(records)
    on_device = torch.frombuffer(bytearray(host), dtype=torch.uint8).cuda()
    with TraceEngine(s.trace_name.decode(), base_time_ns=s.base_time_ns) as eng:
        s.n_generic = 0
        eng.submit_stream(sp)
        for first, n in ((0, many), (many, few), (0, 30000), (many, few), (0, many)):
            print("records", first, n, flush=True)
            s.generic = C.cast(records + first * size, C.POINTER(abi.GenericRec))
            s.n_generic = n
            want = oracle_document(sp)
            eng._chk(eng.lib.ktj_submit_records_device(eng.h, abi.REC_GENERIC, on_device.data_ptr() + first * size, n), "submit")
            eng.process()
            same(eng.output(), want)
