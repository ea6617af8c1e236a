"""GPU: the document on its way to the host (ktj_output_copy, the file sink) at the lengths where the
parts, the slots and the threads that share it change, against the page-locked copy of the same document."""
import os

import numpy as np
import pytest

from kineto_amd import abi
from kineto_amd.engine import TraceEngine

pytestmark = pytest.mark.gpu


# bytes of the document: one transfer; 128 KiB, 256 KiB and 512 KiB parts; more parts than slots
@pytest.mark.parametrize("config,rows", [(1, 5), (1, 400), (1, 420), (1, 1600), (1, 1700), (1, 6600), (1, 6700), (2, 13500), (2, 40000)])
def test_document_reaches_the_host_whole(tmp_path, config, rows):
    sp, release = abi.synth_stream(config, rows, host_name="copy")
    path = str(tmp_path / "trace.json")
    with TraceEngine(path, device=0) as eng:
        eng.submit_stream(sp)
        eng.process()
        first = eng.output()
        again = eng.output()          # other parts' numbers in the same slots
        want = eng.output_view()
        assert len(first) == len(want) and np.array_equal(np.frombuffer(first, dtype=np.uint8), want)
        assert again == first and eng.output() == first   # the last one from the page-locked copy
        n = abi.C.c_uint64()
        assert eng.lib.ktj_output_copy(eng.h, abi.C.create_string_buffer(16), 16, abi.C.byref(n)) == abi.KTJ_ERR_ARG
        assert n.value == len(first)
    with TraceEngine(path, device=0, no_file=False) as eng:
        eng.submit_stream(sp)
        assert eng.finalize() == len(first) == os.path.getsize(path)
        with open(path, "rb") as f:
            assert f.read() == first
    release()


def test_two_engines_copy_at_once(tmp_path):
    """Two threads, an engine each, their documents (more parts than slots, fewer) crossing at the same time, again and
    again into a buffer that held something else, and into a file."""
    import threading
    failures = []
    start = threading.Barrier(2)

    def work(name, config, rows):
        try:
            sp, release = abi.synth_stream(config, rows, host_name=name)
            path = str(tmp_path / (name + ".json"))
            with TraceEngine(path, device=0, no_file=False) as eng, TraceEngine(path, device=0) as other:
                other.submit_stream(sp)
                other.process()
                want = other.output_view()
                eng.submit_stream(sp)
                eng.process()
                dst, n = np.empty(len(want), dtype=np.uint8), abi.C.c_uint64()
                start.wait(60)
                for k in range(8):
                    dst.fill(k)
                    eng._chk(eng.lib.ktj_output_copy(eng.h, dst.ctypes.data, len(dst), abi.C.byref(n)), "ktj_output_copy")
                    assert n.value == len(want) and np.array_equal(dst, want), "copy %d of %s" % (k, name)
                assert eng.finalize() == len(want)
                assert np.array_equal(np.fromfile(path, dtype=np.uint8), want), "the file of " + name
            release()
        except BaseException as x:
            failures.append(x)
            start.abort()

    threads = [threading.Thread(target=work, args=a) for a in (("long", 2, 20000), ("short", 1, 6700))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
