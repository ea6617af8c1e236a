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
