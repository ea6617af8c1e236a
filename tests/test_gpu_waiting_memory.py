"""GPU: the device memory that a destroyed engine leaves for the next one is bounded and given back: behind engines
that need little, and when the program asks for it."""
import ctypes as C

import pytest

from kineto_amd import abi
from kineto_amd.engine import TraceEngine

pytestmark = pytest.mark.gpu
MIB = 1 << 20
ROUNDING = 8 * MIB  # what the runtime may hold beside: it hands out pages of 2 MiB


def free_bytes():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def session(config, rows, args_slots=0):
    sp, release = abi.synth_stream(config, rows, host_name="waiting")
    with TraceEngine("t.json") as eng:
        eng.submit_stream(sp)
        if args_slots:
            blob, first = (C.c_uint64 * args_slots)(), C.c_uint64()
            eng._chk(eng.lib.ktj_submit_args(eng.h, blob, args_slots, C.byref(first)), "ktj_submit_args")
        eng.process()
        doc = eng.output()
    release()
    return doc


def trim():
    assert abi.load_engine().ktj_trim(0) == 0


def test_trim_gives_back_what_waits():
    assert abi.load_engine().ktj_trim(77) == 0          # no engine has been on such a device: nothing to give back
    first = session(4, 120000)
    trim()
    before = free_bytes()
    assert session(4, 120000) == first                  # from a set without device memory
    held = before - free_bytes()
    assert held > 64 * MIB - ROUNDING, "the test's session leaves too little to tell anything"
    assert held <= (512 + 64) * MIB + ROUNDING
    trim()
    assert abs(before - free_bytes()) <= ROUNDING
    trim()
    with TraceEngine("t.json"):                         # a set in use is not touched
        trim()
    assert session(4, 120000) == first


@pytest.mark.parametrize("mib", [20, 24, 28, 31])
def test_input_memory_is_bounded(mib):
    """An array of so many MiB gets room for twice as much from the engine that follows, 64 MiB at most."""
    want = session(1, 5)
    trim()
    before = free_bytes()
    assert session(1, 5, args_slots=mib * MIB // 8) == want
    assert before - free_bytes() <= 64 * MIB + ROUNDING
    assert session(1, 5, args_slots=mib * MIB // 8) == want
    assert before - free_bytes() <= 64 * MIB + ROUNDING
    trim()


def test_engines_that_need_little_give_back():
    want = session(1, 5)
    trim()
    before = free_bytes()
    session(4, 120000, args_slots=18 * MIB // 8)   # room for its inputs grows to some 64 MiB
    assert before - free_bytes() > 100 * MIB
    for _ in range(17):
        assert session(1, 5) == want
    assert before - free_bytes() <= ROUNDING
