"""GPU: a stream submitted in one call: which of the calls that it stands for failed."""
import pytest

from kineto_amd import abi
from kineto_amd.engine import EngineError, TraceEngine

pytestmark = pytest.mark.gpu


def stream(**change):
    from stream_builder import B, StreamBuilder
    b = StreamBuilder()
    schema = b.schema([("x", change.get("field", abi.F_I64_ARRAY), 2)])
    b.add_generic("op", 0, B, B + 10, 1, 2, id=1, schema=schema, values=[3, 4])
    b.add_device(5, B + 20, B + 30, name="kernel")
    b.clock.device_mode = change.get("device_mode", 0)
    return b.build()


@pytest.mark.parametrize("change,call", [({"field": 999}, "ktj_register_schema"), ({"device_mode": 7}, "ktj_set_clock_model")])
def test_the_call_that_failed_is_named(change, call):
    sp = stream(**change)
    with TraceEngine("t.json") as eng:
        with pytest.raises(EngineError) as x:
            eng.submit_stream(sp)
        assert "rc=%d" % abi.KTJ_ERR_ARG in str(x.value) and call in str(x.value)


def test_the_records_that_were_refused_are_named():
    import torch
    sp = stream()
    on_device = torch.zeros(256, dtype=torch.uint8, device="cuda:0")
    with TraceEngine("t.json") as eng:
        assert eng.lib.ktj_submit_records_device(eng.h, abi.REC_DEVICE, on_device.data_ptr(), 1) == 0
        with pytest.raises(EngineError) as x:
            eng.submit_stream(sp)
        assert "rc=%d" % abi.KTJ_ERR_STATE in str(x.value) and "ktj_submit_records (device)" in str(x.value)
