"""The sort's last launch makes the rows of CPU ops and kernels as well (k_finish_and_rows): documents against the oracle where its
workgroups are of every kind, with groups that are put into order there and with one that has the order made again."""
import ctypes as C

import numpy as np
import pytest

from kineto_amd import abi
from kineto_amd.engine import TraceEngine
from stream_builder import B
from test_gpu_sort_finish import ALL_BITS, groups, left_to_the_last_launch, ops, same_as_oracle

pytestmark = pytest.mark.gpu


def ops_and_kernels(n_ops, n_kernels, size, order):
    """The groups' rows on three threads, and kernels on three streams in groups of their own."""
    sp = ops(*groups(max(n_ops, 1), size, order))
    sp.contents.n_generic = n_ops
    ts, stream = groups(n_kernels, size, order, seed=2)
    rec = np.zeros(n_kernels, dtype=np.dtype(abi.DeviceRec))
    rec["begin"], rec["end"], rec["stream"], rec["id"] = ts, ts + 3 + np.arange(n_kernels) % 700, stream, np.arange(n_kernels) + 10**6
    rec["name_id"], rec["queue"] = np.arange(n_kernels) % 7, 1
    held = (abi.DeviceRec * n_kernels).from_buffer_copy(rec.tobytes())
    sp.contents.device, sp.contents.n_device = C.cast(held, type(sp.contents.device)), n_kernels
    sp._held += (held,)
    return sp


@pytest.mark.parametrize("size, order", ((1, "forwards"), (256, "backwards"), (257, "halves")))
@pytest.mark.parametrize("n_ops, n_kernels", ((4096, 1), (1, 4500), (0, 4097), (257, 98304 - 257), (98304, 1), (40000, 70001), (600000, 500000)))
def test_rows_come_with_the_sorts_last_launch(n_ops, n_kernels, size, order):
    print(n_ops, n_kernels, size, order, flush=True)
    info = same_as_oracle(ops_and_kernels(n_ops, n_kernels, size, order))
    if size > 256:
        assert info == ALL_BITS
    else:
        left_to_the_last_launch(info)


@pytest.mark.parametrize("n", (393215, 393216, 2**20 - 1, 2**20, 2**21 - 1, 2**21))
def test_tiles_of_each_size(n):
    """The fewest and the most keys of tiles of 512, 1024, 2048 and 4096 each."""
    print(n, flush=True)
    left_to_the_last_launch(same_as_oracle(ops(*groups(n, 97, "shuffled", threads=5))))


def test_the_last_launchs_bytes_are_counted_with_its_time():
    """12 bytes a row, under the rows' stage where they are made there, and under the sort's otherwise."""
    sp = ops_and_kernels(4096, 4096, 3, "backwards")
    counted = []
    for as_tiles in (False, True):
        with TraceEngine(sp.contents.trace_name.decode(), tile_emit=as_tiles) as e:
            e.submit_stream(sp)
            e.process()
            counted.append([int(e.stats().stage_bytes[abi.STAGE_NAMES.index(k)]) for k in ("sort", "size")])
    assert counted[1][0] == 56 * 8192 and counted[0][0] == 44 * 8192
    assert sum(counted[0]) == sum(counted[1])
