"""Device rows take the number of their (device, stream) pair where the sort gathers its values (k_collect_distinct): documents against
the oracle with few and with more pairs than a workgroup remembers, in runs and in any order, with queues in the place of streams, with
and without runtime rows that carry streams, and where the spans of user annotations need the numbers before."""
import numpy as np
import pytest

import oracle_glue as og
from kineto_amd.engine import TraceEngine
from stream_builder import B, StreamBuilder

pytestmark = pytest.mark.gpu


def stream(n, pairs, runs, carried, spans=False, seed=9):
    rng = np.random.default_rng(seed)
    b = StreamBuilder(window=(B, B + 10**9), host_name="pairs")
    b.api(["hipLaunchKernel"], flow_start=[0])
    names = ["kernel%d" % k for k in range(5)]
    pair = np.arange(n) * pairs // n if runs else rng.integers(0, pairs, n)
    for k in range(n):
        p, begin = int(pair[k]), B + 1000 + int(rng.integers(0, 11 * 10**8))   # a few rows behind the window
        device, stream_of, queue = (-1, 0, 3, 2**31 - 1)[p % 4], p // 4 * 2654435761 + 1, 0
        if p % 3 == 1:
            stream_of, queue = 0, p // 4 + 1      # queues in their place
        elif p % 30 == 2:
            stream_of = 0                         # neither
        elif p % 30 == 5:
            stream_of = 2**64 - 1
        b.add_runtime(k + 1, begin - 900, begin - 800, 0, 4242, 5, kind=1, stream=7 if carried and k % 50 == 0 else 0)
        if spans:
            b.add_usercorr(k + 1, 1)
        if k % 11 == 0:
            b.add_memset(k + 1, begin, begin + 90, device=device, context=1, stream=stream_of & 0xFFFF, nbytes=64)
        else:
            b.add_device(k + 1, begin, begin + 500, domain=k % 2, op=1, device=device, name=names[k % 5], stream=stream_of, queue=queue)
    if spans:
        b.add_generic("annotation", 2, B + 10, B + 10**8, 4242, 5, id=1)
    return b.build()


def same_as_oracle(sp):
    ora = og.OracleRun(sp)
    want = ora.output()
    with TraceEngine(sp.contents.trace_name.decode()) as eng:
        eng.submit_stream(sp)
        for turn in range(2):
            eng.process()
            assert eng.output() == want, turn
    ora.close()


@pytest.mark.parametrize("carried", (True, False))
@pytest.mark.parametrize("runs", (True, False))
@pytest.mark.parametrize("pairs", (1, 6, 900, 3000))
def test_pairs(pairs, runs, carried):
    print(pairs, runs, carried, flush=True)
    same_as_oracle(stream(9001, pairs, runs, carried))


@pytest.mark.parametrize("n", (1025, 2047, 40001))
def test_sizes(n):
    print(n, flush=True)
    same_as_oracle(stream(n, 40, False, True))


@pytest.mark.parametrize("pairs", (6, 900))
def test_with_spans(pairs):
    print(pairs, flush=True)
    same_as_oracle(stream(3001, pairs, False, True, spans=True))
