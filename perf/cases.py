"""The work that a program has the trace engine do, as measurable cases.

A case is a workload (`config`, one of the five synthetic configurations: 1 small training trace,
2 kernels, copies and memsets with a clock model, 3 many streams with shuffled arrival, 4 graph
launches with fan-out and orphans, 5 string-heavy kernels with typed args), its size in device rows
(`rows`; configuration 5 has generic kernel records instead), and how the program goes about it
(`way`):

  pass    an engine that holds its records in device memory processes them and leaves the document
          there (a serving loop, the benchmark of this repository)
  trace   a profiling session from host memory to host memory: engine created, records and infos
          submitted, processed, the document's bytes taken, engine destroyed
  file    the same with the renamed trace file as its result, which is how libkineto writes a trace
"""
import ctypes as C
import os
import tempfile

import numpy as np
import torch

from kineto_amd import abi
from kineto_amd.engine import TraceEngine

FULL_ROWS = {1: 10000, 2: 1000000, 3: 10000000, 4: 11000000, 5: 5000000}
MOST_HOST_ROWS = 200000  # sessions whose document goes to the host: up to some 250 MB


def listed():
    return [
        # a handful of records: what every call costs whatever the trace holds
        {"name": "trace_15_records", "way": "trace", "config": 1, "rows": 5},
        {"name": "pass_15_records", "way": "pass", "config": 1, "rows": 5},
        # one training step of a small model: 30 000 records, a few threads and streams
        {"name": "trace_30k_records", "way": "trace", "config": 1, "rows": 10000},
        {"name": "pass_30k_records", "way": "pass", "config": 1, "rows": 10000},
        # a few steps of a job that replays graphs: few launches, 118 000 kernels, 60 MB of text
        {"name": "trace_graphs_118k", "way": "trace", "config": 4, "rows": 120007},
        # a short trace of kernels with long templated names and launch dimensions
        {"name": "trace_strings_4k", "way": "trace", "config": 5, "rows": 4001},
        # a usual trace file: kernels, copies and memsets, 90 000 records, 37 MB
        {"name": "file_mixed_90k", "way": "file", "config": 2, "rows": 30011},
        # a longer capture on many streams, an odd number of records
        {"name": "pass_streams_733k", "way": "pass", "config": 3, "rows": 333337},
        # a million device rows of each mix, and the ten-million-row captures of large jobs
        {"name": "pass_mixed_3m", "way": "pass", "config": 2, "rows": FULL_ROWS[2]},
        {"name": "pass_strings_5m", "way": "pass", "config": 5, "rows": FULL_ROWS[5]},
        {"name": "pass_graphs_11m", "way": "pass", "config": 4, "rows": FULL_ROWS[4]},
        {"name": "pass_streams_22m", "way": "pass", "config": 3, "rows": FULL_ROWS[3]},
    ]


def draw(rng):
    way = rng.choice(("pass", "pass", "trace", "file"))
    config = rng.randint(1, 5)
    most = FULL_ROWS[config] if way == "pass" else min(FULL_ROWS[config], MOST_HOST_ROWS)
    least = {3: 50, 4: 1100}.get(config, 5)  # below that configurations 3 and 4 hold next to nothing
    return {"way": way, "config": config, "rows": round(least * (most / least) ** rng.random())}


def _records(pointer, n, record):
    """A C array of records as a structured array on the same memory."""
    return np.frombuffer((C.c_char * (n * C.sizeof(record))).from_address(C.addressof(pointer.contents)), dtype=np.dtype(record))


def _other_values(s, seed):
    """Names, durations, launch dimensions and argument values dealt out to other rows for this seed.
    Each stays as often in the stream as the configuration says, so that the document keeps its
    length; what joins what, the streams and the order of arrival stay too."""
    rng = np.random.default_rng(seed)

    def deal(column, which=slice(None)):
        values = column[which]
        if len(values) > 1:
            column[which] = np.roll(values, int(rng.integers(1, len(values))), axis=0)

    def deal_durations(rec, begin, end, which=slice(None)):
        duration = rec[end] - rec[begin]
        deal(duration, which)
        rec[end] = rec[begin] + duration

    if s.n_generic:
        rec = _records(s.generic, s.n_generic, abi.GenericRec)
        deal(rec["name_id"])
        deal_durations(rec, "start_ns", "end_ns")
        deal(np.ctypeslib.as_array(s.args, shape=(s.n_generic, s.n_args // s.n_generic)))
    def inside(rec, mode):
        """Rows that the capture window keeps whatever duration of theirs they have."""
        offset = {0: 0, 1: s.clock.t0 - s.clock.t0_approx, 2: s.clock.async_offset}[mode]
        begin = rec["begin"].astype(np.int64) + offset
        longest = int((rec["end"] - rec["begin"]).max())
        return (begin > s.window_start_ns + 5000) & (begin + longest + 5000 < s.window_end_ns)

    if s.n_device:
        rec = _records(s.device, s.n_device, abi.DeviceRec)
        kernels = ((rec["domain"] & 0xFFFF) == 0) & inside(rec, s.clock.device_mode)
        if s.clock.device_mode == 2:  # an offset; a scaled clock would round other durations to other texts
            deal_durations(rec, "begin", "end", kernels)
        deal(rec["name_id"], kernels)
        if s.n_runtime == s.n_device:  # one launch per kernel, in the same order: both print its dimensions
            rec = _records(s.runtime, s.n_runtime, abi.RuntimeRec)
            launches = (rec["kind"] == 1) & inside(rec, s.clock.runtime_mode) & kernels
            deal(rec["u"]["kernel"]["grid"], launches)
            deal(rec["u"]["kernel"]["workgroup"], launches)


class _State:
    """What the program holds between passes; released with the last reference to it."""

    def __init__(self, case, seed):
        self.way = case["way"]
        self.engine, self.path = None, None
        self.stream, self._release = abi.synth_stream(case["config"], case["rows"], host_name="host")
        _other_values(self.stream.contents, seed)
        self.name = self.stream.contents.trace_name.decode()
        if self.way == "pass":
            self.engine = TraceEngine(self.name)
            self.engine.submit_stream(self.stream)
            torch.cuda.synchronize()
            self._free_stream()
        elif self.way == "file":
            # a file system in memory where there is one: the engine's part of the work, not a disk's
            top = "/dev/shm" if os.path.isdir("/dev/shm") and os.access("/dev/shm", os.W_OK) else tempfile.gettempdir()
            folder = os.path.join(top, "kineto_amd_cases_%d" % os.getuid())
            os.makedirs(folder, mode=0o700, exist_ok=True)
            self.path = os.path.join(folder, "trace_%d_%d_%d.json" % (case["config"], case["rows"], seed))

    def _free_stream(self):
        if self._release is not None:
            self._release()
            self.stream = self._release = None

    def __del__(self):
        if getattr(self, "engine", None) is not None:
            self.engine.close()
        if getattr(self, "_release", None) is not None:
            self._free_stream()
        if getattr(self, "path", None) is not None and os.path.exists(self.path):
            os.remove(self.path)


class _DeviceDocument:
    """The engine's document buffer for torch, without a copy; holds the state that owns it."""

    def __init__(self, state):
        p, n = C.c_void_p(), C.c_uint64()
        state.engine._chk(state.engine.lib.ktj_output_device(state.engine.h, C.byref(p), C.byref(n)), "ktj_output_device")
        self.state = state
        self.__cuda_array_interface__ = {"shape": (n.value,), "typestr": "|u1", "data": (p.value, False), "version": 2}


def _counters(engine):
    st = engine.stats()
    return [int(v) for v in (st.n_emitted, st.out_of_range_events, st.gpu_and_cpu_op_out_of_order, st.n_flow_events, st.n_linked, st.n_blank_names)]


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    if state.way == "pass":
        state.engine.process()
        return {"document": torch.as_tensor(_DeviceDocument(state), device="cuda"), "counters": _counters(state.engine)}
    if state.way == "trace":
        with TraceEngine(state.name, no_stage_times=True) as engine:
            engine.submit_stream(state.stream)
            engine.process()
            return {"document": np.frombuffer(engine.output(), dtype=np.uint8), "counters": _counters(engine)}
    with TraceEngine(state.path, no_file=False, no_stage_times=True) as engine:
        engine.submit_stream(state.stream)
        engine.finalize()
        return {"document": np.memmap(state.path, dtype=np.uint8, mode="r"), "counters": _counters(engine)}


def work(case):
    """The packed records, argument slots and strings once in, the document once out."""
    config, rows = case["config"], case["rows"]
    strings = {1: 14771, 2: 13278, 3: 320870, 4: 64297, 5: 2217666}[config]
    if config == 5:  # 64-byte record, nine argument slots; 1446 bytes of text each
        return {"bytes": strings + rows * (64 + 72 + 1446), "flops": 0}
    if config == 4:  # a launch (96), its op (64 + 32) and its correlation pair (16) per 550 device rows
        return {"bytes": strings + rows * 1.045 * (64 + 208 / 550 + 478), "flops": 0}
    ops = (rows + 4) // 5 if config == 3 else rows  # five launches per op in configuration 3
    text = {1: 1258, 2: 1250, 3: 1032}[config]
    return {"bytes": strings + ops * (64 + 32) + rows * (96 + 64 + 16 + text), "flops": 0}


def tolerance(case):
    return "exact"
