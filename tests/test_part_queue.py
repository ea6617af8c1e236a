"""CPU: the threads that copy a document's parts out as these arrive (kineto_amd/csrc/part_queue.h)."""
import ctypes as C
import os

import numpy as np
import pytest

SIM_SO = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_sim", "libktjsim.so")


def run(n_parts, arrive, threads, gap_us):
    lib = C.CDLL(SIM_SO)
    lib.ktjsim_part_queue.restype = None
    lib.ktjsim_part_queue.argtypes = [C.c_uint64, C.c_uint64, C.c_uint, C.c_uint, C.c_void_p, C.POINTER(C.c_double), C.POINTER(C.c_double)]
    taken, wall, cpu = np.zeros(n_parts, dtype=np.uint32), C.c_double(), C.c_double()
    lib.ktjsim_part_queue(n_parts, arrive, threads, gap_us, taken.ctypes.data, C.byref(wall), C.byref(cpu))
    return taken, wall.value, cpu.value


@pytest.mark.timeout(120)
@pytest.mark.parametrize("n_parts,threads,gap_us", [(1, 1, 0), (1, 6, 300), (2, 5, 300), (7, 5, 100), (1000, 5, 0), (200000, 6, 0), (2000, 1, 0), (500, 5, 60)])
def test_every_part_is_taken_once(n_parts, threads, gap_us):
    for _ in range(3):
        taken, _, _ = run(n_parts, n_parts, threads, gap_us)
        assert (taken == 1).all()


@pytest.mark.timeout(60)
@pytest.mark.parametrize("n_parts,arrive,gap_us", [(5, 0, 0), (5, 4, 0), (100, 30, 200), (100000, 99999, 0)])
def test_all_go_when_the_rest_is_given_up(n_parts, arrive, gap_us):
    taken, _, _ = run(n_parts, arrive, 5, gap_us)
    assert (taken[:arrive] <= 1).all() and (taken[arrive:] == 0).all()


def test_waiting_for_parts_does_not_keep_the_cores():
    """Parts 2 ms apart: five threads that waited awake would use five seconds of processor time per second."""
    taken, wall, cpu = run(200, 200, 5, 2000)
    assert (taken == 1).all() and wall >= 0.4
    assert cpu < 0.5 * wall
