"""CPU test of the arrival counters (csrc/arrival_counter.h) that decide which workgroup of a tile finishes it."""
import ctypes
import itertools
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def weight(tmp_path_factory):
    """rf::arrival_weight, compiled for the host."""
    d = tmp_path_factory.mktemp("arrival")
    src = d / "weight.cpp"
    src.write_text('#include "%s"\nextern "C" unsigned weight(unsigned part, unsigned parts) '
                   '{ return rf::arrival_weight(part, parts); }\n'
                   % os.path.join(ROOT, "radeonflow_kernels_amd", "csrc", "arrival_counter.h"))
    so = str(d / "weight.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", so, str(src)], check=True)
    f = ctypes.CDLL(so).weight
    f.argtypes, f.restype = [ctypes.c_uint, ctypes.c_uint], ctypes.c_uint
    return f


def _arrive(weight, counter, part, parts):
    now = (counter + weight(part, parts)) & 0xffffffff
    return now, now == 0


def test_exactly_the_last_arrival_of_a_launch_finds_zero(weight):
    """Every order of up to six parts, and random orders of many."""
    rng = random.Random(1)
    orders = [o for parts in range(2, 7) for o in itertools.permutations(range(parts))]
    orders += [rng.sample(range(parts), parts) for parts in (7, 8, 14, 56, 4096) for _ in range(20)]
    for order in orders:
        counter, last = 0, []
        for part in order:
            counter, is_last = _arrive(weight, counter, part, len(order))
            last.append(is_last)
        assert last == [False] * (len(order) - 1) + [True] and counter == 0, order


def test_launches_that_overlap_on_a_counter_leave_it_at_zero(weight):
    """Two to four launches of different numbers of parts, arrivals mixed at random: the counter ends at zero, so the next
    launch on it is right again (a count that wraps at each launch's own limit does not: 2 and 4 parts can end at 4)."""
    rng = random.Random(2)
    for _ in range(3000):
        launches = [rng.randint(2, 14) for _ in range(rng.randint(2, 4))]
        arrivals = [(part, parts) for parts in launches for part in range(parts)]
        rng.shuffle(arrivals)
        counter = 0
        for part, parts in arrivals:
            counter, _ = _arrive(weight, counter, part, parts)
        assert counter == 0, launches
