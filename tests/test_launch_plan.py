"""The shapes of the class launches (tonto_amd/csrc/launch_plan.h), compiled for the CPU."""
import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tonto_amd", "csrc")
SOURCE = """
#include "launch_plan.h"
extern "C" void plan(long long *v, int n, long long slots) { plan_wave(reinterpret_cast<WavePlan *>(v), n, slots); }
"""


@pytest.fixture(scope="module")
def plan_lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + CSRC, str(d / "plan.cpp"), "-o",
                           str(d / "plan.so")])
    return ctypes.CDLL(str(d / "plan.so"))


def _plan(L, parts, slots):
    v = np.array([[b, c, 0, 0] for b, c in parts], dtype=np.int64)
    L.plan(v.ctypes.data_as(ctypes.c_void_p), ctypes.c_int(len(parts)), ctypes.c_longlong(slots))
    return [tuple(int(x) for x in r[2:]) for r in v]


def test_workspace_grids_fit_their_slots(plan_lib):
    rng = random.Random(3)
    for _ in range(3000):
        n = rng.randint(1, 16)
        parts = [(int(2 ** rng.uniform(0, 26)), int(2 ** rng.uniform(0, 20))) for _ in range(n)]
        slots = n + int(2 ** rng.uniform(0, 13)) - 1
        got = _plan(plan_lib, parts, slots)
        assert all(1 <= gx <= b and 1 <= gy <= c for (b, c), (gx, gy) in zip(parts, got))
        assert sum(gx * gy for gx, gy in got) <= slots
        if sum(b * c for b, c in parts) <= slots:
            assert got == parts


@pytest.mark.parametrize("parts,slots,least", [
    # a class pair of 2080 bra pairs, most of its kets in one of two parts: three ket chunks of a
    # bra pair at once there, as with the slots to itself
    ([(2080, 1536), (2080, 256)], 8192, 3 * 2080),
    ([(2080, 256), (2080, 1536), (1, 1)], 8192, 1024),
    # one part has all slots
    ([(100, 1000)], 8192, 8100)])
def test_workspace_slots_by_work(plan_lib, parts, slots, least):
    got = _plan(plan_lib, parts, slots)
    big = max(range(len(parts)), key=lambda k: parts[k][0] * parts[k][1])
    assert got[0][0] * got[0][1] >= min(least, parts[0][0] * parts[0][1])
    assert got[big][0] * got[big][1] >= slots // 2


def test_grids_without_workspace(plan_lib):
    # about 65536 work-groups a part, long prefixes split where there are few bra pairs
    assert _plan(plan_lib, [(10, 100), (100000, 7), (7, 100000)], 0) == [(10, 100), (100000, 1), (7, 9363)]
