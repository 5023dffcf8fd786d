"""The library's own sources on the CPU (tests/emu): lanes as fibers, device memory and LDS under
the address sanitizer, the runtime's calls logged.  For what a GPU test cannot show safely:
launches beyond the hardware's limits, failing runtime calls, accesses out of range."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def emulated(tmp_path_factory):
    d = os.path.join(str(tmp_path_factory.mktemp("emu")), "build")
    r = subprocess.run([sys.executable, os.path.join(HERE, "emu", "build.py"), d], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    asan = subprocess.run(["g++", "-print-file-name=libasan.so"], capture_output=True, text=True).stdout.strip()
    env = dict(os.environ, TONTO_GPU_LIB=os.path.join(d, "libemu.so"), LD_PRELOAD=asan,
               ASAN_OPTIONS="detect_leaks=0:detect_stack_use_after_return=0", OMP_NUM_THREADS="1")

    def run(name, **more):
        r = subprocess.run([sys.executable, os.path.join(HERE, "emu", "checks.py"), name], capture_output=True,
                           text=True, env=dict(env, **more), timeout=600)
        print(r.stdout[-2000:])
        assert r.returncode == 0 and r.stdout.rstrip().endswith("passed"), r.stdout[-1500:] + r.stderr[-4000:]
    return run


def test_launch_limits(emulated):
    emulated("launch_limits")


def test_failing_runtime_calls(emulated):
    emulated("failing_runtime_calls")


def test_kept_workspace(emulated):
    emulated("kept_workspace")


def test_side_streams_per_stream(emulated):
    emulated("side_streams_per_stream")


def test_wavefront_forms(emulated):
    emulated("wavefront_forms")


def test_lane_forms(emulated):
    emulated("lane_forms")


def test_f_shells(emulated):
    emulated("f_shells")


def test_captured_by_the_caller(emulated):
    emulated("captured_by_the_caller")
