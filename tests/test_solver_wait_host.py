"""The host's wait for the solver's scalars, without a device: it gives up the processor to other contexts' threads."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    out = str(tmp_path_factory.mktemp("host") / "host_solver_wait")
    # the device's code and the other files' stages are not built, and are not called
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-no-hip-rt", "-O1", "-std=c++17", "-pthread",
                    os.path.join(ROOT, "tests", "host_solver_wait.cpp"), "-o", out, "-Wl,--unresolved-symbols=ignore-all"],
                   check=True, timeout=120)
    return out


def _run(program, ms):
    res = subprocess.run([program, str(ms)], capture_output=True, text=True, timeout=20)
    assert res.returncode == 0, res.stderr
    word = res.stdout.split()
    return int(word[1]), int(word[3])


def test_a_long_wait_gives_up_the_processor(program):
    status, yields = _run(program, 50)
    assert status == 0 and yields > 0


def test_scalars_that_are_there_cost_no_system_call(program):
    assert _run(program, 0) == (0, 0)


def test_scalars_that_never_arrive_are_an_error(program):
    assert _run(program, -1)[0] == 2
