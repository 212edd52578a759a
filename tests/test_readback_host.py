"""The host side of the copies to host memory (fsim_readback.hip) over a stand-in runtime: the pinned memory it asks for,
its waits and its threads, without a device."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    out = str(tmp_path_factory.mktemp("host") / "host_readback")
    # the device's code is not built, and is not called
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-no-hip-rt", "-O1", "-std=c++17", "-pthread",
                    os.path.join(ROOT, "tests", "host_readback.cpp"), "-o", out, "-Wl,--unresolved-symbols=ignore-all"],
                   check=True, timeout=120)
    return out


def _run(program, *args):
    res = subprocess.run([program, *args], capture_output=True, text=True, timeout=20)
    assert res.returncode == 0, res.stderr
    return res.stdout.splitlines()


@pytest.mark.parametrize("threads", ["team", "alone"])
def test_pinned_memory_is_coherent(program, threads):
    """The host polls flags and copies data while later kernels run: only coherent memory promises that they are there
    before the stream is synchronised."""
    lines = _run(program, "memory", threads)
    assert lines[0].split("mallocs")[0].strip() == f"copy {67 << 20} status 0 whole 1"
    assert lines[1] == "flags coherent 1 portable 1 noncoherent 0"
    assert lines[2] == "end mallocs 1 frees 1"


# of 34 pieces through 12 slots: the first, the last of the first round, one whose slot is not needed again, the last
@pytest.mark.parametrize("piece", [0, 11, 12, 25, 33])
@pytest.mark.parametrize("threads", ["team", "alone"])
def test_a_piece_that_never_arrives_ends_the_copy(program, threads, piece):
    """A stream that has finished without a piece's flag is an error, and not a wait without end."""
    lines = _run(program, "lost", threads, str(piece))
    assert lines[0].split()[3] == "2" and "arrive" in lines[1]
    # and the next copy is whole again
    assert lines[2].split()[3:6] == ["0", "whole", "1"]
    assert lines[3] == "end mallocs 1 frees 1"


def test_small_results_take_the_runtimes_plain_copy(program):
    """A copy on the stream and its synchronisation cost a result of a few KB half as much again."""
    sizes = [1, 4096, 100_000, (1 << 20) - 1]
    lines = _run(program, "direct", *map(str, sizes))
    assert all(v.split()[3:6] == ["0", "whole", "1"] for v in lines[0:-1:2])
    assert lines[1:-1:2] == ["plain 1 on the stream 0"] * len(sizes)
