"""The host's walk over the solver's storage order, cell by cell against the index function that the kernels use."""
import os
import shutil
import subprocess

from conftest import ROOT


def test_walk_equals_index_function(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    out = str(tmp_path / "host_rotated")
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-no-hip-rt", "-O1", "-std=c++17",
                    os.path.join(ROOT, "tests", "host_rotated.cpp"), "-o", out, "-Wl,--unresolved-symbols=ignore-all"],
                   check=True, timeout=120)
    # every remainder of a plane group, widths below, at and above the 64 columns of a tile and their multiples
    sizes = [(nx, 4 + nx % 3, nz) for nx in (4, 5, 6, 7, 8, 15, 16, 31, 59, 60, 61, 62, 63, 64, 65, 127, 130)
             for nz in (3, 4, 5, 64, 65, 66, 67, 129, 131)]
    res = subprocess.run([out, *(str(v) for s in sizes for v in s)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
    assert int(res.stdout) == sum(a * b * c for a, b, c in sizes)
