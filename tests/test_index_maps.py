"""Which item of a launch owns which rows and columns: the index arithmetic of
the kernels' work maps, compiled for the host from the headers that the library
is built from and checked against plain divisions and an exact cover of the
grid, over far more sizes than any GPU test runs."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not found")
@pytest.mark.parametrize("name", ["stage_map", "flux_items"])
def test_every_point_has_one_owner(name, tmp_path):
    exe = tmp_path / name
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17",
                    os.path.join(HERE, "native", f"{name}_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.rstrip().endswith(" bad 0"), r.stdout
