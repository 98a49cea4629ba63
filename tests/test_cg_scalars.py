"""The CG driver reads its final scalars after a wait for the stream, not on
sight of the done flags that a kernel still running may show
(tests/cg_scalars_check.cpp: the driver on the CPU against a stand-in runtime)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
PKG = os.path.join(ROOT, "geoflow_amd")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("cg") / "cg_scalars_check")
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "--cuda-host-only", "-O1",
                    "-std=c++17", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(PKG, "csrc"), "-x", "hip",
                    os.path.join(HERE, "cg_scalars_check.cpp"), "-rdynamic",
                    "-L" + PKG, "-lgeoflow_hip", "-Wl,-rpath," + PKG, "-o", out],
                   check=True, capture_output=True)
    return out


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("systems", ["single", "batched"])
def test_final_scalars_follow_a_stream_wait(exe, systems, precision):
    r = subprocess.run([exe, systems, precision], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
