"""The bound that keeps the first raycast pass inside the cube whose blocks it
can name, on the CPU, in the steps' own float arithmetic (cpp/ray_cube_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_samples_stay_in_the_cube(tmp_path):
    src, obj, exe = os.path.join(HERE, "cpp", "ray_cube_check.cpp"), tmp_path / "o", tmp_path / "x"
    for cmd in ([HIPCC, "-O1", "-fPIC", "-std=c++17", "-ffp-contract=off", "--offload-host-only",
                 "--offload-arch=gfx950", "-x", "hip", "-c", src, "-o", obj],
                ["g++", obj, "-Wl,--unresolved-symbols=ignore-in-object-files", "-o", exe]):
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.stdout.strip() == "ok", r.stdout + r.stderr
