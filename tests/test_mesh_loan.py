"""The mesh extraction's kept memory after a call that failed half way, on the
CPU: mesh.hip's host side against a stand-in HIP runtime (cpp/mesh_loan_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "semantic_icpslam_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("mesh_loan")
    objs = []
    for src in (os.path.join(CSRC, "mesh.hip"), os.path.join(HERE, "cpp", "mesh_loan_check.cpp")):
        objs.append(str(d / (os.path.basename(src) + ".o")))
        r = subprocess.run([HIPCC, "-O1", "-fPIC", "-std=c++17", "--offload-host-only",
                            "--offload-arch=gfx950", "-x", "hip", "-c", src, "-o", objs[-1]],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
    exe = str(d / "check")
    # (the kernels' code, which the stand-in never looks at, stays unresolved)
    r = subprocess.run(["g++", *objs, "-Wl,--unresolved-symbols=ignore-in-object-files", "-o",
                        exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("failing_check", [0, 1, 2, 3])
@pytest.mark.parametrize("wait_fails", [0, 1])
def test_memory_is_lent_again_only_when_nothing_writes_it(check, failing_check, wait_fails):
    r = subprocess.run([check, str(failing_check), str(wait_fails)], capture_output=True,
                       text=True, timeout=60)
    assert r.stdout.strip() == "ok", r.stdout + r.stderr
