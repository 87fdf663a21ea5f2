"""Reading the state back when the runtime reports an error (csrc/
host_state.hip), on the CPU with a stand-in runtime: no copy may be under way
to the caller's array once the call has returned."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("readback") / "readback_errors")
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objs = []
    for src in ("volcano-ash3d_amd/csrc/host_state.hip", "tests/native/readback_errors.cpp"):
        objs.append(out + str(len(objs)) + ".o")
        subprocess.run([hipcc, "-x", "hip", "--cuda-host-only", "-O1", "-fPIC", "-std=c++17", "-I", "volcano-ash3d_amd/csrc",
                        "-c", src, "-o", objs[-1]], cwd=ROOT, check=True)
    subprocess.run(["g++", *objs, "-o", out, "-lpthread"], check=True)
    return out


@pytest.mark.parametrize("call,count", [("none", 0), ("copy", 0), ("copy", 3), ("copy", 9), ("record", 2), ("wait", 0),
                                        ("wait", 4)])
def test_no_copy_outlives_the_call(program, call, count):
    r = subprocess.run([program, call, str(count)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
