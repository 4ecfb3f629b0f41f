"""sddmm_gpu when an allocation fails part of the way (host_call_stub.cpp), on the CPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_a_failed_call_leaves_nothing_on_the_streams(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    obj, exe = str(tmp_path / "stub.o"), str(tmp_path / "stub")
    subprocess.run([hipcc, "-O1", "-std=c++20", "-fPIC", "-fuse-cuid=none", "--offload-host-only", "-x", "hip", "-c", "-o", obj,
                    os.path.join(HERE, "host_call_stub.cpp")], check=True, timeout=120)
    subprocess.run(["g++", "-o", exe, obj, "-pthread"], check=True, timeout=60)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout + run.stderr
