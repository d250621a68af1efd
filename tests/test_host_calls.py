"""The library's host code (gpu_ai_amd/csrc/capi.cpp, mlp.cpp) without a device: built with stand-ins
for the HIP runtime and the launches (tests/hip_stub.hpp), which record what they are given, make an
allocation fail or choose a kernel's time."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CSRC = os.path.join(ROOT, "gpu_ai_amd", "csrc")


def _sh(cmd: list[str]) -> str:
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                          timeout=300)
    assert proc.returncode == 0, proc.stdout
    return proc.stdout


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    """Builds a check program over the host code and runs it."""
    if not (os.path.exists(HIPCC) or shutil.which("hipcc")):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("host_calls")

    def compiled(source: str) -> str:
        obj = str(out / (os.path.basename(source) + ".o"))
        if not os.path.exists(obj):
            _sh([HIPCC, "-O1", "-std=c++17", "-x", "hip", "--offload-host-only", "-fPIC", "-I" + CSRC,
                 "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "tests"), "-c",
                 source, "-o", obj])
        return obj

    def run(source: str) -> str:
        exe = str(out / source[:-4])
        _sh(["g++", compiled(os.path.join(ROOT, "tests", source)),
             *(compiled(os.path.join(CSRC, s)) for s in ("capi.cpp", "mlp.cpp")), "-lpthread",
             "-o", exe])
        return _sh([exe])

    return run


def test_a_set_that_does_not_fit_leaves_none(check):
    out = check("dataset_check.cpp")
    assert "failed allocations 4, null arguments 0, mismatches 0" in out, out


def test_routes_of_shaped_and_tuned_contexts(check):
    assert "mismatches 0" in check("tuning_check.cpp")


def test_the_time_of_an_epoch_is_all_of_it(check):
    assert "mismatches 0" in check("epoch_check.cpp")
