"""The lookups of the playout kernels' lane logic (remainders, slots of a square, move masks),
compiled for the host and checked entry by entry (tests/lane_tables_check.cpp)."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def build_and_run(source: str, out: str) -> str:
    if not (os.path.exists(HIPCC) or shutil.which("hipcc")):
        pytest.skip("hipcc not available")
    cmd = [HIPCC, "-O2", "-std=c++17", "-x", "hip", "--offload-host-only",
           "-I" + os.path.join(ROOT, "gpu_ai_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", source), "-o", out]
    for c in (cmd, [out]):
        proc = subprocess.run(c, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                              timeout=300)
        assert proc.returncode == 0, proc.stdout
    return proc.stdout


def test_lookups(tmp_path):
    out = build_and_run("lane_tables_check.cpp", str(tmp_path / "check"))
    assert "mismatches 0" in out and int(out.split()[1].rstrip(",")) > 2_000_000, out
