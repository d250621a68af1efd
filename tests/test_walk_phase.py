"""The plies that wait for the playout kernel's walk phase, compiled for the host and checked against
the oracle's traces (tests/walk_phase_check.cpp): the functions that the kernel's lanes run."""
from __future__ import annotations

import os
import re
import subprocess

from test_lane_logic_host import HIPCC, ROOT, _link, _run

import pytest


@pytest.fixture(scope="module")
def checker_obj(tmp_path_factory, oracle):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    obj = str(tmp_path_factory.mktemp("walk") / "check.o")
    _run([HIPCC, "-O2", "-std=c++17", "-x", "hip", "--offload-host-only",
          "-I" + os.path.join(ROOT, "gpu_ai_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
          "-I" + os.path.join(ROOT, "oracle"), "-c",
          os.path.join(ROOT, "tests", "walk_phase_check.cpp"), "-o", obj])
    return obj


def test_waiting_plies_match_oracle(checker_obj):
    exe = _link(checker_obj, os.path.join(ROOT, "oracle", "liboracle.so"), checker_obj[:-2])
    proc = subprocess.run([exe, "2048"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                          timeout=300)
    assert proc.returncode == 0 and "mismatches 0" in proc.stdout, proc.stdout
    counts = list(map(int, re.findall(r"(?:captures|steps|walks) (\d+)", proc.stdout)))
    assert min(counts) > 500, proc.stdout


@pytest.mark.parametrize("k", [3, 5, 7, 8])
def test_planted_oracle_mistake_is_caught(checker_obj, tmp_path, k):
    """Draw ply, heuristic ties, the noisy heuristic's sigma and the order of its draws."""
    so = str(tmp_path / f"liboracle_m{k}.so")
    _run(["gcc", "-O2", "-std=c11", "-fopenmp", "-fPIC", "-shared", f"-DOR_MUTATION={k}",
          os.path.join(ROOT, "oracle", "oracle.c"), "-o", so])
    exe = _link(checker_obj, so, str(tmp_path / "check"))
    proc = subprocess.run([exe, "256"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                          timeout=300)
    assert proc.returncode != 0 and "mismatches 0" not in proc.stdout, proc.stdout
