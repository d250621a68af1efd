"""The capture plies' closed forms (every origin's capture tree as masks of origins), compiled for
the host and checked move by move against the depth-first walk (tests/capture_trees_check.cpp)."""
from __future__ import annotations

import re

from test_lane_tables import build_and_run


def test_capture_trees(tmp_path):
    out = build_and_run("capture_trees_check.cpp", str(tmp_path / "check"))
    plies, deep, moves = map(int, re.match(r"plies (\d+) \(deep (\d+)\), moves (\d+)", out).groups())
    assert "mismatches 0" in out and deep > 1000 and plies - deep > 100_000 and moves > 500_000, out
