"""mi_run_playouts_noalloc with counts in device memory around one game a wave (3072 waves on 256
CUs), where its kernel goes from a game per wave to a game per lane, against mi_run_playouts."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_ai_amd.engine import POLICY_HEURISTIC, POLICY_HEURISTIC_NOISY, POLICY_RANDOM
from test_zz_no_alloc import _noalloc, announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("total", [0, 1, 63, 64, 65, 1000, 3071, 3072, 3073])
@pytest.mark.parametrize("policy", [POLICY_RANDOM, POLICY_HEURISTIC, POLICY_HEURISTIC_NOISY])
def test_counted_noalloc_around_a_game_per_wave(engine, golden, policy, total):
    pos = golden["positions"]["mid1024"][:90].copy()
    pos[7]["p1" if pos[7]["turn"] == 0 else "p2"] = 0  # the mover has lost
    pos[7]["kings"] &= pos[7]["p1"] | pos[7]["p2"]
    pos[9]["counter"] = 50  # a draw
    counts = np.bincount(np.random.default_rng(total).integers(0, 90, total) * 7 % 90,
                         minlength=90).astype(np.uint32)
    announce(f"counted noalloc of {total} games, policy {policy}")
    got, status = _noalloc(engine, pos, 0, counts, 31, 5, policy)
    assert status == 0
    if total:
        ref = engine.run_playouts(pos, counts=counts, seed=31, epoch=5, policy=policy)
        assert np.array_equal(got, ref.winners)
