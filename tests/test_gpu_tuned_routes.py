"""A context that was tuned on one large batch and on small sizes: every size takes a route as fast as
an untuned context's, with the oracle's games."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from gpu_ai_amd.engine import POLICY_HEURISTIC_NOISY, POLICY_RANDOM, Engine

pytestmark = pytest.mark.gpu


def announce(msg: str) -> None:
    print(f"[gpu] {msg}", file=sys.stderr, flush=True)


@pytest.mark.parametrize("policy", [POLICY_RANDOM, POLICY_HEURISTIC_NOISY])
def test_sizes_of_a_tuned_context(oracle, policy):
    pos = oracle.start_positions(2016, 1024, 0, 30, False)
    with Engine(0) as eng, Engine(0) as plain:
        announce(f"mi_autotune on 1024 x 256, policy {policy}")
        best, _ = eng.autotune(pos, per_pos=256, policy=policy, reps=1)
        for total in (256, 4095, 16384, 70000):
            counts = np.full(1024, total // 1024, np.uint32)
            counts[:total % 1024] += 1
            announce(f"{total} playouts, policy {policy}")
            r = eng.run_playouts(pos, counts=counts, seed=4, epoch=2, policy=policy)
            u = plain.run_playouts(pos, counts=counts, seed=4, epoch=2, policy=policy)
            for key in ("block_size", "grid_blocks", "refill"):
                assert r.stats[key] == u.stats[key], (total, key)
            w, _ = oracle.run_playouts(pos, counts=counts, seed=4, epoch=2, policy=policy, traces=False)
            assert np.array_equal(r.winners, w), total
        assert eng.run_playouts(pos, per_pos=256, policy=policy).stats["block_size"] == best["block_size"]
        announce("mi_autotune_sizes 64, 1024, 2048")
        for e in eng.autotune_sizes(pos, [64, 1024, 2048], policy=policy, reps=3):
            # a wave per game takes less than three fifths of the time at all of these
            assert e["blocks_per_cu"] == 0 and e["block_size"] == 64, e
        for total in (64, 1500, 2048):
            counts = np.full(1024, total // 1024, np.uint32)
            counts[:total % 1024] += 1
            r = eng.run_playouts(pos, counts=counts, seed=5, epoch=3, policy=policy)
            assert r.stats["grid_blocks"] == total and r.stats["block_size"] == 64
            w, _ = oracle.run_playouts(pos, counts=counts, seed=5, epoch=3, policy=policy, traces=False)
            assert np.array_equal(r.winners, w), total
            with eng.graph(1024, 70000, policy) as g:
                assert np.array_equal(g.run(pos, counts, seed=5, epoch=3).winners, w)
