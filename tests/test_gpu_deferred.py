"""Plies that wait for the walk phase, on the device against the oracle: boards on which every game
of a wave has one at once (steps of two weights with long move lists, crowded capture boards with
many kings), from a walk phase per deferred ply to one of a full wave, for small and large
workgroups."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from gpu_ai_amd.engine import (POLICY_HEURISTIC, POLICY_HEURISTIC_NOISY, POLICY_RANDOM,
                               REFILL_QUEUE, REFILL_STATIC, Engine)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def shaped():
    with Engine(0) as eng:
        yield eng


def boards(dtype, n: int, kind: str) -> np.ndarray:
    rng = np.random.default_rng(len(kind) * 1000 + n)
    pos = np.zeros(n, dtype)
    for i in range(n):
        if kind == "steps":  # player 1: kings on rows 0-5, men before the far row
            kings = rng.choice(24, size=int(rng.integers(1, 11)), replace=False)
            men = 24 + rng.choice(4, size=int(rng.integers(1, 4)), replace=False)
            other = rng.choice(np.setdiff1d(np.arange(8), kings), size=1)
            pos["p1"][i] = sum(1 << int(s) for s in np.concatenate([kings, men]))
            pos["p2"][i] = sum(1 << int(s) for s in other)
            pos["kings"][i] = sum(1 << int(s) for s in kings)
        else:
            occ = rng.integers(0, 2**32) & (rng.integers(0, 2**32) | rng.integers(0, 2**32))
            side, kings = rng.integers(0, 2**32), rng.integers(0, 2**32) & rng.integers(0, 2**32)
            pos["p1"][i], pos["p2"][i], pos["kings"][i] = occ & side, occ & ~side, occ & kings
            pos["turn"][i] = i & 1
    pos["counter"][5::11] = 49
    pos["counter"][7::13] = 50
    return pos


@pytest.mark.parametrize("policy", [POLICY_RANDOM, POLICY_HEURISTIC, POLICY_HEURISTIC_NOISY])
@pytest.mark.parametrize("kind", ["steps", "captures"])
@pytest.mark.parametrize("block,per_cu,refill,defer", [
    (64, 12, REFILL_QUEUE, 1), (64, 12, REFILL_QUEUE, 64), (256, 3, REFILL_STATIC, 16),
    (1024, 1, REFILL_QUEUE, 33)])
def test_deferred_plies(shaped, oracle, policy, kind, block, per_cu, refill, defer):
    per = 67  # a wave plays one board's games or two boards'
    pos = boards(oracle.start_positions(1, 1, 0, 1, False).dtype, 96, kind)
    w, tr = oracle.run_playouts(pos, per_pos=per, seed=5, epoch=6, policy=policy)
    shaped.set_tuning(block_size=block, blocks_per_cu=per_cu, refill=refill, defer_min=defer)
    print(f"[gpu] deferred plies: {kind}, policy {policy}, {block}x{per_cu}, refill {refill}, "
          f"threshold {defer}", file=sys.stderr, flush=True)
    res = shaped.run_playouts(pos, per_pos=per, seed=5, epoch=6, policy=policy)
    assert res.stats["block_size"] == block
    assert np.array_equal(res.winners, w)
    assert res.stats["plies"] == int(tr["plies"].sum(dtype=np.uint64))
    assert res.stats["max_moves"] == int(tr["max_n"].max())


@pytest.mark.parametrize("policy", [POLICY_RANDOM, POLICY_HEURISTIC, POLICY_HEURISTIC_NOISY])
@pytest.mark.parametrize("kind", ["steps", "captures"])
def test_the_same_with_a_wave_per_game(oracle, policy, kind):
    pos = boards(oracle.start_positions(1, 1, 0, 1, False).dtype, 300, kind)
    with Engine(0) as eng:
        print(f"[gpu] a wave per game: {kind}, policy {policy}", file=sys.stderr, flush=True)
        res = eng.run_playouts(pos, per_pos=25, seed=6, epoch=7, policy=policy)
    assert res.stats["grid_blocks"] == 300 * 25
    w, tr = oracle.run_playouts(pos, per_pos=25, seed=6, epoch=7, policy=policy)
    assert np.array_equal(res.winners, w)
    assert res.stats["plies"] == int(tr["plies"].sum(dtype=np.uint64))
    assert res.stats["max_moves"] == int(tr["max_n"].max())
