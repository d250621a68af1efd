"""Small batches on the device: one wave per game (gpu_ai_amd/csrc/wave_playouts.hip) against the
oracle, over the sizes and layouts that take that route, and the size at which the route ends."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from gpu_ai_amd.engine import (POLICY_HEURISTIC, POLICY_HEURISTIC_NOISY, POLICY_RANDOM, Engine)
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu

POLICIES = [POLICY_RANDOM, POLICY_HEURISTIC, POLICY_HEURISTIC_NOISY]


def announce(msg: str) -> None:
    print(f"[gpu] {msg}", file=sys.stderr, flush=True)


@pytest.fixture(scope="module")
def fresh():
    with Engine(0) as eng:  # no shape given
        yield eng


def positions(oracle, n: int, seed: int) -> np.ndarray:
    """Openings, midgames, endgames with kings, and positions at the end of the draw count."""
    parts = [oracle.start_positions(seed + i, (n + 3) // 4, lo, hi, False)
             for i, (lo, hi) in enumerate(((0, 30), (20, 60), (60, 150), (30, 90)))]
    pos = np.stack(parts, axis=1).reshape(-1)[:n].copy()
    pos["counter"][3::16] = 48
    return pos


@pytest.mark.parametrize("policy", POLICIES)
@pytest.mark.parametrize("n,per", [(1, 1), (1, 3), (63, 1), (65, 7), (700, 4), (257, 16), (3000, 1)])
def test_uniform_counts(fresh, oracle, policy, n, per):
    pos = positions(oracle, n, 500 + n)
    announce(f"one wave per game: {n} x {per}, policy {policy}")
    res = fresh.run_playouts(pos, per_pos=per, seed=77, epoch=5, policy=policy)
    w, tr = oracle.run_playouts(pos, per_pos=per, seed=77, epoch=5, policy=policy)
    assert res.stats["grid_blocks"] == n * per and res.stats["block_size"] == 64
    assert np.array_equal(res.winners, w)
    assert res.stats["plies"] == int(tr["plies"].sum(dtype=np.uint64))
    assert res.stats["max_moves"] == int(tr["max_n"].max())


@pytest.mark.parametrize("policy", POLICIES)
@pytest.mark.parametrize("n", [1, 64, 65, 4097])
def test_uneven_keyed_graph_and_noalloc(fresh, oracle, policy, n):
    pos = positions(oracle, n, 900 + n)
    rng = np.random.default_rng(n)
    counts = rng.integers(0, 4, n).astype(np.uint32)
    counts[-1] = 2
    keys = rng.integers(0, 2**32, n, dtype=np.uint64).astype(np.uint32)
    announce(f"one wave per game: {n} positions uneven ({int(counts.sum())}), policy {policy}")
    w, _ = oracle.run_playouts(pos, counts=counts, seed=3, epoch=9, policy=policy, keys=keys)
    res = fresh.run_playouts(pos, counts=counts, seed=3, epoch=9, policy=policy, keys=keys)
    assert res.stats["grid_blocks"] == int(counts.sum())
    assert np.array_equal(res.winners, w)
    with fresh.graph(n, int(counts.sum()), policy) as g:
        for _ in range(2):
            got = g.run(pos, counts, seed=3, epoch=9, keys=keys)
            assert np.array_equal(got.winners, w) and got.stats["plies"] == res.stats["plies"]
    got, status = _noalloc(fresh, pos, 1, None, 3, 9, policy)
    w, _ = oracle.run_playouts(pos, per_pos=1, seed=3, epoch=9, policy=policy)
    assert status == 0 and np.array_equal(got, w)


@pytest.mark.parametrize("policy", POLICIES)
def test_route_ends_at_its_limit(fresh, oracle, policy):
    """The last size with one wave per game and the first with one lane per game: the same games."""
    limit = fresh.device_info()["compute_units"] * (48 if policy == POLICY_HEURISTIC_NOISY else 32)
    pos = positions(oracle, limit + 1, 41)
    announce(f"{limit} and {limit + 1} playouts, policy {policy}")
    a = fresh.run_playouts(pos[:limit], per_pos=1, seed=8, epoch=2, policy=policy)
    b = fresh.run_playouts(pos, per_pos=1, seed=8, epoch=2, policy=policy)
    assert a.stats["grid_blocks"] == limit and b.stats["grid_blocks"] < limit
    assert np.array_equal(a.winners, b.winners[:limit])
    fresh.stage(pos[:limit], per_pos=1)
    assert fresh.launch_staged(seed=8, epoch=2, policy=policy)["plies"] == a.stats["plies"]
    assert np.array_equal(fresh.fetch_winners(), a.winners)
