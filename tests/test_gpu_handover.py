"""Waves that hand their last games over to other waves of their workgroup, on the device against
the oracle: workgroups from the smallest that does it to the largest, batches from a game for the
whole workgroup to several for every lane, both refills, results and traces; and the shapes that
batches take by themselves, on both sides of each size where that shape changes."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from gpu_ai_amd.engine import (POLICY_HEURISTIC, POLICY_HEURISTIC_NOISY, POLICY_RANDOM,
                               REFILL_QUEUE, REFILL_STATIC, Engine)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("policy", [POLICY_RANDOM, POLICY_HEURISTIC, POLICY_HEURISTIC_NOISY])
@pytest.mark.parametrize("block,refill", [(320, REFILL_QUEUE), (512, REFILL_STATIC),
                                          (768, REFILL_QUEUE), (1024, REFILL_STATIC),
                                          (1024, REFILL_QUEUE)])
def test_handover(oracle, policy, block, refill):
    with Engine(0) as eng:
        eng.set_tuning(block_size=block, blocks_per_cu=1, refill=refill, defer_min=16)
        for n, per in ((1, 1), (1, 65), (33, 31), (500, 9), (700, 1001)):
            pos = oracle.start_positions(40 + n, n, 0, 80, False)
            print(f"[gpu] handover: block {block}, refill {refill}, policy {policy}, {n} x {per}",
                  file=sys.stderr, flush=True)
            few = n * per < 100_000
            w, tr = oracle.run_playouts(pos, per_pos=per, seed=9, epoch=4, policy=policy)
            run = eng.run_traced if few else eng.run_playouts
            res = run(pos, per_pos=per, seed=9, epoch=4, policy=policy)
            assert np.array_equal(res.winners, w)
            assert res.stats["plies"] == int(tr["plies"].sum(dtype=np.uint64))
            assert res.stats["block_size"] == block
            assert res.stats["max_moves"] == int(tr["max_n"].max())
            if few:
                assert np.array_equal(res.plies, tr["plies"])
                assert np.array_equal(res.hashes, tr["hash"])


def test_shapes_of_batches(oracle):
    pos = oracle.start_positions(3, 64, 30, 70, True)
    with Engine(0) as eng:
        lanes = 64 * eng.device_info()["compute_units"]
        for total, block in ((4 * lanes, 64), (4 * lanes + 1, 320), (12 * lanes, 768),
                             (12 * lanes + 1, 768), (32 * lanes - 64, 768), (32 * lanes, 1024)):
            counts = np.full(64, total // 64, np.uint32)
            counts[5] += total % 64
            print(f"[gpu] shape of {total} playouts", file=sys.stderr, flush=True)
            res = eng.run_playouts(pos, counts=counts, seed=2, epoch=1)
            assert res.stats["block_size"] == block, total
            w, _ = oracle.run_playouts(pos, counts=counts, seed=2, epoch=1, traces=False)
            assert np.array_equal(res.winners, w)
