"""mi_run_playouts_noalloc against the oracle on a context without a shape of its own, around the sizes
where the launch changes (a wave per game, one workgroup per CU of 5 to 16 waves, the longest-first
order), on a tuned one, and replayed from a captured graph."""
from __future__ import annotations

import ctypes
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
    with Engine(0) as eng:
        yield eng


@pytest.mark.parametrize("policy", POLICIES)
def test_uniform_sizes(fresh, oracle, policy):
    cus = fresh.device_info()["compute_units"]
    # positions, playouts per CU: the last wave per game, lanes, 5, 8 and 12 waves (ordered), 16
    for n, per_cu in ((512, 32), (512, 50), (1024, 258), (512, 512), (768, 1023), (1024, 2052)):
        per = per_cu * cus // n
        pos = oracle.start_positions(60 + n, n, 10, 60, False)
        announce(f"noalloc {n} x {per}, policy {policy}")
        got, status = _noalloc(fresh, pos, per, None, 14, 6, policy)
        w, _ = oracle.run_playouts(pos, per_pos=per, seed=14, epoch=6, policy=policy, traces=False)
        assert status == 0 and np.array_equal(got, w), (n, per)


@pytest.mark.parametrize("policy", POLICIES)
def test_counted_and_ordered(fresh, oracle, policy):
    pos = oracle.start_positions(9, 1500, 0, 80, True)
    counts = np.random.default_rng(policy).integers(0, 180, 1500).astype(np.uint32)
    announce(f"counted noalloc of {int(counts.sum())} games, policy {policy}")
    got, status = _noalloc(fresh, pos, 0, counts, 15, 7, policy)
    w, _ = oracle.run_playouts(pos, counts=counts, seed=15, epoch=7, policy=policy, traces=False)
    assert status == 0 and np.array_equal(got, w)


def test_on_a_tuned_context(oracle):
    pos = oracle.start_positions(10, 512, 0, 60, False)
    counts = np.random.default_rng(1).integers(0, 300, 512).astype(np.uint32)
    with Engine(0) as eng:
        announce("mi_autotune_sizes 1024, 65536, then mi_autotune on 512 x 256")
        eng.autotune_sizes(pos, [1024, 65536], reps=1)
        eng.autotune(pos, per_pos=256, reps=1)
        for per in (2, 128, 256, 700):
            announce(f"noalloc 512 x {per} on a tuned context")
            got, status = _noalloc(eng, pos, per, None, 16, 8, POLICY_RANDOM)
            w, _ = oracle.run_playouts(pos, per_pos=per, seed=16, epoch=8, traces=False)
            assert status == 0 and np.array_equal(got, w), per
        got, status = _noalloc(eng, pos, 0, counts, 16, 8, POLICY_RANDOM)
        w, _ = oracle.run_playouts(pos, counts=counts, seed=16, epoch=8, traces=False)
        assert status == 0 and np.array_equal(got, w)


@pytest.mark.parametrize("policy", POLICIES)
@pytest.mark.parametrize("n,per", [(64, 16), (128, 1100), (90, 0)])
def test_captured(fresh, oracle, policy, n, per):
    """One wave per game, workgroups of nine waves, and counts on the device: replays on other
    positions each time, with eager calls between them."""
    from devmem import DeviceArray, Stream, hip
    lib = hip()
    counts = np.arange(n, dtype=np.uint32) if per == 0 else None
    total = int(counts.sum()) if per == 0 else n * per
    sets = [oracle.start_positions(70 + i, n, 0, 70, False) for i in range(3)]
    d_win = DeviceArray(np.full(total, 7, dtype=np.int8))
    d_pos = DeviceArray(sets[0])
    d_counts = None if counts is None else DeviceArray(counts)
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()
    try:
        with Stream() as s:
            announce(f"noalloc {n} x {per} captured, policy {policy}")
            assert lib.hipStreamBeginCapture(s.handle, 1) == 0
            fresh.run_playouts_noalloc(d_pos.address, n, d_counts.address if d_counts else None, per,
                                       d_win.address, seed=17, epoch=9, policy=policy,
                                       stream=s.handle.value)
            assert lib.hipStreamEndCapture(s.handle, ctypes.byref(graph)) == 0
            assert lib.hipGraphInstantiate(ctypes.byref(run), graph, None, None,
                                           ctypes.c_size_t(0)) == 0
            for i, pos in enumerate(sets):
                d_pos.upload(pos)
                announce(f"replay {i}")
                assert lib.hipGraphLaunch(run, s.handle) == 0
                s.synchronize()
                w, _ = oracle.run_playouts(pos, per_pos=per or None, counts=counts, seed=17, epoch=9,
                                           policy=policy, traces=False)
                assert np.array_equal(d_win.download(np.int8, total), w), i
                eager = fresh.run_playouts(pos[:33], per_pos=40, seed=i, epoch=1, policy=policy)
                assert len(eager.winners) == 33 * 40
    finally:
        if run:
            lib.hipGraphExecDestroy(run)
        if graph:
            lib.hipGraphDestroy(graph)
        for b in (d_win, d_pos, d_counts):
            if b is not None:
                b.free()
