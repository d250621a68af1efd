"""Start positions on the device against the oracle, over the sizes at which the waves' slots, the
attempts played ahead and the claims change (k_start_positions)."""
from __future__ import annotations

import sys

import pytest

pytestmark = pytest.mark.gpu


# (n, kmin, kmax): one position a wave with 64 attempts ahead, several, all lanes with a position of
# their own; lengths at which hardly any attempt is accepted (windows of 64 attempts and more)
@pytest.mark.parametrize("reject", [False, True])
@pytest.mark.parametrize("n,kmin,kmax", [(1, 0, 150), (17, 0, 0), (40, 150, 170), (3071, 0, 90),
                                         (3073, 30, 150), (9000, 100, 140), (65535, 0, 150),
                                         (65536, 0, 30), (200001, 0, 120)])
def test_start_positions_match_oracle(engine, oracle, n, kmin, kmax, reject):
    print(f"[gpu] {n} start positions, k in [{kmin}, {kmax}], reject {reject}", file=sys.stderr,
          flush=True)
    got = engine.start_positions(11 + n, n, kmin, kmax, reject_terminal=reject)
    want = oracle.start_positions(11 + n, n, kmin, kmax, reject_terminal=reject)
    assert got.tobytes() == want.tobytes()


# around one and two waves a SIMD (1024 and 2048), and around 64 positions for each of their waves:
# dealt out to the slots up to 131,072 positions, claimed from a queue beyond
@pytest.mark.parametrize("n", [1023, 1025, 65537, 131071, 131072, 131073])
def test_start_positions_dealt_and_claimed(engine, oracle, n):
    print(f"[gpu] {n} start positions", file=sys.stderr, flush=True)
    got = engine.start_positions(n, n, 0, 60, reject_terminal=True)
    want = oracle.start_positions(n, n, 0, 60, reject_terminal=True)
    assert got.tobytes() == want.tobytes()
