"""Gradients of the value network at the edges of the update kernel's rounds (32 splits of 128 rows):
less than a split, a half-filled last split, a full round, one split past it, two rounds and a bit.
Oracle and tolerances as in test_gpu_mlp.py."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import mlp_ref as M
from test_gpu_mlp import TENSORS, _net, _params, positions  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [33, 65, 129, 4097, 4160, 8300])
def test_gradients_at_round_edges(engine, positions, n):  # noqa: F811
    w = _params(16)
    pos = positions[:n]
    t = np.random.default_rng(n).uniform(-1, 1, n).astype(np.float32)
    with _net(engine, 9000) as net:
        net.set_params(w)
        g, loss = net.gradients(pos, t)
    ref, ref_loss = M.gradients(w, M.encode(pos), t)
    assert abs(loss - ref_loss) <= 1e-4 * ref_loss
    for name, (lo, hi) in TENSORS.items():
        a, b = g[lo:hi].astype(np.float64), ref[lo:hi]
        err = np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)
        cos = np.dot(a, b) / (np.linalg.norm(a) * np.linalg.norm(b))
        assert err <= 2e-3 and cos >= 0.99999, (name, err, cos)
