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


@pytest.mark.parametrize("batch,n", [(64, 64), (64, 127), (256, 4096), (256, 4097), (1024, 5003),
                                     (4096, 12399)])
def test_epoch_order(engine, oracle, positions, batch, n):  # noqa: F811
    """An epoch's order drawn on the host (up to 4096 positions) and on the device: the epoch equals
    its steps taken one by one in the oracle's order, bit for bit."""
    pos = positions[:n]
    t = np.random.default_rng(n).uniform(-1, 1, n).astype(np.float32)
    with _net(engine, batch, seed=4) as a, _net(engine, batch, seed=4) as b:
        a.set_dataset(pos, t)
        for epoch in (0, 3):
            a.train_epoch(batch, 1e-3, shuffle_seed=21, epoch=epoch)
            order = M.epoch_order(n, 21, epoch, oracle.philox)
            for k in range(n // batch):
                idx = order[k * batch:(k + 1) * batch]
                b.train_step(pos[idx], t[idx], 1e-3)
            np.testing.assert_array_equal(a.get_params(), b.get_params())
