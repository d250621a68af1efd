"""A device allocation that is refused fails its own call and none after it."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_ai_amd.engine import Engine, MiError

pytestmark = pytest.mark.gpu


def test_the_call_after_a_refused_allocation(oracle):
    pos = oracle.start_positions(12, 64, 0, 30, False)
    with Engine(0) as eng:
        print("[gpu] a copy between buffers of 16 TiB, then 64 x 300 playouts", flush=True)
        with pytest.raises(MiError) as e:
            eng.copy_calibration(1 << 44)
        assert "out of memory" in str(e.value)
        got = eng.start_positions(12, 64, 0, 30)
        assert got.tobytes() == pos.tobytes()
        with pytest.raises(MiError):
            eng.copy_calibration(1 << 44)
        w, _ = oracle.run_playouts(pos, per_pos=300, seed=2, epoch=1, traces=False)
        assert np.array_equal(eng.run_playouts(pos, per_pos=300, seed=2, epoch=1).winners, w)
