"""Chains that outgrow their lane finish in another form also where no chain can exceed the
row form's 64 positions (Nk = 50: columns of 48)."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_state

pytestmark = pytest.mark.gpu


def test_chains_beyond_low_columns_finish():
    import gpu_dsm_amd as g
    n, nk = 300, 50
    Z = np.array([nk, 49, 48, 47, 46, 20])[np.arange(n) % 6].astype(np.int32)
    N = np.zeros((n, nk), np.int32)
    Q = np.zeros((n, nk, 3), np.float32)
    w = np.zeros((n, nk), np.float32)
    rng = np.random.default_rng(4)
    for i, z in enumerate(Z):
        N[i, :z] = 1
        N[i, z // 2] += nk - z
        Q[i, 1:z - 1] = rng.standard_normal((z - 2, 3))
        w[i, :z - 1] = 0.01
    out = []
    for lane in (0, 2):
        with g.Engine(0) as e:
            e.set_option("small_per_cu", 0)
            e.set_option("lane", lane)
            ens = e.add_ensemble(n, nk, 1.0, 1, seed=12)
            e.set_state(ens, Z, N, Q, w)
            st = e.advance(ens, 4.0)
            out.append(dict(e.state(ens), events=st["events"]))
    a, b = out
    assert a["events"] == b["events"]
    assert_same_state(b, a, "outgrown")
    assert b["t"].min() >= 4.0
