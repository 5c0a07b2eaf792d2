"""Ensemble stress and integrity scan, one wave per chain: against FP64 sums and counts over
the state read back, for lengths around the wave size and chain counts around the grid's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nk,beta", [(1, 2, 1.0), (3, 130, 0.05), (17, 64, 0.02), (4097, 20, 1.0), (8200, 33, 0.5)])
def test_stress_and_check_match_the_state(engine, n, nk, beta):
    ens = engine.add_ensemble(n, nk, beta, 1, seed=n)
    engine.init_equilibrium(ens)
    s = engine.state(ens)
    Z, N, Q, w = s["Z"], s["N"], s["Q"].copy(), s["w"].copy()
    assert all(v == 0 for v in engine.check(ens).values())
    q = Q.astype(np.float64)
    t3 = np.where(N > 0, 3.0 / np.maximum(N, 1), 0.0)
    want = [-(t3 * q[..., a] * q[..., b]).sum() for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2))]
    want += [np.sqrt((q ** 2).sum(-1)).sum(), Z.sum()]
    got, healthy = engine.stress(ens)
    assert healthy == n
    np.testing.assert_allclose(got, np.array(want) / n, rtol=1e-12, atol=1e-12 * np.abs(want).max() / n)
    # planted faults: an end strand with a vector, a non-finite CD rate, a late clock, stalls
    long = np.nonzero(Z > 2)[0]
    if long.size == 0:
        engine.remove_ensemble(ens)
        return
    i, j = int(long[0]), int(long[-1])
    Q[i, Z[i] - 1, 1] = 1.0
    w[j, Z[j] - 2] = np.inf
    t = np.full(n, 5.0)
    t[i] = 1.0
    stall = np.zeros(n, np.int32)
    stall[:: max(1, n // 3)] = 2
    engine.set_state(ens, Z, N, Q, w, t=t, stall=stall)
    c = engine.check(ens, t_min=2.0)
    assert (c["end_q"], c["nonfinite"], c["stalled"], c["behind"]) == (1, 1, int((stall != 0).sum()), 1)
    assert c["z_range"] == c["n_below_1"] == c["n_sum"] == 0
    assert engine.stress(ens)[1] == int((stall == 0).sum())
    engine.remove_ensemble(ens)
