"""Ensemble stress and integrity scan of more chains than waves: short ones four at a time,
beside waves that meet a longer one, and stalled ones among them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,lo,hi,beta", [(60000, 2, 24, 1.0), (33000, 8, 17, 0.02), (30001, 60, 70, 0.02),
                                          (20000, 10, 160, 0.5)])
def test_stress_and_check_of_many_chains(engine, n, lo, hi, beta):
    rng = np.random.default_rng(n)
    lens = rng.integers(lo, hi + 1, n).astype(np.int32)
    ens = engine.add_ensemble(n, int(lens.max()), beta, 1, seed=n, nk_per_chain=lens)
    engine.init_equilibrium(ens)
    s = engine.state(ens)
    Z, N, Q, w = s["Z"], s["N"], s["Q"].copy(), s["w"].copy()
    assert all(v == 0 for v in engine.check(ens).values())
    stall = (rng.random(n) < 0.1).astype(np.int32)
    long = np.nonzero(Z > 2)[0]
    bad_q, bad_w = rng.choice(long, 40, replace=False), rng.choice(long, 30, replace=False)
    Q[bad_q, Z[bad_q] - 1, 2] = 1.0
    w[bad_w, Z[bad_w] - 2] = np.inf
    t = rng.random(n)
    engine.set_state(ens, Z, N, Q, w, t=t, stall=stall)
    c = engine.check(ens, t_min=0.25)
    assert (c["end_q"], c["nonfinite"], c["stalled"], c["behind"]) == (40, 30, int(stall.sum()), int((t < 0.25).sum()))
    assert c["z_range"] == c["n_below_1"] == c["n_sum"] == 0
    q = Q.astype(np.float64) * (stall == 0)[:, None, None]
    t3 = np.where(N > 0, 3.0 / np.maximum(N, 1), 0.0)
    want = [-(t3 * q[..., a] * q[..., b]).sum() for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2))]
    want += [np.sqrt((q ** 2).sum(-1)).sum(), Z[stall == 0].sum()]
    got, healthy = engine.stress(ens)
    assert healthy == int((stall == 0).sum())
    np.testing.assert_allclose(got, np.array(want) / healthy, rtol=1e-12, atol=1e-12 * np.abs(want).max() / healthy)
    engine.remove_ensemble(ens)
