"""Equilibrium draw by 16-lane rows and flow rows summed in parts, at the sizes where their
splits end: lengths around 64 boundaries and 16 strands, chain counts around the rows of a
block and the parts of a reduction, next to an ensemble whose staging rows have an odd size."""
import numpy as np
import pytest

from test_gpu_parity import GEX, assert_same_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nk,beta,partner", [(1, 2, 1.0, None), (15, 3, 0.1, None), (17, 64, 0.02, None),
                                               (33, 65, 1.0, None), (16, 66, 30.0, None), (5, 2047, 0.01, None),
                                               (250, 129, 0.5, "gex")])
def test_equilibrium_draw_matches_oracle(oracle, engine, n, nk, beta, partner):
    P = oracle.Params(beta, nk, 1, nmax=nk, partner=partner, gex=GEX)
    ens = engine.add_ensemble(n, nk, beta, 1, seed=31, salt=6, partner=partner, gex=GEX, sample="msd")
    engine.init_equilibrium(ens)
    engine.advance_events(ens, 3)
    engine.init_equilibrium(ens)  # a second draw starts over
    g = engine.state(ens)
    assert_same_state(g, oracle.Ensemble(P, seed=31, n=n, salt=6).state(), "initial")
    assert not g["R1"].any() and not g["stall"].any() and not g["dt_prev"].any()
    engine.remove_ensemble(ens)


@pytest.mark.parametrize("n", [1, 255, 1023, 1025, 3000])
def test_flow_rows_match_the_samples(engine, n):
    odd = engine.add_ensemble(3, 10, 1.0, 0, seed=1, sample="gt", delta=1.0, window=5)
    ens = engine.add_ensemble(n, 14, 1.0, 1, kappa=[0, 0.1, 0, 0, 0, 0, 0, 0, 0], seed=3, sample="flow", delta=0.5,
                              window=9)
    engine.init_equilibrium(ens)
    engine.advance(ens, 4.0)
    k0, s = engine.last_samples(ens)
    assert s.shape == (8, n, 8) and k0 == 1
    rows = engine.flow_stress(ens)
    want = s.astype(np.float64)
    np.testing.assert_allclose(rows[:, :8], want.sum(axis=1), rtol=1e-13, atol=1e-13 * np.abs(want).sum(axis=1).max())
    assert np.array_equal(rows[:, 8], np.full(8, n))
    engine.remove_ensemble(ens)
    engine.remove_ensemble(odd)
