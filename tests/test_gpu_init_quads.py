"""Equilibrium draw by quads of lanes (ensembles of short chains): lengths around 16
boundaries and four strands, chain counts around a block's 64, a long chain among short
ones, and both sides of the rule."""
import numpy as np
import pytest

from test_gpu_parity import GEX, assert_same_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nk,beta,partner", [(1, 2, 1.0, None), (63, 4, 0.1, None), (64, 5, 0.02, None),
                                               (65, 16, 1.0, None), (129, 17, 1.0, None), (500, 19, 1.0, "gex"),
                                               (70, 100, 30.0, None), (300, 20, 1.0, None)])
def test_draw_matches_oracle(oracle, engine, n, nk, beta, partner):
    P = oracle.Params(beta, nk, 1, nmax=nk, partner=partner, gex=GEX)
    ens = engine.add_ensemble(n, nk, beta, 1, seed=7, salt=2, partner=partner, gex=GEX)
    engine.init_equilibrium(ens)
    assert_same_state(engine.state(ens), oracle.Ensemble(P, seed=7, n=n, salt=2).state(), "initial")
    engine.remove_ensemble(ens)


def test_draw_of_a_long_chain_among_short_ones(oracle, engine):
    lens = np.full(300, 6, np.int32)
    lens[[0, 130, 299]] = (700, 33, 65)
    P = oracle.Params(1.0, 700, 1, nmax=700, partner="melt", nk_chains=lens)
    ens = engine.add_ensemble(lens.size, 700, 1.0, 1, seed=9, nk_per_chain=lens, partner="melt")
    engine.init_equilibrium(ens)
    assert_same_state(engine.state(ens), oracle.Ensemble(P, seed=9, n=lens.size, nk_per_chain=lens).state(), "initial")
    engine.remove_ensemble(ens)
