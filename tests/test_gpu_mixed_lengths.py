"""Passes of mixed lengths whose short chains run in the lane form: the split (by what a
chain may reach, not by its Z alone) loses and repeats none, and every chain makes the
oracle's jumps."""
import numpy as np
import pytest

from test_gpu_parity import GEX, assert_same_state

pytestmark = pytest.mark.gpu

CASES = [
    dict(n=1500, lo=10, hi=420),            # more than a block of the split, every bin to 512 positions
    dict(n=1025, lo=180, hi=240),           # around the lane form's 128 positions: some outgrow it
    dict(n=70, lo=400, hi=500, T=1.0),      # none for the lanes
    dict(n=400, lo=10, hi=300, partner="melt"),
    dict(n=300, lo=30, hi=400, beta=3.0, cd=0),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "_".join("%s%s" % kv for kv in c.items()))
def test_mixed_lengths_match_oracle(oracle, case):
    import gpu_dsm_amd as g
    n, beta, cd, partner = case["n"], case.get("beta", 1.0), case.get("cd", 1), case.get("partner")
    lens = np.random.default_rng(8).integers(case["lo"], case["hi"] + 1, n).astype(np.int32)
    nk = int(lens.max())
    P = oracle.Params(beta, nk, cd, nmax=nk, partner=partner, gex=GEX, nk_chains=lens)
    O = oracle.Ensemble(P, seed=17, n=n, salt=1, nk_per_chain=lens)
    with g.Engine(0) as e:
        e.set_option("lane", 2)
        e.set_option("concurrent", 1)
        ens = e.add_ensemble(n, nk, beta, cd, seed=17, salt=1, nk_per_chain=lens, partner=partner, gex=GEX)
        e.init_equilibrium(ens)
        T = case.get("T", 2.0)
        for t in (0.5 * T, T):
            st = e.advance(ens, t)
            assert st["events"] == O.advance(t_end=t)[0]
            assert_same_state(e.state(ens), O.state(), "t = %g" % t)
