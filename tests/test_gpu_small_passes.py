"""Passes whose bookkeeping one block does, and the first that need more: every chain of the
list runs, once, and the totals are the chains' own."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flow", [False, True])
@pytest.mark.parametrize("sizes", [(1,), (1023,), (1025,), (8192,), (8193,), (5, 1024, 3)], ids=str)
def test_small_passes(oracle, sizes, flow):
    import gpu_dsm_amd as g
    kappa = [0, 1e-2, 0, 0, 0, 0, 0, 0, 0] if flow else [0.0] * 9
    with g.Engine(0) as e:
        ids, ref = [], []
        for q, n in enumerate(sizes):
            P = oracle.Params(1.0, 6, 1, kappa=np.array(kappa), nmax=6)
            ref.append(oracle.Ensemble(P, seed=2, n=n, salt=q))
            ids.append(e.add_ensemble(n, 6, 1.0, 1, kappa=kappa, seed=2, salt=q))
            e.init_equilibrium(ids[-1])
        for t in (1.0, 2.5):
            st = e.advance_many(ids, t)
            assert st["events"] == sum(O.advance(t_end=t)[0] for O in ref)
            for i, O in zip(ids, ref):
                assert_same_state(e.state(i), O.state(), "t = %g" % t)
