"""The multi-tau update takes a window's samples level by level with the lags side by side:
G(t) and MSD(t) against the sample-by-sample oracle correlator over windows that are not
multiples of the chunk or block size, few and many chains, lag counts below and above the
lag threads, and a lag count too large for the kernel's LDS."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (n, p, m, window, T, sample): 64 rows is the kernel's chunk, 16 / 4 its chains a block
CASES = [(5, 16, 2, 64, 130, "gt"), (4097, 16, 2, 100, 130, "gt"), (37, 64, 8, 130, 300, "gt"),
         (4111, 64, 8, 33, 90, "msd"), (9, 2, 2, 7, 40, "gt"), (50, 6, 3, 129, 140, "msd"),
         (33, 200, 2, 70, 140, "gt"), (3, 2000, 2, 40, 80, "gt")]


@pytest.mark.parametrize("n,p,m,window,T,sample", CASES)
def test_window_update_matches_sample_by_sample(oracle, engine, n, p, m, window, T, sample):
    s = 3
    ens = engine.add_ensemble(n, 12, 1.0, 1, seed=8, sample=sample, delta=1.0, corr_p=p, corr_m=m, corr_levels=s,
                              window=window)
    engine.init_equilibrium(ens)
    corr = oracle.Correlator(p, m, s, n, type=1 if sample == "msd" else 0)
    t = 0
    while t < T:
        t = min(T, t + window)
        engine.advance(ens, float(t))
        for row in engine.last_samples(ens)[1]:
            corr.add_row(row)
        if t == window or t == T:
            lag_o, g_o = corr.result()
            lag, g = engine.correlator(ens)
            assert np.array_equal(lag, lag_o)
            # FP64 sums over the chains in another order: n * 2^-53 of the largest term
            np.testing.assert_allclose(g, g_o, rtol=1e-11, atol=1e-12 * np.abs(g_o).max())
    engine.remove_ensemble(ens)
