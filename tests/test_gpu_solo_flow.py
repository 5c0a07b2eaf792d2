"""The solo form for passes with flow repeats the oracle's jumps bit for bit, and the wave
forms' samples: one strand to two groups of 256 positions and over, every component of
kappa, strong flow (stalls), still ensembles in the same pass (alone and beside, in the
sequential and the concurrent order), partner backgrounds, exponential waiting times, fixed
jump counts."""
import numpy as np
import pytest

from test_gpu_parity import GEX, _bits, assert_same_state

pytestmark = pytest.mark.gpu

SHEAR = np.array([0, 1, 0, 0, 0, 0, 0, 0, 0.0])
FULL = np.array([0.3, 1.0, -0.2, 0.1, -0.5, 0.7, 0.4, -0.9, 0.2])

CASES = [
    dict(n=1, nk=30),
    dict(n=70, nk=2, cd=0, T=30.0),
    dict(n=64, nk=3, T=30.0),
    dict(n=200, nk=60, kappa=1e-2 * FULL),
    dict(n=50, nk=255, T=2.0),                       # one group
    dict(n=30, nk=256, beta=0.02, T=0.5),            # Z ~ Nk: a group and one more
    dict(n=30, nk=510, kappa=1e-3 * FULL, T=1.5),    # Z ~ 256: over and back
    dict(n=8, nk=1040, T=0.5),                       # beyond two groups
    dict(n=60, nk=400, beta=20.0, kappa=0.05 * FULL, T=3.0),
    dict(n=100, nk=40, beta=2.0, exp_wait=True),
    dict(n=100, nk=90, partner="gex"),
]


def _engine(solo, concurrent=-1):
    import gpu_dsm_amd as g
    e = g.Engine(0)
    e.set_option("solo", solo)
    e.set_option("lane", 0)
    e.set_option("concurrent", concurrent)
    return e


@pytest.mark.parametrize("case", CASES, ids=lambda c: "_".join("%s%s" % (k, v) for k, v in c.items() if k != "kappa"))
def test_solo_flow_matches_oracle(oracle, case):
    n, nk, beta, cd = case["n"], case["nk"], case.get("beta", 1.0), case.get("cd", 1)
    partner, ew, kappa = case.get("partner"), case.get("exp_wait", False), case.get("kappa", 1e-2 * SHEAR)
    P = oracle.Params(beta, nk, cd, kappa=kappa, exp_wait=ew, nmax=nk, partner=partner, gex=GEX)
    O = oracle.Ensemble(P, seed=51, n=n, salt=3)
    with _engine(1) as e:
        ens = e.add_ensemble(n, nk, beta, cd, kappa=list(kappa), seed=51, salt=3, exp_wait=ew, partner=partner, gex=GEX)
        e.init_equilibrium(ens)
        T = case.get("T", 6.0)
        for t in (0.5 * T, T):
            st = e.advance(ens, t)
            assert st["events"] == O.advance(t_end=t)[0]
            assert_same_state(e.state(ens), O.state(), "t = %g" % t)
        st = e.advance_events(ens, 70)
        assert st["events"] == O.advance(max_events=70)[0] == 70 * n
        assert_same_state(e.state(ens), O.state(), "70 jumps")


@pytest.mark.parametrize("concurrent", [0, 1])
@pytest.mark.parametrize("rate", [1e-3, 1.0])
def test_mixed_passes(rate, concurrent):
    """Ensembles of every bin to 512 positions, every other one still, G(t) and flow samples."""
    sizes = [(300, 60), (260, 160), (200, 330), (150, 500), (90, 700)]
    out = []
    for solo in (0, 1):
        with _engine(solo, concurrent) as e:
            ids = []
            for q, (n, nk) in enumerate(sizes):
                still = q % 2
                ids.append(e.add_ensemble(n, nk, 1.0, 1, kappa=[0.0] * 9 if still else list(rate * FULL), seed=6,
                                          salt=q, sample="gt" if still else "flow", delta=0.25, corr_levels=3, window=4))
            for i in ids:
                e.init_equilibrium(i)
            for T in (1.0, 2.0):
                st = e.advance_many(ids, T)
                for i in ids:
                    s = e.state(i)
                    s["events"], s["zs"] = st["events"], st["z_sum"]
                    s["k0"], s["rows"] = e.last_samples(i)
                    out.append(s)
    half = len(out) // 2
    for a, b in zip(out[:half], out[half:]):
        assert np.array_equal(a["stall"], b["stall"])
        keep = a["stall"] == 0
        assert_same_state({k: b[k][keep] for k in ("Z", "N", "Q", "w", "t", "ev")},
                          {k: a[k][keep] for k in ("Z", "N", "Q", "w", "t", "ev")}, "mixed")
        assert (a["events"], a["zs"], a["k0"]) == (b["events"], b["zs"], b["k0"])
        assert np.array_equal(_bits(a["rows"]), _bits(b["rows"]))
        assert np.array_equal(a["dt_prev"], b["dt_prev"]) and np.array_equal(a["next_sample"], b["next_sample"])
