"""The solo form (one chain per wave, out of LDS) repeats the oracle's jumps bit for bit, and
the wave forms' samples.

Chains of one strand, of a whole block and group of positions and one more, of several
groups; chains that outgrow a launch's capacity; the free-slot list at full length (Z = Nk);
strands beyond the short-strand tables; partner backgrounds, exponential waiting times,
fixed jump counts, and chains that stall.
"""
import numpy as np
import pytest

from test_gpu_parity import GEX, _bits, assert_same_state

pytestmark = pytest.mark.gpu

CASES = [
    dict(n=1, nk=30),
    dict(n=70, nk=2, cd=0, T=40.0),
    dict(n=64, nk=3, T=40.0),
    dict(n=300, nk=25, cd=0),
    dict(n=100, nk=127),                            # Z ~ 64
    dict(n=60, nk=255, T=2.0),                      # one group
    dict(n=40, nk=256, beta=0.02, T=0.5),           # Z ~ Nk: the whole of a group and one more
    dict(n=40, nk=510, T=1.5),                      # Z ~ 256: over and back
    dict(n=12, nk=1100, T=0.5),                     # three groups
    dict(n=6, nk=2047, beta=0.1, T=0.1),            # eight
    dict(n=60, nk=400, beta=20.0, T=3.0),           # strands of 20 Kuhn steps and more
    dict(n=120, nk=40, beta=2.0, exp_wait=True),
    dict(n=120, nk=60, partner="gex"),
    dict(n=120, nk=300, partner="melt", T=1.5),
]


def _engine(solo, concurrent=-1):
    import gpu_dsm_amd as g
    e = g.Engine(0)
    e.set_option("solo", solo)
    e.set_option("lane", 0)
    e.set_option("concurrent", concurrent)
    return e


@pytest.mark.parametrize("case", CASES, ids=lambda c: "_".join("%s%s" % kv for kv in c.items()))
def test_solo_form_matches_oracle(oracle, case):
    n, nk, beta, cd = case["n"], case["nk"], case.get("beta", 1.0), case.get("cd", 1)
    partner, ew = case.get("partner"), case.get("exp_wait", False)
    lens = np.random.default_rng(2).integers(10, nk + 1, n).astype(np.int32) if partner == "melt" else None
    if lens is not None:
        lens[0] = nk
    P = oracle.Params(beta, nk, cd, exp_wait=ew, nmax=nk, partner=partner, gex=GEX, nk_chains=lens)
    O = oracle.Ensemble(P, seed=31, n=n, salt=2, nk_per_chain=lens)
    with _engine(1) as e:
        ens = e.add_ensemble(n, nk, beta, cd, seed=31, salt=2, exp_wait=ew, nk_per_chain=lens, partner=partner, gex=GEX)
        e.init_equilibrium(ens)
        T = case.get("T", 6.0)
        for t in (0.5 * T, T):
            st = e.advance(ens, t)
            ev, _ = O.advance(t_end=t)
            assert st["events"] == ev
            assert_same_state(e.state(ens), O.state(), "t = %g" % t)
        st = e.advance_events(ens, 70)  # more than the random words of one refill
        assert st["events"] == O.advance(max_events=70)[0] == 70 * n
        assert_same_state(e.state(ens), O.state(), "70 jumps")


@pytest.mark.parametrize("concurrent", [0, 1])
@pytest.mark.parametrize("sample", ["gt", "msd"])
@pytest.mark.parametrize("n,nk,partner", [(130, 25, None), (150, 260, "gex"), (40, 700, None)])
def test_solo_form_samples(sample, n, nk, partner, concurrent):
    out = []
    for solo in (0, 1):
        with _engine(solo, concurrent) as e:
            ens = e.add_ensemble(n, nk, 1.0, 1, seed=5, sample=sample, delta=0.25, corr_p=16, corr_m=2, corr_levels=3,
                                 window=7, partner=partner, gex=GEX)
            e.init_equilibrium(ens)
            st = e.advance(ens, 3.0)
            s = e.state(ens)
            s["events"], s["zs"] = st["events"], st["z_sum"]
            s["k0"], s["rows"] = e.last_samples(ens)
            s["lag"], s["G"] = e.correlator(ens)
            out.append(s)
    a, b = out
    assert_same_state(b, a, sample)
    assert (a["events"], a["zs"], a["k0"]) == (b["events"], b["zs"], b["k0"])
    assert np.array_equal(_bits(a["rows"]), _bits(b["rows"])) and np.array_equal(a["G"], b["G"])
    assert np.array_equal(a["dt_prev"], b["dt_prev"]) and np.array_equal(a["next_sample"], b["next_sample"])
    if sample == "msd":
        assert np.array_equal(_bits(a["R1"]), _bits(b["R1"]))


def test_solo_form_outgrown_and_stalled_chains():
    """Chains of one Kuhn step per strand (Z = Nk = 300, no slot free) and of 253 .. 257
    strands, around the first launch's 256 positions; a chain with a NaN vector stops at its
    first jump, one with an infinite one as in the wave forms."""
    n, nk = 60, 300
    rng = np.random.default_rng(1)
    Z = np.where(np.arange(n) % 2, nk, 253 + np.arange(n) % 5).astype(np.int32)
    N = np.zeros((n, nk), np.int32)
    Q = np.zeros((n, nk, 3), np.float32)
    w = np.zeros((n, nk), np.float32)
    for i in range(n):
        z = Z[i]
        N[i, :z] = 1
        N[i, z // 2] += nk - z
        Q[i, 1:z - 1] = rng.standard_normal((z - 2, 3))
        w[i, :z - 1] = 0.01
    mid = Z // 2
    Q[4, mid[4], 2] = np.nan
    Q[6, mid[6], 1] = np.inf
    out = []
    for solo in (0, 1):
        with _engine(solo) as e:
            ens = e.add_ensemble(n, nk, 1.0, 1, seed=9)
            e.set_state(ens, Z, N, Q, w)
            st = e.advance(ens, 2.0)
            out.append(dict(e.state(ens), events=st["events"], check=e.check(ens)))
    a, b = out
    assert a["events"] == b["events"] and a["check"] == b["check"]
    assert np.array_equal(a["stall"], b["stall"]) and a["stall"][4] == 2
    keep = a["stall"] == 0
    assert_same_state({k: b[k][keep] for k in ("Z", "N", "Q", "w", "t", "ev")},
                      {k: a[k][keep] for k in ("Z", "N", "Q", "w", "t", "ev")}, "outgrown")
