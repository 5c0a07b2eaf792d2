"""The lane form (one chain per lane) repeats the oracle's jumps bit for bit, and the other
forms' samples.

Chain counts around the wave size and lengths at the ends of its range (Nk = 2, Z = 1; the
size steps of 4 quads; chains that start beyond its capacity or outgrow it), long strands
(beyond its short-strand tables), partner backgrounds, exponential waiting times, fixed jump
counts, and chains that stall.
"""
import numpy as np
import pytest

from test_gpu_parity import GEX, _bits, assert_same_state

pytestmark = pytest.mark.gpu

CASES = [
    dict(n=1, nk=30),
    dict(n=63, nk=2, cd=0, T=40.0),
    dict(n=64, nk=3, T=40.0),
    dict(n=700, nk=16, beta=0.5),
    dict(n=2065, nk=50, cd=0),
    dict(n=600, nk=100),                       # Z ~ 50, capacity 76
    dict(n=300, nk=100, beta=0.5),             # Z ~ 67, two blocks
    dict(n=200, nk=200, T=3.0),                # Z ~ 100
    dict(n=200, nk=220, T=2.0),
    dict(n=150, nk=400, beta=20.0),            # strands of 20 Kuhn steps and more
    dict(n=300, nk=40, beta=2.0, exp_wait=True),
    dict(n=300, nk=60, partner="gex"),
    dict(n=300, nk=60, partner="melt"),
]


def _engine(lane):
    import gpu_dsm_amd as g
    e = g.Engine(0)
    e.set_option("small_per_cu", 0)
    e.set_option("lane", lane)
    return e


@pytest.mark.parametrize("case", CASES, ids=lambda c: "_".join("%s%s" % kv for kv in c.items()))
def test_lane_form_matches_oracle(oracle, case):
    n, nk, beta, cd = case["n"], case["nk"], case.get("beta", 1.0), case.get("cd", 1)
    partner, ew = case.get("partner"), case.get("exp_wait", False)
    lens = np.random.default_rng(2).integers(10, nk + 1, n).astype(np.int32) if partner == "melt" else None
    if lens is not None:
        lens[0] = nk
    P = oracle.Params(beta, nk, cd, exp_wait=ew, nmax=nk, partner=partner, gex=GEX, nk_chains=lens)
    O = oracle.Ensemble(P, seed=21, n=n, salt=4, nk_per_chain=lens)
    with _engine(2) as e:
        ens = e.add_ensemble(n, nk, beta, cd, seed=21, salt=4, exp_wait=ew, nk_per_chain=lens, partner=partner, gex=GEX)
        e.init_equilibrium(ens)
        T = case.get("T", 6.0)
        for t in (0.5 * T, T):
            st = e.advance(ens, t)
            ev, _ = O.advance(t_end=t)
            assert st["events"] == ev
            assert_same_state(e.state(ens), O.state(), "t = %g" % t)
        st = e.advance_events(ens, 37)
        assert st["events"] == O.advance(max_events=37)[0] == 37 * n
        assert_same_state(e.state(ens), O.state(), "37 jumps")


@pytest.mark.parametrize("sample", ["gt", "msd"])
@pytest.mark.parametrize("n,nk,partner", [(130, 25, None), (2100, 60, "gex"), (300, 160, None)])
def test_lane_form_samples(sample, n, nk, partner):
    out = []
    for lane in (0, 2):
        with _engine(lane) as e:
            ens = e.add_ensemble(n, nk, 1.0, 1, seed=5, sample=sample, delta=0.5, corr_p=16, corr_m=2, corr_levels=3,
                                 window=7, partner=partner, gex=GEX)
            e.init_equilibrium(ens)
            st = e.advance(ens, 8.0)
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


def test_lane_form_outgrown_and_stalled_chains(oracle):
    """Chains set to one Kuhn step per strand (Z = Nk, beyond the form's capacity of 76
    positions) and to 73..75 strands, which soon outgrow it; chains with a NaN vector stop
    at their first jump."""
    n, nk = 200, 100
    P = oracle.Params(1.0, nk, 1)
    O = oracle.Ensemble(P, seed=9, n=n)
    o = O.state()
    Z, N, Q, w = (np.array(o[k]) for k in ("Z", "N", "Q", "w"))
    rng = np.random.default_rng(1)
    for i in range(0, n, 3):
        z = nk if i % 2 else 73 + i % 3
        Z[i] = z
        N[i], Q[i], w[i] = 0, 0.0, 0.0
        N[i, :z] = 1
        N[i, z // 2] += nk - z
        Q[i, 1:z - 1] = rng.standard_normal((z - 2, 3)).astype(np.float32)
        w[i, :z - 1] = 0.01
    # a strand of one Kuhn step between such strands has no shift rate, so no NaN one
    bad = int(np.nonzero((np.arange(n) % 3 != 0) & (Z > 3) & (N[:, 1] > 1))[0][0])
    Q[bad, 1, 2] = np.nan
    out = []
    for lane in (0, 2):
        with _engine(lane) as e:
            ens = e.add_ensemble(n, nk, 1.0, 1, seed=9)
            e.set_state(ens, Z, N[:, :nk], Q[:, :nk], w[:, :nk])
            st = e.advance(ens, 3.0)
            out.append(dict(e.state(ens), events=st["events"], check=e.check(ens)))
    a, b = out
    assert a["events"] == b["events"] and a["stall"][bad] == b["stall"][bad] == 2
    assert np.array_equal(a["stall"], b["stall"]) and a["check"] == b["check"]
    keep = np.arange(n) != bad
    assert_same_state({k: b[k][keep] for k in ("Z", "N", "Q", "w", "t", "ev")},
                      {k: a[k][keep] for k in ("Z", "N", "Q", "w", "t", "ev")}, "outgrown")
