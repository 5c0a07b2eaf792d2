"""The lane form under flow repeats the oracle's jumps bit for bit, and the other forms'
samples: chains of one strand and of whole quads, below and beyond the columns' heights,
that outgrow them, of several ensembles, every component of kappa, strong flow (stalls),
partner backgrounds, exponential waiting times, fixed jump counts."""
import numpy as np
import pytest

from test_gpu_parity import GEX, _bits, assert_same_state

pytestmark = pytest.mark.gpu

SHEAR = np.array([0, 1, 0, 0, 0, 0, 0, 0, 0.0])
UNIAXIAL = np.array([1, 0, 0, 0, -0.5, 0, 0, 0, -0.5])
FULL = np.array([0.3, 1.0, -0.2, 0.1, -0.5, 0.7, 0.4, -0.9, 0.2])

CASES = [
    dict(n=1, nk=14),
    dict(n=70, nk=2, cd=0, T=30.0),
    dict(n=64, nk=3, T=30.0),
    dict(n=2065, nk=9, kappa=1e-2 * UNIAXIAL),
    dict(n=700, nk=25, cd=0),
    dict(n=600, nk=50, kappa=1e-2 * FULL),
    dict(n=300, nk=57, kappa=1e-3 * SHEAR),             # the highest columns
    dict(n=200, nk=200, beta=20.0, kappa=0.05 * FULL),   # strands of 20 Kuhn steps and more
    dict(n=300, nk=40, beta=2.0, exp_wait=True),
    dict(n=300, nk=30, partner="gex"),
]


def _engine(lane):
    import gpu_dsm_amd as g
    e = g.Engine(0)
    e.set_option("small_per_cu", 0)
    e.set_option("lane", lane)
    return e


@pytest.mark.parametrize("case", CASES, ids=lambda c: "_".join("%s%s" % (k, v) for k, v in c.items() if k != "kappa"))
def test_lane_flow_matches_oracle(oracle, case):
    n, nk, beta, cd = case["n"], case["nk"], case.get("beta", 1.0), case.get("cd", 1)
    partner, ew, kappa = case.get("partner"), case.get("exp_wait", False), case.get("kappa", 1e-2 * SHEAR)
    P = oracle.Params(beta, nk, cd, kappa=kappa, exp_wait=ew, nmax=nk, partner=partner, gex=GEX)
    O = oracle.Ensemble(P, seed=41, n=n, salt=3)
    with _engine(2) as e:
        ens = e.add_ensemble(n, nk, beta, cd, kappa=list(kappa), seed=41, salt=3, exp_wait=ew, partner=partner, gex=GEX)
        e.init_equilibrium(ens)
        T = case.get("T", 6.0)
        for t in (0.5 * T, T):
            st = e.advance(ens, t)
            assert st["events"] == O.advance(t_end=t)[0]
            assert_same_state(e.state(ens), O.state(), "t = %g" % t)
        st = e.advance_events(ens, 37)
        assert st["events"] == O.advance(max_events=37)[0] == 37 * n
        assert_same_state(e.state(ens), O.state(), "37 jumps")


@pytest.mark.parametrize("n,nk,rate,delta", [(130, 12, 1e-2, 0.5), (700, 50, 1e-3, 1.0), (400, 40, 2.0, 0.25)])
def test_lane_flow_samples_of_several_ensembles(n, nk, rate, delta):
    out = []
    for lane in (0, 2):
        with _engine(lane) as e:
            ids = [e.add_ensemble(n + 5 * q, nk, 1.0, q % 2, kappa=list(rate * (q + 1) * FULL), seed=6, salt=q,
                                  sample="flow", delta=delta, window=3) for q in range(3)]
            for i in ids:
                e.init_equilibrium(i)
            for T in (2.0, 5.0):
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
                          {k: a[k][keep] for k in ("Z", "N", "Q", "w", "t", "ev")}, "flow")
        assert (a["events"], a["zs"], a["k0"]) == (b["events"], b["zs"], b["k0"])
        assert np.array_equal(_bits(a["rows"]), _bits(b["rows"]))
        assert np.array_equal(a["dt_prev"], b["dt_prev"]) and np.array_equal(a["next_sample"], b["next_sample"])


def test_lane_flow_outgrown_chains():
    """Chains of one Kuhn step per strand (Z = Nk = 50) and of 33 .. 37 strands, around the
    columns' 36 positions."""
    n, nk = 200, 50
    Z = np.where(np.arange(n) % 2, nk, 33 + np.arange(n) % 5).astype(np.int32)
    N = np.zeros((n, nk), np.int32)
    Q = np.zeros((n, nk, 3), np.float32)
    w = np.zeros((n, nk), np.float32)
    rng = np.random.default_rng(4)
    for i, z in enumerate(Z):
        N[i, :z] = 1
        N[i, z // 2] += nk - z
        Q[i, 1:z - 1] = rng.standard_normal((z - 2, 3))
        w[i, :z - 1] = 0.01
    out = []
    for lane in (0, 2):
        with _engine(lane) as e:
            ens = e.add_ensemble(n, nk, 1.0, 1, seed=12, kappa=list(1e-2 * SHEAR))
            e.set_state(ens, Z, N, Q, w)
            st = e.advance(ens, 3.0)
            out.append(dict(e.state(ens), events=st["events"]))
    a, b = out
    assert a["events"] == b["events"]
    assert_same_state(b, a, "outgrown")
