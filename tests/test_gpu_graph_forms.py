"""Captured windows of the lane and solo forms replay to the eager run's state: every window
checked, with the program's own eager work between the replays."""
import numpy as np
import pytest

from test_gpu_parity import GEX, _bits, assert_same_state

pytestmark = pytest.mark.gpu

KAPPA = [0, 1e-2, 0, 0, 0, 0, 0, 0, 0]
CASES = {
    "lanes": dict(ens=[dict(n=700, nk=60)], lane=2),
    "lanes_first": dict(ens=[dict(n=900, lo=10, hi=420)], lane=2, concurrent=1),
    "solo": dict(ens=[dict(n=200, nk=300)], lane=0),
    "solo_few": dict(ens=[dict(n=64, nk=16)], small=12),
    "flow_lanes": dict(ens=[dict(n=300, nk=40, flow=1), dict(n=200, nk=25, flow=1)], lane=2),
    "solo_flow": dict(ens=[dict(n=100, nk=90, flow=1), dict(n=80, nk=60)], small=12),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_captured_windows_match_eager(name):
    import gpu_dsm_amd as g
    case = CASES[name]
    out = []
    for graph in (0, 1):
        with g.Engine(0) as e:
            e.set_option("graph", graph)
            e.set_option("small_per_cu", case.get("small", 0))
            e.set_option("lane", case.get("lane", 1))
            e.set_option("concurrent", case.get("concurrent", -1))
            ids = []
            for q, d in enumerate(case["ens"]):
                lens, nk = None, d.get("nk")
                if "lo" in d:
                    lens = np.random.default_rng(3).integers(d["lo"], d["hi"] + 1, d["n"]).astype(np.int32)
                    nk = int(lens.max())
                flow = d.get("flow")
                ids.append(e.add_ensemble(d["n"], nk, 1.0, 1, seed=4, salt=q, nk_per_chain=lens, gex=GEX,
                                          kappa=KAPPA if flow else [0.0] * 9, sample="flow" if flow else "gt",
                                          delta=0.25, corr_levels=3, window=2))
            for i in ids:
                e.init_equilibrium(i)
            for t in (0.5, 1.0, 1.5, 2.0):  # one window a call: captured, then replayed
                st = e.advance_many(ids, t)
                for i in ids:
                    s = e.state(i)  # eager work between the replays
                    s["rows"] = e.last_samples(i)[1]
                    s["events"], s["zs"] = st["events"], st["z_sum"]
                    out.append(s)
    half = len(out) // 2
    for a, b in zip(out[:half], out[half:]):
        assert_same_state(b, a, name)
        assert (a["events"], a["zs"]) == (b["events"], b["zs"])
        assert np.array_equal(_bits(a["rows"]), _bits(b["rows"]))
