"""The lane and solo forms with full waves and several chains a lane or wave, bit for bit
against the row, pair and wave forms (themselves compared with the oracle elsewhere).  One
wave a CU (DSM_OPT_BLOCKS_PER_CU) lets a few ten thousand chains fill every lane twice over:
rows that serve several chains a turn, records of eight chains shifted at once, column
strides to 65 lanes, the thresholds at which a wave does row work, and lanes that take their
next chain from the queue.  Each column height of both lane forms is met."""
import numpy as np
import pytest

from test_gpu_parity import GEX, _bits, assert_same_state

pytestmark = pytest.mark.gpu


def _run(opts, ens, t):
    import gpu_dsm_amd as g
    out = []
    with g.Engine(0) as e:
        for k, v in opts.items():
            e.set_option(k, v)
        ids = [e.add_ensemble(**d) for d in ens]
        for i in ids:
            e.init_equilibrium(i)
        st = e.advance_many(ids, t)
        for i, d in zip(ids, ens):
            s = e.state(i)
            if d["sample"] == "flow":
                s["rows"] = e.flow_stress(i)
            else:
                s["k0"], s["rows"] = e.last_samples(i)
                s["G"] = e.correlator(i)[1]
            out.append(s)
    return out, (st["events"], st["z_sum"])


def _same(a, b):
    (sa, ca), (sb, cb) = a, b
    assert ca == cb
    for x, y in zip(sa, sb):
        assert_same_state(y, x, "full waves")
        for k in x:
            if k in ("rows", "G"):
                assert np.array_equal(_bits(x[k]) if x[k].dtype == np.float32 else x[k],
                                      _bits(y[k]) if y[k].dtype == np.float32 else y[k]), k
            elif k in ("dt_prev", "next_sample", "stall", "R1"):
                assert np.array_equal(x[k], y[k]), k


def _still(n, nk, sample="gt", **more):
    return dict(n_chains=n, nk=nk, beta=more.pop("beta", 1.0), cd=more.pop("cd", 1), seed=17, sample=sample, delta=0.5,
                corr_p=16, corr_m=2, corr_levels=3, window=4, **more)


# positions a column (and lanes a wave that have room): 32, 48, 64 and 76 (64), 96 (51), 112 (43), 128 (39)
@pytest.mark.parametrize("n,nk,more", [
    (32700, 31, {}), (32700, 47, dict(sample="msd")), (32700, 75, dict(partner="gex", gex=GEX)),
    (32700, 100, {}), (32700, 100, dict(sample="msd", exp_wait=True)), (26100, 130, {}), (22000, 155, dict(cd=0)),
    (19900, 180, dict(sample="msd")), (32700, 90, dict(beta=6.0)), (30000, 3, {})], ids=str)
def test_lanes(n, nk, more):
    ens = [_still(n, nk, **dict(more))]
    base = dict(small_per_cu=0)
    _same(_run(dict(base, lane=0), ens, 3.0), _run(dict(base, lane=2, blocks_per_cu=1), ens, 3.0))


@pytest.mark.parametrize("sample", ["gt", "msd"])
def test_lanes_first_in_a_mixed_pass(sample):
    lens = np.random.default_rng(4).integers(10, 420, 30000).astype(np.int32)
    ens = [_still(lens.size, int(lens.max()), sample, nk_per_chain=lens, partner="melt")]
    _same(_run(dict(lane=0, concurrent=1), ens, 2.0), _run(dict(lane=2, concurrent=1, blocks_per_cu=1), ens, 2.0))


# 8, 12, ... 40 positions a chain (64 lanes to 16 positions, 27 at 40), of one and of four ensembles
@pytest.mark.parametrize("n,nk", [(32700, 7), (32700, 11), (32700, 15), (26000, 20), (22000, 27), (19000, 32),
                                  (16000, 40), (14500, 47), (13500, 54)])
def test_lanes_under_flow(n, nk):
    ens = [dict(n_chains=n // 4 + q, nk=nk, beta=1.0, cd=1, kappa=[0, 0.02 * (q + 1), 0, 0, 0, 0, 0, 0, 0], seed=5, salt=q,
                sample="flow", delta=0.5, window=4) for q in range(4)]
    base = dict(small_per_cu=0)
    for some in (ens, [dict(ens[0], n_chains=n)]):
        _same(_run(dict(base, lane=0), some, 2.0), _run(dict(base, lane=2, blocks_per_cu=1), some, 2.0))


@pytest.mark.parametrize("ens", [
    [_still(2000, 40)], [_still(1500, 200, "msd")], [_still(1200, 700)],
    [dict(n_chains=2000, nk=60, beta=1.0, cd=1, kappa=[0, 0.05, 0, 0, 0, 0, 0, 0, 0], seed=5, sample="flow", delta=0.5,
          window=4)]], ids=["short", "msd", "long", "flow"])
def test_waves_that_take_several_chains(ens):
    _same(_run(dict(solo=0), ens, 3.0), _run(dict(solo=1, blocks_per_cu=1), ens, 3.0))


def test_bin_2_two_chains_a_wave_beside_the_solo_form():
    ens = [_still(30000, 167, beta=0.4)]
    _same(_run(dict(lane=0, solo=0), ens, 1.5), _run(dict(lane=0), ens, 1.5))
