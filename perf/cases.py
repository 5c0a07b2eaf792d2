"""The work that users of this framework have it do, as timed cases.

Every case goes through the package's public entry points (Engine, serve).  A pass of an
equilibrium case advances every chain by a fixed number of Kuhn times (tau_K) and reads
the correlator, as a run that reports G(t) or MSD(t) while it goes on does; a pass of a
flow case is a start-up of flow from a new equilibrium draw with its stress rows; a pass
of a serving case is a whole burst of requests; a pass of an analysis case is the
ensemble stress and the integrity scan of a state in hand.  Jumps follow the seed, so the
outputs of a pass are the same for every layout of the work on the device.
"""
import math

import numpy as np

import gpu_dsm_amd as dsm
from gpu_dsm_amd.workloads import c3_lengths

JUMPS = 0.22        # jumps per chain, tau_K and Kuhn step, from the runs of the workloads
LEVELS = {2: 12, 8: 5}  # correlator levels by block factor: lags to 16 * 2**11 or 64 * 8**4 samples


def listed():
    return [
        # interactive stepping of a small system: 64 short chains, one tau_K a call
        dict(name="gt_tiny", kind="gt", n=64, nk=16, beta=1.0, cd=0, p=16, m=2, t=1.0),
        # the small command-line job: 1000 chains of 25 Kuhn steps, no constraint dynamics
        dict(name="gt_small_job", kind="gt", n=1000, nk=25, beta=1.0, cd=0, p=16, m=2, t=64.0),
        # an ordinary job with the driver's default correlator (64 points, factor 8), odd sizes
        dict(name="gt_default_lags", kind="gt", n=20011, nk=50, beta=2.0, cd=1, p=64, m=8, t=64.0),
        # the monodisperse melt: 131,072 chains of 100 Kuhn steps
        dict(name="gt_melt", kind="gt", n=131072, nk=100, beta=1.0, cd=1, p=16, m=2, t=16.0),
        # the polydisperse melt with constraint release by its own chains: the largest case
        dict(name="gt_polydisperse", kind="melt", n=262144, nk=200, beta=1.0, cd=1, p=16, m=2, t=16.0),
        # few well-entangled long chains: serial runs of thousands of jumps
        dict(name="gt_long_chains", kind="gt", n=1500, nk=1000, beta=1.0, cd=1, p=16, m=2, t=4.0),
        # diffusion: centre-of-mass MSD(t) of a medium ensemble
        dict(name="msd_medium", kind="msd", n=30011, nk=100, beta=1.0, cd=1, p=16, m=2, t=16.0),
        # probe chains in a polydisperse background (GEX weight distribution)
        dict(name="gt_gex_background", kind="gex", n=50021, nk=150, beta=1.0, cd=1, p=16, m=2, t=8.0),
        # shear-rate sweep: 16 ensembles of 16,384 chains advanced together
        dict(name="flow_sweep", kind="flow", n=16384, nk=50, beta=1.0, cd=1, ens=16, rate=1e-5, top=1e-1,
             shape="shear", delta=1.0, t=8.0),
        # start-up of uniaxial extension of one small ensemble, with the final chain state
        dict(name="flow_startup", kind="flow", n=3001, nk=30, beta=1.0, cd=1, ens=1, rate=1e-2, top=1e-2,
             shape="uniaxial", delta=0.5, t=10.0),
        # serving: a burst of mixed requests, half of them sheared
        dict(name="serve_burst", kind="serve", n=24, nk=512, low=1024, high=16384, t=10.0, window=5.0),
        # post-processing of a loaded state: ensemble stress and integrity scan
        dict(name="analysis", kind="analysis", n=20011, nk=200, beta=1.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above: chain counts 64..262,144 and lengths 10..1000
    over their logarithm, with the run length bounded so that none costs more than the
    polydisperse melt."""
    kind = rng.choice(["gt", "gt", "gt", "msd", "gex", "melt", "flow", "serve", "analysis"])
    if kind == "serve":
        return dict(kind="serve", n=rng.randint(4, 24), nk=16 * rng.randint(4, 32), low=1024,
                    high=_log(rng, 2048, 16384), t=5.0 * rng.randint(1, 2), window=5.0)
    beta = rng.choice([0.5, 1.0, 1.0, 2.0])
    if kind == "analysis":
        nk = _log(rng, 20, 600)
        return dict(kind="analysis", n=min(_log(rng, 500, 60000), 4000000 // nk), nk=nk, beta=beta)
    if kind == "flow":
        ens = rng.choice([1, 1, 2, 5, 16])
        nk = _log(rng, 10, 120)
        n = min(_log(rng, 64, 16384), 800000 // (ens * nk // 16 + 1))
        rate = 10.0 ** rng.uniform(-5.0, -1.5)
        return dict(kind="flow", n=n, nk=nk, beta=beta, cd=rng.randint(0, 1), ens=ens, rate=rate,
                    top=rate * (10.0 if ens > 1 else 1.0), shape=rng.choice(["shear", "uniaxial"]), delta=1.0,
                    t=float(rng.randint(2, 8)))
    nk = _log(rng, 10, 1000 if kind == "gt" else 300)
    n = min(_log(rng, 64, 262144), 16000000 // nk)
    most = min(4.0e7 / (JUMPS * n * nk), 2000.0 / (JUMPS * nk))  # all jumps, and those of one chain
    t = float(max(1, min(64, int(rng.uniform(0.3, 1.0) * most))))
    p, m = rng.choice([(16, 2), (16, 2), (64, 8)])
    return dict(kind=kind, n=n, nk=nk, beta=beta, cd=1 if kind in ("gex", "melt") else rng.randint(0, 1), p=p, m=m, t=t)


def _lengths(case, seed):
    """Log-normal lengths around the case's number average (Mw/Mn 1.5), 10..2000."""
    if case["nk"] == 200:
        return c3_lengths(case["n"], seed=seed)
    s2 = math.log(1.5)
    x = np.random.default_rng(seed).lognormal(math.log(case["nk"]) - s2 / 2, math.sqrt(s2), case["n"])
    return np.clip(np.rint(x), 10, 2000).astype(np.int32)


def _kappa(shape, rate):
    if shape == "shear":
        return [0, rate, 0, 0, 0, 0, 0, 0, 0]
    return [rate, 0, 0, 0, -rate / 2, 0, 0, 0, -rate / 2]


def _chains(case, seed):
    """A chain state: strand lengths cut at random Kuhn steps, Gaussian strand vectors
    (zero at both ends), exponentially distributed constraint-release rates."""
    n, nk = case["n"], case["nk"]
    rng = np.random.default_rng(seed)
    cut = rng.random((n, nk), dtype=np.float32) < 1.0 / (1.0 + case["beta"])
    cut[:, -1] = True
    row, col = np.nonzero(cut)
    Z = cut.sum(axis=1).astype(np.int32)
    start = np.concatenate([[0], np.cumsum(Z)[:-1]])
    k = np.arange(row.size) - start[row]
    length = np.where(k == 0, col + 1, col - np.concatenate([[0], col[:-1]])).astype(np.int32)
    N = np.zeros((n, nk), np.int32)
    N[row, k] = length
    Q = np.zeros((n, nk, 3), np.float32)
    inner = (k > 0) & (k < Z[row] - 1)
    sig = np.sqrt(length / 3.0).astype(np.float32) * inner
    Q[row, k] = rng.standard_normal((row.size, 3), dtype=np.float32) * sig[:, None]
    w = np.zeros((n, nk), np.float32)
    w[row, k] = (rng.standard_exponential(row.size, dtype=np.float32) * np.float32(0.02)) * (k < Z[row] - 1)
    return Z, N, Q, w


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, seed=seed, t=0.0)
    if kind == "serve":
        return s
    e = s["engine"] = dsm.Engine(0)
    common = dict(n_chains=case["n"], nk=case["nk"], beta=case["beta"], seed=seed)
    if kind == "analysis":
        ens = e.add_ensemble(cd=1, **common)
        e.set_state(ens, *_chains(case, seed))
        s["ids"] = [ens]
        return s
    if kind == "flow":
        k = case["ens"]
        s["ids"] = []
        for q in range(k):
            rate = case["rate"] * (case["top"] / case["rate"]) ** (q / max(1, k - 1))
            s["ids"].append(e.add_ensemble(cd=case["cd"], kappa=_kappa(case["shape"], rate), salt=q, sample="flow",
                                           delta=case["delta"], window=64, **common))
        return s
    more = {}
    if kind == "melt":
        lengths = _lengths(case, seed)
        common["nk"] = int(lengths.max())
        more = dict(nk_per_chain=lengths, partner="melt")
    elif kind == "gex":
        more = dict(partner="gex", gex=(1.5, 1.0, 40000.0, 120.0))
    ens = e.add_ensemble(cd=case["cd"], sample="msd" if kind == "msd" else "gt", delta=1.0, corr_p=case["p"],
                         corr_m=case["m"], corr_levels=LEVELS[case["m"]], window=64, **common, **more)
    e.init_equilibrium(ens)
    s["ids"] = [ens]
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "serve":
        # every request is in the queue at the start: the backlog sets the pace
        rep, _, summary = dsm.serve(summary=True, n_requests=case["n"], arrival_rate=1.0e9, seed=s["seed"],
                                    nk_min=16, nk_max=case["nk"], nk_step=16, nch_min=case["low"],
                                    nch_max=case["high"], horizon=case["t"], window=case["window"])
        return dict(completed=rep["completed"], jumps=rep["jumps"], summary=summary)
    e, ids = s["engine"], s["ids"]
    if kind == "analysis":
        stress, healthy = e.stress(ids[0])
        return dict(stress=stress, healthy=healthy, check=e.check(ids[0]))
    if kind == "flow":
        for ens in ids:
            e.init_equilibrium(ens)
        st = e.advance_many(ids, case["t"])
        out = dict(events=st["events"], rows=[e.flow_stress(ens) for ens in ids])
        if len(ids) == 1:
            state = e.state(ids[0])
            out["state"] = {k: state[k] for k in ("Z", "N", "Q", "w", "t")}
        return out
    s["t"] += case["t"]
    st = e.advance(ids[0], s["t"])
    lag, g = e.correlator(ids[0])
    return dict(events=st["events"], z_sum=st["z_sum"], lag=lag, g=g)


def work(case):
    """Bytes and operations of one pass.  Bytes: the chain state read and written once
    (Q, N, the CD rate: 20 per strand; about 80 per chain), the samples, and the
    correlator's registers that the samples touch.  Operations: per jump the rates of the
    three pairs next to the change (two exponentials each) and the choice of the event,
    about 250; under flow the rates of every pair; per sample 12 a strand and 6 a lag."""
    kind = case["kind"]
    if kind == "serve":
        n = case["n"] * (case["high"] - case["low"]) / math.log(case["high"] / case["low"])
        nk = (16 + case["nk"]) / 2.0
        z = nk / 2.0
        jumps = JUMPS * n * nk * case["t"]
        return dict(bytes=n * (40.0 * z + 160.0) + 32.0 * n * case["t"], flops=jumps * 250.0 + 0.5 * jumps * z * 90.0)
    n, nk = case["n"] * case.get("ens", 1), case["nk"]
    z = 1.0 + (nk - 1) / (1.0 + case["beta"])
    if kind == "analysis":
        return dict(bytes=2.0 * n * (20.0 * z + 60.0), flops=n * z * 30.0)
    t = case["t"]
    jumps = JUMPS * n * nk * t
    state = 2.0 * n * (20.0 * z + 80.0)
    if kind == "flow":
        rows = t / case["delta"]
        return dict(bytes=state + 32.0 * n * rows, flops=jumps * (250.0 + 90.0 * z) + rows * n * z * 30.0)
    return dict(bytes=state + n * (12.0 * t + 2 * 32.0 * case["p"]), flops=jumps * 250.0 + t * n * (12.0 * z + 6.0 * case["p"]))


def exact(case, seed):
    """The stress averages of the analysis cases in 64 bits.  The others are trajectories
    of a jump process: which event a jump picks follows the 32-bit rates, so they have no
    64-bit value to compare a single trajectory with."""
    if case["kind"] != "analysis":
        return None
    Z, N, Q, _ = _chains(case, seed)
    q = Q.astype(np.float64)
    t3 = np.where(N > 0, 3.0 / np.maximum(N, 1), 0.0)
    pairs = [(0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2)]
    sums = [-(t3 * q[..., a] * q[..., b]).sum() for a, b in pairs]
    sums += [np.sqrt((q ** 2).sum(axis=-1)).sum(), float(Z.sum())]
    return dict(stress=np.array(sums) / case["n"], healthy=None, check=None)
