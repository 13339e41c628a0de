"""Timed cases of the RR / DET / LAM engine: the calls a program makes through the public entry points.

Kinds:
  host    RR / DET / LAM of one numpy series over a tau x emb grid (one call per measure asked for)
  device  rqa_device: RR, DET and LAM of one (tau, emb) for a series in GPU memory
  target  RR_target: the threshold of a wanted recurrence rate
  batch   rqa_batch: many series of mixed lengths in one call
  plot    rp_device: the recurrence plot, bytes in GPU memory

Sizes are those of the repository's benchmark configurations and tests, with odd lengths beside the round ones.
Series: the logistic map, an AR(1) process with a slow sine, the Lorenz and Roessler flows and white noise, drawn
from the seed.
"""
import math

import numpy as np
import torch

import accrqa_amd

EUCLIDEAN, MAXIMAL = accrqa_amd.DST_EUCLIDEAN, accrqa_amd.DST_MAXIMAL


def _case(name, kind, **kw):
    c = dict(kind=kind, series="ar1", n=10000, f64=False, norm=EUCLIDEAN, taus="1", embs="3", nthr=5, lo=0.1, hi=1.0,
             lmins="2", want="RR,DET,LAM")
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one recurrence rate of a short recording: call latency
        _case("rr_1000", "host", series="logistic", n=1000, embs="2", nthr=3, lo=0.05, hi=0.25, want="RR"),
        # the usual small study: one chaotic map series, every measure
        _case("logistic_10k", "device", series="logistic", n=10000, embs="3", nthr=5, lo=0.05, hi=0.25),
        # a parameter grid over one double-precision recording, DET and LAM asked one after the other
        _case("grid_4001_f64_max", "host", series="noise", n=4001, f64=True, norm=MAXIMAL, taus="1,2,4", embs="2,3,5",
              nthr=8, lo=0.05, hi=0.4, lmins="2,3", want="DET,LAM"),
        # a batch of recordings of mixed length on the same grid
        _case("batch_64", "batch", n=64, taus="1,2,4", embs="2,3,5", nthr=8, lo=0.05, hi=0.4),
        # DET alone of a long recording in a high embedding dimension
        _case("det_100003_m32", "host", n=100003, embs="32", nthr=16, lo=0.5, hi=8.0, want="DET"),
        # the threshold search, 20 bisection steps
        _case("target_65536_m16", "target", n=65536 + 15, embs="16", nthr=1, lo=0.05, hi=0.05),
        # a flow in its usual three-dimensional embedding, maximal norm, 20 thresholds
        _case("lorenz_131k_max", "device", series="lorenz", n=131072, norm=MAXIMAL, taus="8", embs="3", nthr=20,
              lo=0.02, hi=0.5),
        # double precision, odd length, high embedding dimension
        _case("ar1_65521_f64_m16", "device", n=65521, f64=True, embs="16", nthr=12, lo=0.4, hi=6.4),
        # the headline configuration
        _case("ar1_262k_m16", "device", n=262144, embs="16", nthr=16, lo=0.4, hi=6.4),
        # the longest series, 32 thresholds
        _case("rossler_1m_m10", "device", series="rossler", n=1048576, embs="10", nthr=32, lo=0.01, hi=0.3),
        # recurrence plots: a large aligned one, and one of odd size
        _case("plot_65536_m16", "plot", n=65536 + 15, embs="16", nthr=1, lo=4.0, hi=4.0),
        _case("plot_30011_m3", "plot", series="lorenz", n=30011 + 16, taus="8", embs="3", nthr=1, lo=0.25, hi=0.25),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "host", "device", "device", "device", "alone", "target", "batch", "plot", "plot"])
    c = dict(series=rng.choice(["logistic", "ar1", "lorenz", "noise"]), f64=rng.random() < 0.3,
             norm=rng.choice([EUCLIDEAN, EUCLIDEAN, MAXIMAL]))
    m = rng.choice([1, 2, 3, 3, 4, 5, 8, 10, 13, 16, 16, 24, 32, 64])
    tau = rng.choice([1, 1, 2, 3, 8])
    nthr = rng.randint(1, 32)
    if kind == "host":
        c["n"] = _log(rng, 600, 16384)
        c["taus"] = ",".join(map(str, sorted(rng.sample([1, 2, 3, 4], rng.randint(1, 2)))))
        c["embs"] = ",".join(map(str, sorted(rng.sample([1, 2, 3, 4, 5, 8, 12], rng.randint(1, 2)))))
        m = max(int(v) for v in c["embs"].split(","))
        c["lmins"] = rng.choice(["2", "2,3", "2,3,5,8"])
        c["want"] = rng.choice(["RR", "DET", "LAM", "RR,DET,LAM"])
        nthr = rng.randint(1, 12)
    elif kind == "alone":
        kind, c["n"], c["embs"], c["taus"] = "host", _log(rng, 16384, 131072), str(m), str(tau)
        c["want"] = rng.choice(["RR", "DET", "LAM"])
    elif kind == "device":
        c["n"] = _log(rng, 2000, 131072 if c["f64"] else 786432)
        if c["n"] > 262144:
            c["series"], m, tau = rng.choice(["rossler", "ar1"]), min(m, 10), 1
        c["embs"], c["taus"] = str(m), str(tau)
        c["lmins"] = rng.choice(["2", "2", "2,3,5"])
    elif kind == "target":
        m, nthr, c["f64"] = min(m, 16), 1, False
        c["n"], c["embs"], c["taus"] = _log(rng, 2000, 80000), str(m), str(tau)
        c["lo"] = c["hi"] = round(rng.uniform(0.01, 0.2), 4)
    elif kind == "batch":
        c["n"] = _log(rng, 4, 128)
        c["taus"], c["embs"], nthr, m = rng.choice(["1", "1,2", "1,2,4"]), rng.choice(["3", "2,3", "2,3,5"]), rng.randint(1, 12), 3
    else:
        m, nthr = min(m, 32), 1
        c["n"], c["embs"], c["taus"] = _log(rng, 1500, 80000), str(m), str(tau)
    c["nthr"] = nthr
    if "lo" not in c:
        # logistic series keep their range [0, 1]; the others have unit standard deviation
        scale = (0.4 if c["series"] == "logistic" else 1.0) * (math.sqrt(m) if c["norm"] == EUCLIDEAN else 1.0)
        c["lo"], c["hi"] = round(scale * rng.uniform(0.02, 0.2), 4), round(scale * rng.uniform(0.3, 1.2), 4)
    return _case(None, kind, **c)


# ---------------------------------------------------------------- series
def _flow(f, y, dt, steps):
    """x and dx/dt of a flow along RK4 steps of dt (a short transient dropped)."""
    a, b, c = y
    h, s = 0.5 * dt, dt / 6.0
    xs, ds = [], []
    for k in range(steps + 500):
        k1, l1, m1 = f(a, b, c)
        if k >= 500:
            xs.append(a)
            ds.append(k1)
        k2, l2, m2 = f(a + h * k1, b + h * l1, c + h * m1)
        k3, l3, m3 = f(a + h * k2, b + h * l2, c + h * m2)
        k4, l4, m4 = f(a + dt * k3, b + dt * l3, c + dt * m3)
        a += s * (k1 + 2.0 * (k2 + k3) + k4)
        b += s * (l1 + 2.0 * (l2 + l3) + l4)
        c += s * (m1 + 2.0 * (m2 + m3) + m4)
    return np.array(xs), np.array(ds)


def _dense(x, d, dt, per, n):
    """`per` samples a step between the steps, by cubic Hermite interpolation."""
    out = np.empty(((len(x) - 1), per))
    for k in range(per):
        u = k / per
        out[:, k] = ((1 + 2 * u) * (1 - u) ** 2 * x[:-1] + u * (1 - u) ** 2 * dt * d[:-1]
                     + u * u * (3 - 2 * u) * x[1:] + u * u * (u - 1) * dt * d[1:])
    return out.reshape(-1)[:n]


def _series(kind, n, rng):
    if kind == "logistic":
        v, out = rng.uniform(0.1, 0.9), [0.0] * n
        r = rng.uniform(3.9, 4.0)
        for k in range(n):
            out[k] = v
            v = r * v * (1.0 - v)
        return np.array(out)
    if kind == "noise":
        return rng.standard_normal(n)
    if kind == "ar1":
        v, out = 0.0, rng.standard_normal(n).tolist()
        for k in range(n):
            v = 0.95 * v + out[k]
            out[k] = v
        x = np.array(out) + 0.3 * np.sin(2 * np.pi * np.arange(n) / 1000.0 + rng.uniform(0, 6.0))
    elif kind == "lorenz":   # 0.01 a sample
        y = (1.0 + rng.uniform(0, 5), 1.0 + rng.uniform(0, 5), 20.0 + rng.uniform(0, 5))
        x, d = _flow(lambda a, b, c: (10.0 * (b - a), a * (28.0 - c) - b, a * b - 8.0 / 3.0 * c), y, 0.02, n // 2 + 2)
        x = _dense(x, d, 0.02, 2, n)
    else:                    # rossler, 0.05 a sample
        y = (1.0 + rng.uniform(0, 2), rng.uniform(0, 2), rng.uniform(0, 1))
        x, d = _flow(lambda a, b, c: (-b - c, a + 0.2 * b, 0.2 + c * (a - 5.7)), y, 0.2, n // 4 + 2)
        x = _dense(x, d, 0.2, 4, n)
    return (x - x.mean()) / x.std()


def _ints(text):
    return [int(v) for v in text.split(",")]


def _thresholds(case):
    return np.linspace(case["lo"], case["hi"], case["nthr"])


def _batch_lengths(case):
    """Lengths of the batch's series, log-uniform from 512 to 32,768: a part of the case, not of its seed."""
    rng = np.random.default_rng([7, case["n"], case["nthr"]])
    return [int(v) for v in np.exp(rng.uniform(np.log(512), np.log(32768), case["n"]))]


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    dt = np.float64 if case["f64"] else np.float32
    s = dict(kind=case["kind"], norm=case["norm"], taus=_ints(case["taus"]), embs=_ints(case["embs"]),
             lmins=_ints(case["lmins"]), dtype=dt, thr=_thresholds(case).astype(dt))
    if s["kind"] == "batch":
        # one third AR(1), one third logistic maps, one third white noise; thresholds relative to each series
        s["series"] = [_series(("ar1", "logistic", "noise")[k % 3], n, rng).astype(dt)
                       for k, n in enumerate(_batch_lengths(case))]
        s["thr"] = np.array([_thresholds(case) * x.std() for x in s["series"]]).astype(dt)
        return s
    x = _series(case["series"], case["n"], rng).astype(dt)
    if s["kind"] in ("host", "target"):
        s["x"], s["want"], s["target"] = x, case["want"].split(","), case["lo"]
        return s
    s["x"] = torch.from_numpy(x).cuda()
    if s["kind"] == "device":
        t, nl, td = case["nthr"], len(s["lmins"]), s["x"].dtype
        s["rr"] = torch.empty(t, dtype=td, device="cuda")
        s["det"] = torch.empty(t, nl, 5, dtype=td, device="cuda")
        s["lam"] = torch.empty(nl, t, 5, dtype=td, device="cuda")
    else:
        nc = case["n"] - (s["embs"][0] - 1) * s["taus"][0]
        s["plot"] = torch.empty(nc, nc, dtype=torch.int8, device="cuda")
    return s


def run(s):
    k = s["kind"]
    if k == "host":
        out = {}
        if "RR" in s["want"]:
            out["RR"] = accrqa_amd.RR(s["x"], s["taus"], s["embs"], s["thr"], s["norm"])
        if "DET" in s["want"]:
            out["DET"] = accrqa_amd.DET(s["x"], s["taus"], s["embs"], s["lmins"], s["thr"], s["norm"])
        if "LAM" in s["want"]:
            out["LAM"] = accrqa_amd.LAM(s["x"], s["taus"], s["embs"], s["lmins"], s["thr"], s["norm"])
        return out
    if k == "target":
        thr, rr = accrqa_amd.RR_target(s["x"], s["taus"][0], s["embs"][0], s["target"], s["norm"], epsilon=1e-5)
        return {"threshold": thr, "RR": rr}
    if k == "batch":
        return accrqa_amd.rqa_batch(s["series"], s["taus"], s["embs"], s["lmins"], s["thr"], s["norm"])
    x = s["x"]
    st = torch.cuda.current_stream().cuda_stream
    if k == "device":
        accrqa_amd.rqa_device(x.data_ptr(), x.numel(), s["taus"][0], s["embs"][0], s["thr"], s["lmins"], s["norm"],
                              s["rr"].data_ptr(), s["det"].data_ptr(), s["lam"].data_ptr(), st, s["dtype"])
        return {"RR": s["rr"], "DET": s["det"], "LAM": s["lam"]}
    accrqa_amd.rp_device(x.data_ptr(), x.numel(), s["taus"][0], s["embs"][0], float(s["thr"][0]), s["norm"],
                         s["plot"].data_ptr(), st, s["dtype"])
    return {"RP": s["plot"]}


# ---------------------------------------------------------------- work
def _blocks(case):
    lengths = _batch_lengths(case) if case["kind"] == "batch" else [case["n"]]
    return [(n - (m - 1) * t, m) for n in lengths for t in _ints(case["taus"]) for m in _ints(case["embs"])]


def work(case):
    """Each sample read once, each result written once; every distinct pair's distance (subtract, multiply, add per
    dimension; subtract, compare for the maximal norm) and its comparison with every threshold."""
    es = 8 if case["f64"] else 4
    per = 3 if case["norm"] == EUCLIDEAN else 2
    nb = _blocks(case)
    pairs = sum(nc * (nc + 1) / 2 * (per * m + case["nthr"]) for nc, m in nb)
    samples = sum(_batch_lengths(case)) if case["kind"] == "batch" else case["n"]
    outs = len(nb) * case["nthr"] * (1 + 10 * len(_ints(case["lmins"])))
    b = samples * es + outs * es
    if case["kind"] == "plot":
        b = samples * es + nb[0][0] ** 2
    return {"bytes": b, "flops": pairs}


# ---------------------------------------------------------------- 64 bits
def _distances(x, tau, m, norm, rows):
    nc = x.numel() - (m - 1) * tau
    d = torch.zeros(rows.stop - rows.start, nc, dtype=torch.float64, device=x.device)
    for k in range(m):
        v = x[k * tau:k * tau + nc]
        e = (v[rows, None] - v[None, :]).abs_()
        d = torch.maximum(d, e) if norm == MAXIMAL else d.addcmul_(e, e)
    return d if norm == MAXIMAL else d.sqrt_()


def _runs(seqs):
    """Histogram of the run lengths of ones along the rows."""
    rows, n = seqs.shape
    h = torch.zeros(n + 1, dtype=torch.int64, device=seqs.device)
    step = max(1, (1 << 27) // n)
    for r in range(0, rows, step):
        f = torch.nn.functional.pad(seqs[r:r + step], (1, 1)).reshape(-1)
        e = f[1:].to(torch.int8) - f[:-1].to(torch.int8)
        h += torch.bincount((e == -1).nonzero()[:, 0] - (e == 1).nonzero()[:, 0], minlength=n + 1)[:n + 1]
    return h.double().cpu().numpy()


def _five(h, lmin, nc, longest):
    f = np.arange(nc + 1, dtype=np.float64)
    part, fp = h[lmin:], f[lmin:]
    s, m, m0 = part.sum(), (part * fp).sum(), (h * f).sum()
    p = part[part > 0] / s if s > 0 else np.zeros(0)
    return [m / m0 if m0 > 0 else np.nan, m / s if s > 0 else np.nan, longest, -(p * np.log(p)).sum() if s > 0 else 0.0,
            m0 / (nc * nc)]


def _exact_block(x, tau, m, thr, lmins, norm, det, lam):
    """(rr [T], DET [T][nL][5], LAM [nL][T][5]) of one (tau, emb), from the full matrix."""
    nc = x.numel() - (m - 1) * tau
    d = torch.cat([_distances(x, tau, m, norm, slice(r, min(r + 2048, nc))) for r in range(0, nc, 2048)])
    rr, dd, ll = [], [], []
    for t in thr:
        R = d <= float(t)
        rr.append(float(R.sum()) / (nc * nc))
        if lam:
            h = _runs(R)
            top = np.flatnonzero(h)
            ll.append([_five(h, v, nc, float(top[-1]) if top.size else 0.0) for v in lmins])
        if det:
            W = torch.nn.functional.pad(R, (0, nc))
            h = 2.0 * _runs(W.as_strided((nc - 1, nc), (1, 2 * nc + 1), 1)) if nc > 1 else np.zeros(nc + 1)
            top = np.flatnonzero(h)
            h[nc] += 1.0
            dd.append([_five(h, v, nc, float(top[-1]) if top.size else 0.0) for v in lmins])
    return np.array(rr), np.array(dd), np.array(ll).transpose(1, 0, 2) if lam else None


def exact(case, seed):
    s = prepare(case, seed)
    thr, nb = s["thr"].astype(np.float64), _blocks(case)
    if case["kind"] == "target":
        x = torch.as_tensor(s["x"]).cuda().double()
        nc, m = nb[0]
        d = torch.cat([_distances(x, s["taus"][0], m, s["norm"], slice(r, min(r + 1024, nc))) for r in range(0, nc, 1024)])

        def rate(t):
            return sum(int((d[r:r + 4096] <= float(np.float32(t))).sum()) for r in range(0, nc, 4096)) / (nc * nc)

        lo, hi = 0.0, 10.0
        span = rate(hi) - rate(lo)
        for _ in range(20):
            mid = (hi - lo) / 2.0 + lo
            rr = rate(mid)
            if abs(rr - s["target"]) < 1e-5 or span < 1e-5:
                return {"threshold": mid, "RR": rr}
            lo, hi = (mid, hi) if rr < s["target"] else (lo, mid)
        return {"threshold": (hi - lo) / 2.0 + lo, "RR": rr}
    if case["kind"] in ("plot", "batch"):
        return None   # whole numbers; and too many blocks
    want = s["want"] if case["kind"] == "host" else ["RR", "DET", "LAM"]
    kinds = ("DET" in want) + ("LAM" in want)
    if max(nc for nc, _ in nb) > 20000 or sum(nc * nc for nc, _ in nb) * case["nthr"] * (1 + 8 * kinds) > 4e10:
        return None   # too long
    x = torch.as_tensor(s["x"]).cuda().double()
    got = [_exact_block(x, t, m, thr, s["lmins"], s["norm"], "DET" in want, "LAM" in want)
           for t in s["taus"] for m in s["embs"]]
    if case["kind"] == "device":
        return dict(zip(("RR", "DET", "LAM"), got[0]))
    lead = (len(s["taus"]), len(s["embs"]))
    return {k: np.stack([g[i] for g in got]).reshape(lead + got[0][i].shape)
            for i, k in enumerate(("RR", "DET", "LAM")) if k in want}
