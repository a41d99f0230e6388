"""Performance cases: the pricings a user of this engine runs, and their values in plain 64-bit arithmetic.

A case names a product, its sizes and its options; the market (spot, strike,
rate, volatilities, maturity, correlations) and the generator seed come from
the seed given to prepare().  One pass is one call of a public entry point of
parcompfin_amd (Engine.mc_eur, mc_asia, mc_eur_multi, mc_amer, binom_embar,
binom_vanilla), or one set of requests through the Server.  Results of FP32
pricings are returned as float32, those of FP64 pricings as float64.
"""
import functools
import math
import weakref

import numpy as np
import torch

from parcompfin_amd import Engine, Server

# The American pricing carries a path store; the others only parameters.
PRODUCTS = ("european", "asian", "basket", "american", "binomial", "lattice")


def listed():
    return [
        # One quote of a European option at the smallest path count that is
        # worth a GPU: the latency of a call.
        dict(name="european 16k fp32", product="european", paths=1 << 14, precision="fp32k", payoff="call"),
        # The reference's largest published European run, in FP64.
        dict(name="european 100M fp64", product="european", paths=10**8, precision="fp64", payoff="put"),
        # The daily-averaged Asian at its configuration's full size.
        dict(name="asian 4M x 252 fp32", product="asian", paths=1 << 22, steps=252, precision="fp32k",
             payoff="call", control=False),
        # An FP64 Asian with its geometric control, calendar-day averaging: a
        # path count and a step count that no tile divides.
        dict(name="asian 500k x 365 fp64 control", product="asian", paths=500_003, steps=365, precision="fp64",
             payoff="call", control=True),
        # A small index: 8 names, one correlation, a volatility each.
        dict(name="basket 8 x 4M fp32", product="basket", paths=1 << 22, assets=8, precision="fp32k",
             payoff="call", correlation="one"),
        # A wider index with an estimated correlation matrix.
        dict(name="basket 32 x 3M matrix fp32", product="basket", paths=3_000_001, assets=32, precision="fp32k",
             payoff="call", correlation="matrix"),
        # A quick American put: latency of the date sweep.
        dict(name="american 16k x 50 fp32", product="american", paths=1 << 14, steps=50, precision="fp32k",
             payoff="put"),
        # The American put at its configuration's full size.
        dict(name="american 1M x 50 fp32", product="american", paths=1 << 20, steps=50, precision="fp32k",
             payoff="put"),
        # An FP64 American put with twice the dates, ragged path count.
        dict(name="american 600k x 100 fp64", product="american", paths=600_002, steps=100, precision="fp64",
             payoff="put"),
        # The closed binomial sum in the reference's own operation order, at
        # the size whose value the reference publishes.
        dict(name="binomial 100k chain", product="binomial", levels=10**5, chain=True, payoff="call"),
        # The American lattice that the reference compares its LSM prices with.
        dict(name="lattice american 10k", product="lattice", levels=10**4, american=True, payoff="put"),
        # A desk's request set through the server: the four Monte Carlo
        # products over their range of path counts.
        dict(name="served mix of 24", product="mix", requests=24, log2_from=14, log2_to=21, precision="fp32k"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    product = rng.choice(PRODUCTS)
    precision = rng.choice(("fp32k", "fp32k", "fp64"))
    payoff = rng.choice(("call", "put"))
    if product == "european":
        return dict(product=product, paths=_log_uniform(rng, 1 << 10, 10**8), precision=precision, payoff=payoff)
    if product == "asian":
        steps = _log_uniform(rng, 4, 365)
        most = min(1 << 22, ((1 << 30) if precision == "fp32k" else (1 << 27)) // steps)
        return dict(product=product, paths=_log_uniform(rng, 1 << 10, most), steps=steps, precision=precision,
                    payoff=payoff, control=rng.random() < 0.4)
    if product == "basket":
        assets = _log_uniform(rng, 2, 64)
        most = ((1 << 27) if precision == "fp32k" else (1 << 24)) // assets
        return dict(product=product, paths=_log_uniform(rng, 1 << 10, most), assets=assets, precision=precision,
                    payoff=payoff, correlation=rng.choice(("one", "one", "matrix")))
    if product == "american":
        steps = _log_uniform(rng, 6, 252)
        most = min(1 << 22, ((1 << 26) if precision == "fp32k" else (1 << 25)) * 3 // steps)
        return dict(product=product, paths=2 * _log_uniform(rng, 1 << 9, most // 2), steps=steps,
                    precision=precision, payoff=payoff)
    if product == "binomial":
        return dict(product=product, levels=_log_uniform(rng, 50, 10**5), chain=rng.random() < 0.6, payoff=payoff)
    return dict(product=product, levels=_log_uniform(rng, 50, 10**4), american=rng.random() < 0.6, payoff=payoff)


# ---------------------------------------------------------------- inputs

@functools.lru_cache(maxsize=1)
def _engine():
    """The process's context, as a pricing program keeps one."""
    return Engine(0)


_servers = weakref.WeakValueDictionary()


def _server():
    """The process's server; closed when no request set refers to it."""
    srv = _servers.get(0)
    if srv is None:
        srv = _servers[0] = Server(_engine(), mem_budget_bytes=16 << 30, max_inflight=4)
    return srv


def _market(case, seed):
    """Market data and generator seed of a pricing."""
    rng = np.random.default_rng([int(seed), 17])
    S0 = float(rng.uniform(80.0, 120.0))
    m = dict(S0=S0, E=S0 * float(rng.uniform(0.9, 1.1)), r=float(rng.uniform(0.01, 0.07)),
             sigma=float(rng.uniform(0.15, 0.4)), T=float(rng.uniform(0.5, 2.0)), seed=int(rng.integers(1, 2**62)))
    if case["product"] == "basket":
        d = case["assets"]
        m["rho"] = float(rng.uniform(0.1, 0.7))
        m["sigmas"] = rng.uniform(0.15, 0.4, size=d)
        if case["correlation"] == "matrix":
            # a factor model's correlations: two factors and specific risk
            f = rng.normal(size=(d, 2)) * np.array([0.5, 0.4]) + np.array([0.8, 0.0])
            cov = f @ f.T + np.diag(rng.uniform(0.3, 0.8, size=d))
            s = np.sqrt(np.diag(cov))
            m["corr"] = cov / np.outer(s, s)
            m["corr"] = 0.5 * (m["corr"] + m["corr"].T)
            np.fill_diagonal(m["corr"], 1.0)
    return m


def _mix(case):
    """The request set of a served mix: its products and path counts."""
    n = case["requests"]
    kinds = ("european", "basket", "asian", "american")
    made = []
    for i in range(n):
        kind = kinds[i % 4]
        # each product runs over the whole range of path counts
        at = ((i // 4) * 4 + (i * 7 + 2) % 4 + 0.5) / n
        paths = int(round(2 ** (case["log2_from"] + at * (case["log2_to"] - case["log2_from"])))) // 2 * 2
        c = dict(product=kind, paths=paths, precision=case["precision"], payoff="put" if kind == "american" else "call")
        if kind == "basket":
            c.update(assets=8, correlation="one")
        elif kind == "asian":
            c.update(steps=252, control=False)
        elif kind == "american":
            c.update(steps=50)
        made.append(c)
    return made


def prepare(case, seed):
    if case["product"] == "mix":
        cases = _mix(case)
        return dict(case=case, server=_server(), cases=cases,
                    markets=[_market(c, seed * 1000 + i) for i, c in enumerate(cases)])
    return dict(case=case, engine=_engine(), market=_market(case, seed))


# ---------------------------------------------------------------- one pass

def _outputs(case, r):
    """The numbers of a pricing, in the type it was computed in."""
    t = np.float32 if case.get("precision") == "fp32k" else np.float64
    if case["product"] in ("binomial", "lattice"):
        return dict(price=t(r.price))
    out = dict(price=t(r.price), std_err=t(r.std_err), mean=t(r.mean), variance=t(r.variance))
    if case["product"] == "american" or case.get("control"):
        out.update(control_price=t(r.control_price), control_se=t(r.control_se))
    if case["product"] == "american":
        out.update(dates_small=int(r.lsm_small_itm), dates_reduced=int(r.lsm_fallback))
    return out


def run(state):
    case = state["case"]
    if case["product"] == "mix":
        srv = state["server"]
        tickets = []
        for c, m in zip(state["cases"], state["markets"]):
            kind = {"european": "eur", "asian": "asia", "american": "amer", "basket": "basket"}[c["product"]]
            kw = dict(M=c.get("steps", 0), precision=c["precision"], seed=m["seed"])
            if kind == "basket":
                kw.update(assets=c["assets"], rho=m["rho"], sigmas=m["sigmas"])
            tickets.append(srv.submit(kind, m["S0"], m["E"], m["r"], m["sigma"], m["T"], c["paths"], c["payoff"], **kw))
        got = [_outputs(c, srv.wait(t)) for c, t in zip(state["cases"], tickets)]
        t = np.float32 if case["precision"] == "fp32k" else np.float64
        return {k: np.array([g[k] for g in got], dtype=t) for k in ("price", "std_err", "mean", "variance")}
    eng, m = state["engine"], state["market"]
    a = (m["S0"], m["E"], m["r"], m["sigma"], m["T"])
    if case["product"] == "european":
        r = eng.mc_eur(*a, case["paths"], case["payoff"], seed=m["seed"], precision=case["precision"])
    elif case["product"] == "asian":
        r = eng.mc_asia(*a, case["paths"], case["steps"], case["payoff"], seed=m["seed"],
                        precision=case["precision"], control=case["control"])
    elif case["product"] == "basket":
        r = eng.mc_eur_multi(*a, case["paths"], case["payoff"], case["assets"], m["rho"], sigmas=m["sigmas"],
                             corr=m.get("corr"), seed=m["seed"], precision=case["precision"])
    elif case["product"] == "american":
        r = eng.mc_amer(*a, case["paths"], case["steps"], case["payoff"], seed=m["seed"],
                        precision=case["precision"])
    elif case["product"] == "binomial":
        r = eng.binom_embar(*a, case["levels"], case["payoff"], ref_exact=case["chain"])
    else:
        r = eng.binom_vanilla(*a, case["levels"], case["payoff"], american=case["american"])
    return _outputs(case, r)


# ---------------------------------------------------------------- work of a pass

def _work(case):
    """Operations that a pricing cannot do without: a fused multiply-add is 2,
    a normal 6, an elementary function 1.  Parameters in and results out are
    its only bytes, except the American's paths, which go out and come back."""
    p = case["product"]
    real = 4.0 if case.get("precision") == "fp32k" else 8.0
    if p == "european":
        return 256.0, 13.0 * case["paths"]
    if p == "asian":
        return 256.0, (14.0 + (2.0 if case["control"] else 0.0)) * case["paths"] * case["steps"]
    if p == "basket":
        d = case["assets"]
        # one correlation: the factor's columns are constant below the diagonal
        per = (4.0 * d if case["correlation"] == "one" else d * (d + 1.0)) + 11.0 * d + 3.0
        return 256.0 + 8.0 * d * d, per * case["paths"]
    if p == "american":
        n = float(case["paths"]) * case["steps"]
        # forward: half a normal, drift 2, exp, product; backward: payoff 2,
        # x and its powers 2, eight sums 12, fit 5, test 1
        return 2.0 * real * n, (3.0 + 4.0 + 22.0) * n
    N = float(case["levels"])
    if p == "binomial":
        return 16.0 * N, (0.375 * N * N if case["chain"] else 0.0) + 24.0 * N
    return 32.0 * N, 0.5 * N * N * (9.0 if case["american"] else 4.0)


def work(case):
    parts = [_work(c) for c in _mix(case)] if case["product"] == "mix" else [_work(case)]
    return {"bytes": sum(b for b, _ in parts), "flops": sum(f for _, f in parts)}


# ---------------------------------------------------------------- values in 64 bits

_MASK = 0xFFFFFFFF
_STREAM = {"european": 1, "asian": 2, "american": 3, "basket": 4}


def _normals(seed, stream, path, block):
    """The four standard normals of (path, block): Philox4x32-10 and Box-Muller in float64."""
    c = [torch.full_like(path, block), path & _MASK, path >> 32, torch.full_like(path, stream)]
    k0, k1 = seed & _MASK, seed >> 32
    for _ in range(10):
        p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
        c = [((p1 >> 32) & _MASK) ^ c[1] ^ k0, p1 & _MASK, ((p0 >> 32) & _MASK) ^ c[3] ^ k1, p0 & _MASK]
        k0, k1 = (k0 + 0x9E3779B9) & _MASK, (k1 + 0xBB67AE85) & _MASK
    u = [(x.double() + 0.5) * 2.0**-32 for x in c]
    z = []
    for a, b in ((u[0], u[1]), (u[2], u[3])):
        R = torch.sqrt(-2.0 * torch.log(a))
        z += [R * torch.cos(2.0 * math.pi * b), R * torch.sin(2.0 * math.pi * b)]
    return z


def _moments(sums, n):
    s, q = sums
    mean = s / n
    return mean, (q - s * mean) / (n - 1.0) if n > 1 else 0.0


def _simulated(case, m):
    """Sums of the payoffs (and of the control's) of a single-pass product."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    sign = 1.0 if case["payoff"] == "call" else -1.0
    S0, E, r, sigma, T = (m[k] for k in ("S0", "E", "r", "sigma", "T"))
    n, product = case["paths"], case["product"]
    stream = _STREAM[product]
    per = 4 if product == "european" else 1
    chunk = 1 << 21
    total = np.zeros(4, dtype=np.longdouble)
    if product == "basket":
        d = case["assets"]
        C = m.get("corr")
        if C is None:
            C = np.full((d, d), m["rho"])
            np.fill_diagonal(C, 1.0)
        L = torch.tensor(np.linalg.cholesky(C), device=dev)
        sg = torch.tensor(m["sigmas"], device=dev)
    for at in range(0, (n + per - 1) // per, chunk):
        path = torch.arange(at, min(at + chunk, (n + per - 1) // per), device=dev)
        geo = None
        if product == "european":
            z = torch.stack(_normals(m["seed"], stream, path, 0), dim=1).reshape(-1)[: n - 4 * at]
            v = S0 * torch.exp((r - 0.5 * sigma * sigma) * T + sigma * math.sqrt(T) * z)
        elif product == "basket":
            z = [t for b in range((d + 3) // 4) for t in _normals(m["seed"], stream, path, b)][:d]
            B = torch.stack(z, dim=1) @ L.T.contiguous()
            v = (S0 / d) * torch.exp((r - 0.5 * sg * sg) * T + sg * math.sqrt(T) * B).sum(dim=1)
        else:
            M = case["steps"]
            dt = T / M
            mu, vol = (r - 0.5 * sigma * sigma) * dt, sigma * math.sqrt(dt)
            S = torch.full(path.shape, S0, dtype=torch.float64, device=dev)
            I, ls, lsum = torch.zeros_like(S), torch.zeros_like(S), torch.zeros_like(S)
            for step in range(M):
                if step % 4 == 0:
                    z4 = _normals(m["seed"], stream, path, step // 4)
                z = z4[step % 4]
                I += S * (1.0 + 0.5 * r * dt + 0.5 * vol * z)
                e = mu + vol * z
                S *= torch.exp(e)
                if case["control"]:
                    ls += e
                    lsum += ls
            v = I / M
            if case["control"]:
                geo = S0 * torch.exp(lsum / M)
        pay = (sign * (v - E)).clamp_min(0.0)
        total[:2] += [float(pay.sum()), float((pay * pay).sum())]
        if geo is not None:
            pay = (sign * (geo - E)).clamp_min(0.0)
            total[2:] += [float(pay.sum()), float((pay * pay).sum())]
    return total


def _exact_american(case, m):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    sign = 1.0 if case["payoff"] == "call" else -1.0
    S0, E, r, sigma, T = (m[k] for k in ("S0", "E", "r", "sigma", "T"))
    N, M = case["paths"], case["steps"]
    half, dt = N // 2, T / M
    mu, vol = (r - 0.5 * sigma * sigma) * dt, sigma * math.sqrt(dt)
    store = torch.empty((M + 1, N), dtype=torch.float64, device=dev)
    store[0] = S0
    path = torch.arange(half, device=dev)
    for step in range(1, M + 1):
        if step % 4 == 1:
            z4 = _normals(m["seed"], _STREAM["american"], path, (step - 1) // 4)
        z = z4[(step - 1) % 4]
        store[step, :half] = store[step - 1, :half] * torch.exp(mu + vol * z)
        store[step, half:] = store[step - 1, half:] * torch.exp(mu - vol * z)
    cash = (sign * (store[M] - E)).clamp_min(0.0)
    mean, var = _moments((float(cash.sum()), float((cash * cash).sum())), N)
    discT = math.exp(-r * T)
    control = dict(control_price=discT * mean, control_se=discT * math.sqrt(var / N))
    when = torch.full((N,), M, dtype=torch.int64, device=dev)
    disc = torch.tensor([math.exp(-r * dt * k) for k in range(M + 1)], dtype=torch.float64, device=dev)
    for date in range(M - 1, 0, -1):
        S = store[date]
        pay = (sign * (S - E)).clamp_min(0.0)
        itm = pay > 0
        n = int(itm.sum())
        if n == 0:
            continue
        y = disc[when - date] * cash
        if n <= 2:
            ex = itm & (pay > y)
        else:
            # the quadratic fit, centred at the strike
            x = S / E - 1.0
            w = itm.double()
            p = [w, w * x, w * x * x, w * x**3, w * x**4]
            s = [float(t.sum()) for t in p]
            G = np.array([[s[i + j] for j in range(3)] for i in range(3)])
            c = np.linalg.lstsq(G, np.array([float((p[i] * y).sum()) for i in range(3)]), rcond=1e-14)[0]
            ex = itm & (pay > c[0] + x * (c[1] + x * c[2]))
        when = torch.where(ex, date, when)
        cash = torch.where(ex, pay, cash)
    v = disc[when] * cash
    mean, var = _moments((float(v.sum()), float((v * v).sum())), N)
    return dict(price=max(max(sign * (S0 - E), 0.0), mean), std_err=math.sqrt(var / N), mean=mean, variance=var,
                dates_small=None, dates_reduced=None, **control)


def _tree(m, N):
    """The beta tree's up and down factors, growth and probability."""
    dt = m["T"] / N
    beta = 0.5 * (math.exp(-m["r"] * dt) + math.exp((m["r"] + m["sigma"] ** 2) * dt))
    root = math.sqrt(beta**2 - 1)
    u, d, R = beta + root, beta - root, math.exp(m["r"] * dt)
    return u, d, R, (R - d) / (u - d)


def _exact_binomial(case, m):
    N = case["levels"]
    u, d, _, p = (np.longdouble(t) for t in _tree(m, N))
    sign = 1.0 if case["payoff"] == "call" else -1.0
    i = np.arange(N + 1, dtype=np.longdouble)
    lf = np.concatenate([[np.longdouble(0)], np.cumsum(np.log(i[1:]))])
    w = np.exp(lf[N] - lf - lf[::-1] + i * np.log(p) + (N - i) * np.log(1 - p))
    S = m["S0"] * np.exp(i * np.log(u) + (N - i) * np.log(d))
    return dict(price=float(np.exp(-np.longdouble(m["r"]) * m["T"]) * np.sum(w * np.maximum(sign * (S - m["E"]), 0))))


def _exact_lattice(case, m):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    N = case["levels"]
    u, d, R, p = _tree(m, N)
    sign = 1.0 if case["payoff"] == "call" else -1.0
    i = torch.arange(N + 1, dtype=torch.float64, device=dev)
    up, dn = torch.pow(u, i), torch.pow(d, i)
    v = (sign * (m["S0"] * up * dn.flip(0) - m["E"])).clamp_min(0.0)
    for n in range(N - 1, -1, -1):
        v = (p * v[1:] + (1.0 - p) * v[:-1]) / R
        if case["american"]:
            v = torch.maximum(v, sign * (m["S0"] * up[: n + 1] * dn[: n + 1].flip(0) - m["E"]))
    return dict(price=float(v[0]))


def _exact(case, m):
    if case["product"] == "american":
        return _exact_american(case, m)
    if case["product"] == "binomial":
        return _exact_binomial(case, m)
    if case["product"] == "lattice":
        return _exact_lattice(case, m)
    total = _simulated(case, m)
    disc, n = math.exp(-m["r"] * m["T"]), case["paths"]
    mean, var = _moments(total[:2], n)
    out = dict(price=disc * mean, std_err=disc * math.sqrt(var / n), mean=mean, variance=var)
    if case.get("control"):
        cmean, cvar = _moments(total[2:], n)
        out.update(control_price=disc * cmean, control_se=disc * math.sqrt(cvar / n))
    return {k: float(v) for k, v in out.items()}


def exact(case, seed):
    def typed(v):
        return {k: None if x is None else np.float64(x) for k, x in v.items()}

    if case["product"] == "mix":
        got = [_exact(c, _market(c, seed * 1000 + i)) for i, c in enumerate(_mix(case))]
        return {k: np.array([g[k] for g in got]) for k in ("price", "std_err", "mean", "variance")}
    return typed(_exact(case, _market(case, seed)))
