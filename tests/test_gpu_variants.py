"""Edges of the kernel variants that the host chooses between: the smallest
sizes, remainders of tiles and both sides of each rule, against the oracle."""
import ctypes as C
import math
import threading
import time

import numpy as np
import pytest

import _oracle as O
from parcompfin_amd import Engine, autotune, tune_reset

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


def close(got, want, tol):
    if not math.isfinite(want):  # a compensated sum over an infinity is not finite either (TwoSum makes it NaN)
        return not math.isfinite(got)
    return abs(got - want) <= tol * max(abs(want), 1e-300)


# ---------------------------------------------------------------- FP64 exponentials
@pytest.mark.parametrize("r,sigma,T", [(0.05, 0.0, 1.0), (0.05, 1e-9, 1.0), (0.03, 0.2, 1.0), (-0.4, 2.0, 1.5),
                                       (0.1, 30.0, 1.0), (340.0, 0.5, 2.0), (360.0, 0.5, 2.0), (-380.0, 0.1, 2.0)])
def test_eur_fp64_exponential_range(engine, r, sigma, T):
    """exp(mu + vol z) from tiny exponents to underflow and overflow."""
    say("mc_eur fp64 exponential range", r, sigma, T)
    N, pf = 1031, "put" if r < 0 or sigma > 10 else "call"
    vol, mu = sigma * math.sqrt(T), (r - 0.5 * sigma * sigma) * T
    se = C.c_double()
    want = O.lib().orc_philox_mc_eur(100, 90 if pf == "call" else 110, r, sigma, T, N, 1.0 if pf == "call" else -1.0,
                                     77, C.byref(se))
    got = engine.mc_eur(100, 90 if pf == "call" else 110, r, sigma, T, N, pf, seed=77, precision="fp64")
    # the exponent carries the normals' error (3.2e-15 at most) and a rounding of its own size
    assert close(got.price, want, 1e-12 + 1e-15 * (7 * vol + abs(mu)))


@pytest.mark.parametrize("M", [1, 3, 4, 9])
@pytest.mark.parametrize("scale", [0.97, 1.03, 20.0])
def test_asia_fp64_step_exponent_bound(engine, M, scale):
    """Both sides of the rule |mu| + 6.77 vol <= 0.3465 for a step."""
    T = 1.0
    dt = T / M
    # sigma for which |mu| + 6.77 vol = scale * 0.3465 at r = 0: a quadratic in sigma
    a, b, c = 0.5 * dt, 6.77 * math.sqrt(dt), -scale * 0.3465
    sigma = (-b + math.sqrt(b * b - 4 * a * c)) / (2 * a)
    say("mc_asia fp64 step bound", M, scale, sigma)
    N = 777
    se, geo = C.c_double(), C.c_double()
    want = O.lib().orc_philox_mc_asia(100, 95, 0.0, sigma, T, N, M, 1.0, 5, C.byref(se), C.byref(geo))
    got = engine.mc_asia(100, 95, 0.0, sigma, T, N, M, "call", seed=5, precision="fp64", control=True)
    assert close(got.price, want, 1e-12)
    assert close(got.control_price, geo.value, 1e-11)


# ---------------------------------------------------------------- binomial chain
@pytest.mark.parametrize("N", [16, 17, 18, 127, 128, 129, 130, 191, 255, 256, 257, 1025, 1026, 1027, 1153, 2177])
@pytest.mark.parametrize("pf", [1.0, -1.0])
def test_binom_chain_turn_edges(engine, N, pf):
    """Chains that end inside, at and after a turn of 128 values, a group of
    16 and a staged chunk of 1024."""
    say("binom chain turn edges", N, pf)
    want = O.lib().orc_binom_embar(100, 103, 0.05, 0.2, 1.0, N, pf, 1)
    got = engine.binom_embar(100, 103, 0.05, 0.2, 1.0, N, "call" if pf > 0 else "put", ref_exact=True)
    assert close(got.price, want, 1e-12)


# ---------------------------------------------------------------- lattice in one launch
@pytest.mark.parametrize("N", [1, 31, 32, 33, 64, 65, 127, 128, 129, 160, 161, 256, 257, 1025, 4129])
@pytest.mark.parametrize("american", [False, True])
@pytest.mark.parametrize("r,sigma,T", [(0.05, 0.2, 1.0), (-0.03, 0.45, 0.7)])
def test_lattice_one_launch_edges(engine, N, american, r, sigma, T):
    """Edges of the 32-level chunks, 32-node waves and 128-node blocks, and both
    signs of the rate (one and two corrections of the quotient), bit for bit."""
    for pf, E in ((1.0, 97.0), (-1.0, 104.0)):
        say("lattice one launch", N, american, r, pf)
        want = O.lib().orc_binom_vanilla(100, E, r, sigma, T, N, pf, 1 if american else 0)
        got = engine.binom_vanilla(100, E, r, sigma, T, N, "call" if pf > 0 else "put", american=american)
        assert got.price == want


@pytest.mark.parametrize("S0,E,sigma,N", [(1e-250, 1e-250, 0.3, 300), (100.0, -5.0, 0.3, 300), (100.0, 0.0, 0.3, 65),
                                          (100.0, 100.0, 12.0, 400), (100.0, 100.0, 60.0, 900), (1e200, 1e200, 0.2, 200),
                                          (100.0, 100.0, 1e-7, 64)])
@pytest.mark.parametrize("american", [False, True])
def test_lattice_outside_the_one_launch_bounds(engine, S0, E, sigma, N, american):
    """Prices, strikes and volatilities on both sides of the one-launch form's
    bounds: the reference's bits, or not finite where the reference is not."""
    for pf in (1.0, -1.0):
        say("lattice bounds", S0, E, sigma, N, american, pf)
        want = O.lib().orc_binom_vanilla(S0, E, 0.05, sigma, 1.0, N, pf, 1 if american else 0)
        got = engine.binom_vanilla(S0, E, 0.05, sigma, 1.0, N, "call" if pf > 0 else "put", american=american).price
        assert got == want or (math.isnan(got) and math.isnan(want))


@pytest.mark.parametrize("american", [False, True])
def test_lattice_finishes_after_a_wait_gave_up(engine, american):
    """A sweep whose waits give up is made by the launches per levels: the same
    bits, and the next sweep is one launch again."""
    lib = engine.lib
    for N, market in ((65, (100, 97, 0.05, 0.2, 1.0)), (1025, (100, 104, -0.03, 0.45, 0.7)),
                      (4129, (100, 97, 0.05, 0.2, 1.0)), (10007, (100, 104, 0.06, 0.3, 2.0))):
        say("lattice gives up", N, american)
        want = O.lib().orc_binom_vanilla(*market, N, -1.0, 1 if american else 0)
        lib.pcf_debug_lattice(1)
        try:
            r = engine.binom_vanilla(*market, N, "put", american=american)
        finally:
            lib.pcf_debug_lattice(0)
        assert r.price == want
        if N > 4000:  # 130 waves and more: some value is always on its way
            assert r.grid_blocks > 1
        r = engine.binom_vanilla(*market, N, "put", american=american)
        assert r.price == want and r.grid_blocks == 1


@pytest.mark.parametrize("american", [False, True])
def test_lattice_orders_of_blocks(engine, american):
    """Blocks placed by their XCDs' numbers and in the order of their own, from
    1 to 128 blocks and above, where neither is used: the oracle's bits."""
    for N in (129, 161, 1025, 1185, 4129, 16384, 16385, 16449):
        say("lattice orders of blocks", N, american)
        want = O.lib().orc_binom_vanilla(100, 97, 0.05, 0.2, 1.0, N, -1.0, 1 if american else 0)
        for bits in (0, 2):
            engine.lib.pcf_debug_lattice(bits)
            try:
                r = engine.binom_vanilla(100, 97, 0.05, 0.2, 1.0, N, "put", american=american)
            finally:
                engine.lib.pcf_debug_lattice(0)
            assert r.price == want and r.grid_blocks == 1


# ---------------------------------------------------------------- lattices beside other contexts' calls
def test_lattices_beside_other_contexts(engine):
    """Lattices share no order with other kinds of launch: beside American,
    Asian, chain and other lattice calls of four more contexts every result is
    the lone call's, and calls of another context end while a long lattice
    runs (90000 levels, about 7 ms; a chain of 1000 takes some 20 us).  The
    contexts' streams share the process's few hardware queues, so that is asked
    of the one that fares best."""
    lat = [lambda e, N=N, am=am: e.binom_vanilla(100, 104, 0.05, 0.2, 1.0, N, "put", american=am)
           for N, am in ((300, True), (4129, False), (10007, True), (50001, True))]
    mc = [lambda e: e.mc_amer(100, 100, 0.06, 0.2, 1.0, 1 << 14, 50, "put", seed=5),
          lambda e: e.mc_amer(100, 100, 0.06, 0.2, 1.0, 1 << 20, 50, "put", seed=6),
          lambda e: e.mc_asia(100, 100, 0.05, 0.25, 1.0, 1 << 21, 252, "call", seed=7),
          lambda e: e.binom_embar(100, 100, 0.05, 0.2, 1.0, 1000, "call", ref_exact=True)]
    say("lattices beside other contexts")
    jobs = [lat, lat[::-1], mc, mc[::-1], lat[2:] + mc[:2]]
    want = {f: f(engine).price for f in lat + mc}
    engines = [Engine(0) for _ in jobs]
    got = [[] for _ in jobs]

    def work(k):
        for _ in range(3):
            for f in jobs[k]:
                got[k].append((f, f(engines[k]).price))

    def run(targets):
        threads = [threading.Thread(target=t, args=a) for t, a in targets]
        for t in threads:
            t.start()
        for t in threads:
            t.join(timeout=100)
            assert not t.is_alive()

    run([(work, (k,)) for k in range(len(jobs))])
    for k, g in enumerate(got):
        assert len(g) == 3 * len(jobs[k]) and all(p == want[f] for f, p in g)

    long = lambda: engines[0].binom_vanilla(100, 104, 0.05, 0.2, 1.0, 90000, "put", american=True)  # noqa: E731
    assert long().grid_blocks == 1
    span, ends = [], [[] for _ in engines]

    def one():
        t = time.perf_counter()
        long()
        span.extend((t, time.perf_counter()))

    def many(k):
        while not span and len(ends[k]) < 10**5:
            mc[3](engines[k])
            ends[k].append(time.perf_counter())

    say("chains beside a long lattice")
    run([(many, (k,)) for k in range(1, len(engines))] + [(one, ())])
    inside = [sum(span[0] < t < span[1] for t in e) for e in ends]
    say("  chains that ended within", span[1] - span[0], "s:", inside)
    assert max(inside) >= 8
    for e in engines:
        e.close()


def test_lattices_and_persistent_launches_are_not_interleaved(engine):
    """A lattice and an American pricing that takes every CU, called over and
    over by two contexts: neither is placed among the blocks of the other, so
    every sweep is one launch (its waits would give up after 20 ms)."""
    amer = lambda e: e.mc_amer(100, 100, 0.06, 0.2, 1.0, 1 << 20, 20, "put", seed=6)  # noqa: E731
    lat = lambda e, N: e.binom_vanilla(100, 104, 0.05, 0.2, 1.0, N, "put", american=True)  # noqa: E731
    say("lattices and persistent launches")
    want = {N: lat(engine, N).price for N in (300, 1000)}
    price = amer(engine).price
    engines = [Engine(0), Engine(0)]
    bad, count, end = [], [0, 0], time.perf_counter() + 1.5

    def lattices():
        while time.perf_counter() < end:
            for N in want:
                r = lat(engines[0], N)
                count[0] += 1
                if r.price != want[N] or r.grid_blocks != 1:
                    bad.append((N, r.price, r.grid_blocks))

    def americans():
        while time.perf_counter() < end:
            r = amer(engines[1])
            count[1] += 1
            if r.price != price:
                bad.append(("american", r.price))

    threads = [threading.Thread(target=f) for f in (lattices, americans)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    say("  lattices and Americans", count, "not as alone", bad)
    assert min(count) > 100 and not bad
    for e in engines:
        e.close()


# ---------------------------------------------------------------- basket, one correlation
@pytest.mark.parametrize("d", [1, 2, 3, 4, 5, 6, 7, 8, 9, 13, 15, 33, 62, 63, 64])
@pytest.mark.parametrize("precision", ["fp32k", "fp64"])
@pytest.mark.parametrize("rho", [0.0, 0.35, 0.95])
def test_basket_one_correlation_equals_general_kernel(engine, d, precision, rho):
    """The prefix form forms each B_i from the same products in the same order
    as the general kernel: the same bits (d < 16 or beyond the MFMA range)."""
    sig = np.random.default_rng(d).uniform(0.1, 0.5, size=d)
    N = 1003
    kw = dict(sigmas=sig, seed=d + 1, precision=precision)
    say("basket one correlation", d, precision, rho)
    a = engine.mc_eur_multi(100, 100, 0.05, 0.2, 1.3, N, "put", d, rho, **kw)
    b = engine.mc_eur_multi(100, 100, 0.05, 0.2, 1.3, N, "put", d, rho, kernel_variant=1, **kw)
    assert (a.price, a.std_err, a.variance) == (b.price, b.std_err, b.variance)


def test_basket_one_correlation_by_matrix(engine):
    """An equicorrelation given as a matrix prices as the scalar does, and a
    matrix with one entry pair changed does not take the prefix form."""
    d, N = 6, 4001
    C = np.full((d, d), 0.4)
    np.fill_diagonal(C, 1.0)
    kw = dict(seed=3, precision="fp64")
    a = engine.mc_eur_multi(100, 95, 0.03, 0.3, 1.0, N, "call", d, 0.4, **kw)
    b = engine.mc_eur_multi(100, 95, 0.03, 0.3, 1.0, N, "call", d, 0.0, corr=C, **kw)
    assert a.price == b.price
    C[5, 1] = C[1, 5] = 0.1
    c = engine.mc_eur_multi(100, 95, 0.03, 0.3, 1.0, N, "call", d, 0.0, corr=C, **kw)
    z = O.philox_normals(3, 4, 0, N, d)
    L = np.linalg.cholesky(C)
    v = (100 / d * np.exp((0.03 - 0.045) + 0.3 * (z @ L.T))).sum(1)
    want = math.exp(-0.03) * np.maximum(v - 95, 0).mean()
    assert close(c.price, want, 1e-12)


def test_basket_tuned_shapes_by_kernel(engine):
    """A tuned shape is used by the kernel that it was measured with: the prefix
    form, the general kernel and the MFMA kernel at two blocks of assets."""
    say("basket tuned shapes")
    N = 1 << 14
    corr = np.full((20, 20), 0.3)
    np.fill_diagonal(corr, 1.0)
    corr[1, 2] = corr[2, 1] = 0.1  # no prefix form

    def shape(d, general):
        kw = dict(corr=corr[:d, :d]) if general else {}
        r = engine.mc_eur_multi(100, 100, 0.05, 0.2, 1.0, N, "call", d, 0.3, seed=2, **kw)
        return r.block_size, r.grid_blocks

    calls = {6: (8, False), 0: (8, True), 1: (20, True), "one block": (16, True)}
    tune_reset()
    builtin = {k: shape(*c) for k, c in calls.items()}
    try:
        found = {e["mode"]: e for e in autotune(engine, kinds=("basket",), max_log2_paths=14)}
        assert sorted(found) == [0, 1, 6]
        for k, c in calls.items():
            B, ipt = (found[k]["block_size"], found[k]["items_per_thread"]) if k in found else (0, 0)
            items, per = ((N + 15) // 16, B // 64) if k == 1 else (N, B)
            assert shape(*c) == ((B, -(-items // (per * ipt))) if B else builtin[k])
    finally:
        tune_reset()


# ---------------------------------------------------------------- Asian, FP32 blocks of four steps
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 7, 8, 63, 252])
@pytest.mark.parametrize("S0,E,r,sigma,T", [(100, 103, 0.05, 0.25, 1.0), (3.7e-4, 3.6e-4, 0.02, 0.6, 2.0),
                                            (100, 100, 0.05, 0.0, 1.0)])
def test_asia_fp32_block_of_steps(engine, M, S0, E, r, sigma, T):
    """FP32 against FP64 on the same paths, with every remainder of four steps."""
    N = 5003
    say("mc_asia fp32 blocks", M, S0, sigma)
    kw = dict(seed=21, control=True)
    a = engine.mc_asia(S0, E, r, sigma, T, N, M, "call", **kw)
    b = engine.mc_asia(S0, E, r, sigma, T, N, M, "call", precision="fp64", **kw)
    # a path's average is off by a few FP32 roundings (exponentials and products
    # of M / 4 blocks, at most 2^-22 each); the payoff's share of it is S0
    tol = math.exp(-r * T) * S0 * (2 + M / 4) * 2.0**-22
    assert abs(a.price - b.price) <= tol
    assert abs(a.control_price - b.control_price) <= tol


# ---------------------------------------------------------------- American, the sweep a date ahead
@pytest.mark.parametrize("N,M,block,pairs", [
    (2, 2, 64, 1), (128, 3, 64, 1), (130, 1, 64, 1), (1000, 2, 64, 1),         # one block; fewer rows than run ahead
    (2048, 4, 64, 2), (2 * 64 * 9 - 2, 5, 64, 1), (2 * 64 * 31, 7, 64, 1),     # all blocks poll each other
    (2 * 64 * 32, 9, 64, 1), (2 * 64 * 32 + 2, 9, 64, 1),                      # last and first grid of each all-reduce
    (2 * 128 * 2 * 65 - 6, 12, 128, 2), (2 * 64 * 255, 6, 64, 1), (2 * 192 * 256, 6, 192, 1),
    (2 * 1024 * 2 * 40, 5, 1024, 2)])
@pytest.mark.parametrize("precision", ["fp32k", "fp64"])
def test_amer_ahead_sweep_matches_graph_form(engine, N, M, block, pairs, precision):
    """The same paths and regressions as the per-date launches; only the order
    of the FP64 sums differs, which moves a coefficient by far less than the
    gap between a path's payoff and its continuation value: the prices agree to
    the rounding of a sum of N terms."""
    say("mc_amer ahead", N, M, block, pairs, precision)
    kw = dict(seed=17, precision=precision)
    g = engine.mc_amer(100, 100, 0.06, 0.2, 1.0, N, M, "put", kernel_variant=1, **kw)
    for _ in range(2):  # the second launch starts from the words the first left
        p = engine.mc_amer(100, 100, 0.06, 0.2, 1.0, N, M, "put", kernel_variant=2, block_size=block,
                           items_per_thread=pairs, **kw)
        assert close(p.price, g.price, 1e-12)
        assert close(p.std_err, g.std_err, 1e-9)
        assert close(p.control_price, g.control_price, 1e-12)


@pytest.mark.parametrize("N,M,block,pairs,ref", [
    (2 * 64 * 3, 4, 64, 3, False), (2 * 64 * 5 * 31, 3, 64, 5, False), (2 * 64 * 8 * 40 - 2, 7, 64, 8, False),
    (2 * 128 * 6 * 200, 5, 128, 6, False), (130, 6, 64, 1, True), (2 * 64 * 33, 5, 64, 1, True),
    (2 * 64 * 2 * 255, 5, 64, 2, True), (2 * 64 * 3 * 20, 5, 64, 3, True)])
def test_amer_tree_sums_at_other_budgets(engine, N, M, block, pairs, ref):
    """3 to 8 pairs per thread and the reference-exact mode, whose sums take the
    same words: as the per-date launches."""
    say("mc_amer tree", N, M, block, pairs, ref)
    kw = dict(seed=19, precision="fp64", ref_exact=ref)
    g = engine.mc_amer(100, 100, 0.06, 0.2, 1.0, N, M, "put", kernel_variant=1, **kw)
    for _ in range(2):
        p = engine.mc_amer(100, 100, 0.06, 0.2, 1.0, N, M, "put", kernel_variant=2, block_size=block,
                           items_per_thread=pairs, **kw)
        assert close(p.price, g.price, 1e-12)
        assert close(p.control_price, g.control_price, 1e-12)


# ---------------------------------------------------------------- basket, blocks of 16 assets
@pytest.mark.parametrize("d", [13, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64])
@pytest.mark.parametrize("precision", ["fp32k", "fp64"])
@pytest.mark.parametrize("full", [False, True])
def test_basket_blocks_match_general_kernel(engine, d, precision, full):
    """Every count of asset blocks, both factors (a singular matrix takes the
    eigenvectors'), tiles with missing paths: as the one-path-per-lane kernel,
    which forms the same exponents with the terms in another order."""
    rng = np.random.default_rng(d)
    f = rng.normal(size=(d, 2 if full else d))
    C = f @ f.T + (0.0 if full else 0.5) * np.eye(d)
    s = np.sqrt(np.diag(C))
    C = C / np.outer(s, s)
    C = 0.5 * (C + C.T)
    np.fill_diagonal(C, 1.0)
    sig = rng.uniform(0.1, 0.5, size=d)
    say("basket blocks", d, precision, full)
    for N in (1, 1003):
        kw = dict(sigmas=sig, corr=C, seed=d, precision=precision)
        a = engine.mc_eur_multi(100, 90, 0.05, 0.2, 1.3, N, "call", d, 0.0, **kw)
        b = engine.mc_eur_multi(100, 90, 0.05, 0.2, 1.3, N, "call", d, 0.0, kernel_variant=1, **kw)
        assert a.lsm_fallback == b.lsm_fallback  # the same factor
        # an exponent is a sum of at most d terms c1 L z of size below 0.6 * 6, off
        # by d roundings of it in each kernel; the basket is off by as much of
        # itself, plus d roundings of its own sum, and so is a mean of payoffs
        eps = 2.0**-24 if precision == "fp32k" else 2.0**-53
        assert abs(a.price - b.price) <= 2 * d * 4.6 * eps * 200
