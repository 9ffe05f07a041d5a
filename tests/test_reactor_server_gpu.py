"""The reactor request server on the GPU: every scheme against the oracle's
reactor on the same request (fixed steps to 1e-9, adaptive ROK4E to its
tolerance), each result identical bit for bit alone and in a mix of two
hundred concurrent requests, the two stepping kernels against each other on
every scheme and kind of mechanism, and admission by slot budget (a three-slot
server queues the rest and returns the same results).  The explicit SSP-RK3
runs at dt = 2e-10 s: at 1e-9 s it sits at its stability limit through the
ignition of the 1400 K case, where the oracle itself moves by 4e-6 for a
1e-15 change of the initial temperature."""
import ctypes as C
import time

import numpy as np
import pytest

from corefl_amd import ReactorServer, _abi, h2_air_mass_fractions, load_air5_tables, load_tables
from oracle import PD, h2_tables, load

pytestmark = pytest.mark.gpu

R_U = 8314.462618
P_ATM = 101325.0


@pytest.fixture(scope="module")
def tables():
    return load_tables()


@pytest.fixture(scope="module")
def oc():
    return h2_tables()


def oracle_reactor(oc, T0, p0, y, scheme, dt, t_end, adaptive=1, rtol=1e-4, atol=1e-8):
    mw = np.array(oc.mw[:9])
    rho = p0 / (R_U * (y / mw).sum() * T0)
    T = C.c_double(T0)
    yy = np.ascontiguousarray(np.concatenate([y, np.zeros(11)]))
    L = load()
    if scheme == 1:
        rej = C.c_long(0)
        n = L.oc_cv_reactor_rok4e(C.byref(oc), rho, C.byref(T), yy.ctypes.data_as(PD), dt, t_end, adaptive, rtol,
                                  atol, C.byref(rej))
    else:
        n = L.oc_cv_reactor_ex(C.byref(oc), rho, C.byref(T), yy.ctypes.data_as(PD), dt, t_end, scheme, 1)
    return T.value, yy[:9].copy(), n


CASES = [(1100.0, 2 * P_ATM, 1.0), (1400.0, 5 * P_ATM, 0.6), (950.0, 1 * P_ATM, 1.8)]


@pytest.mark.parametrize("scheme,dt,t_end", [(1, 2e-8, 1e-4), (0, 1e-8, 1e-4), (3, 2e-10, 2e-6)])
def test_fixed_step_parity(tables, oc, scheme, dt, t_end):
    mw = np.array(tables.mw[:9])
    srv = ReactorServer(tables, budget_bytes=1 << 20, steps_per_launch=4096)
    tickets = []
    for T0, p0, phi in CASES:
        y = h2_air_mass_fractions(phi, mw)
        tickets.append(srv.submit(T0, p0, y, t_end, dt, scheme=scheme, adaptive=False, conserve_mass=True))
    print(f"scheme {scheme} dt {dt} t_end {t_end}", flush=True)
    res = srv.run_until_done(tickets)
    for (T0, p0, phi), t in zip(CASES, tickets):
        r = res[t]
        To, yo, n = oracle_reactor(oc, T0, p0, h2_air_mass_fractions(phi, mw), scheme, dt, t_end, adaptive=0)
        assert r["steps"] == n
        assert abs(r["temperature"] - To) <= 1e-9 * To, (r["temperature"], To)
        assert np.abs(r["y"] - yo).max() <= 1e-9 * np.abs(yo).max()
    srv.close()


def test_adaptive_rok4e_parity(tables, oc):
    mw = np.array(tables.mw[:9])
    srv = ReactorServer(tables, budget_bytes=1 << 20, steps_per_launch=512)
    tickets = [srv.submit(T0, p0, h2_air_mass_fractions(phi, mw), 2e-3, 1e-8, rtol=1e-6, atol=1e-10)
               for T0, p0, phi in CASES]
    res = srv.run_until_done(tickets)
    for (T0, p0, phi), t in zip(CASES, tickets):
        r = res[t]
        To, yo, n = oracle_reactor(oc, T0, p0, h2_air_mass_fractions(phi, mw), 1, 1e-8, 2e-3, rtol=1e-6, atol=1e-10)
        # the step sequences may part where an error estimate sits at 1 to rounding;
        # both integrate to the tolerance
        assert abs(r["temperature"] - To) <= 1e-5 * To, (r["temperature"], To)
        assert np.abs(r["y"] - yo).max() <= 1e-4 * np.abs(yo).max()
        assert abs(r["steps"] - n) <= 0.05 * n
    srv.close()


def random_requests(mw, n, seed):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        T0, p0, phi = rng.uniform(900, 1600), rng.uniform(1, 10) * P_ATM, rng.uniform(0.5, 2.0)
        out.append((T0, p0, h2_air_mass_fractions(phi, mw)))
    return out


def test_alone_and_in_the_mix_are_identical(tables):
    mw = np.array(tables.mw[:9])
    reqs = random_requests(mw, 200, seed=5)
    pick = [0, 57, 199]
    alone = {}
    for i in pick:
        srv = ReactorServer(tables, budget_bytes=1 << 20, steps_per_launch=256)
        T0, p0, y = reqs[i]
        t = srv.submit(T0, p0, y, 5e-4, 1e-8)
        alone[i] = srv.run_until_done([t])[t]
        srv.close()
    srv = ReactorServer(tables, budget_bytes=8 << 20, steps_per_launch=256)
    # requests arrive in two waves: the second joins while the first is in flight
    tickets = [srv.submit(T0, p0, y, 5e-4, 1e-8) for T0, p0, y in reqs[:100]]
    srv.progress()
    tickets += [srv.submit(T0, p0, y, 5e-4, 1e-8) for T0, p0, y in reqs[100:]]
    res = srv.run_until_done(tickets)
    assert len(res) == 200
    for i in pick:
        r = res[tickets[i]]
        assert r["temperature"] == alone[i]["temperature"]
        assert np.array_equal(r["y"], alone[i]["y"])
        assert r["steps"] == alone[i]["steps"] and r["rejected"] == alone[i]["rejected"]
    srv.close()


def test_budget_admission(tables):
    mw = np.array(tables.mw[:9])
    reqs = random_requests(mw, 20, seed=6)
    small = ReactorServer(tables, budget_bytes=4 * 400, steps_per_launch=128)
    assert 1 <= small.capacity <= 8
    big = ReactorServer(tables, budget_bytes=8 << 20, steps_per_launch=128)
    ts = [small.submit(T0, p0, y, 2e-4, 1e-8) for T0, p0, y in reqs]
    tb = [big.submit(T0, p0, y, 2e-4, 1e-8) for T0, p0, y in reqs]
    rs, rb = small.run_until_done(ts), big.run_until_done(tb)
    for a, b in zip(ts, tb):
        assert rs[a]["temperature"] == rb[b]["temperature"]
        assert np.array_equal(rs[a]["y"], rb[b]["y"])
    small.close()
    big.close()


# scheme, adaptive, conserve_mass, dt, steps (0: as many as t_end takes), a third of the requests capped at
KERNEL_CASES = {
    "rok4e": (1, 1, 0, 1e-8, 0, 0), "rok4e_capped": (1, 1, 0, 1e-8, 0, 5), "rok4e_fixed": (1, 0, 0, 1e-8, 24, 0),
    "point_implicit": (0, 0, 0, 1e-9, 24, 0), "point_implicit_conserving": (0, 0, 1, 1e-9, 24, 0),
    "rk3": (3, 0, 0, 2e-10, 24, 0),
}


def five_species_h2():
    """The H2, H, O2, O, OH part of the H2 mechanism (NASA-7)."""
    t = load_tables()
    kept = [r for r in range(t.n_reac) if not any(t.stoi_f[r][l] or t.stoi_b[r][l] for l in range(5, 9))]
    for k, r in enumerate(kept):
        for f in ("reac_type", "rev_type", "order", "A", "b", "Ea", "A2", "b2", "Ea2", "troe_alpha", "troe_t1",
                  "troe_t2", "troe_t3"):
            getattr(t, f)[k] = getattr(t, f)[r]
        for f in ("stoi_f", "stoi_b", "third_body"):
            getattr(t, f)[k][:] = list(getattr(t, f)[r])
    t.n_reac, t.n_spec = len(kept), 5
    return t


def unusual_orders():
    """The 5-species air mechanism with a reaction inhibited by N2 and others of its third and fifth order, their
    rates unchanged where its concentration is 3e-6."""
    t = load_air5_tables(False)
    free = [r for r in range(t.n_reac) if t.stoi_f[r][0] == t.stoi_b[r][0] == 0]
    for r, order in zip(free, (-1, 3, 5)):
        t.stoi_f[r][0] = t.stoi_b[r][0] = order
        t.A[r] *= 3e-6 ** -order
    return t


MECHANISMS = {"h2": load_tables, "h2_5sp": five_species_h2, "air_nasa9": lambda: load_air5_tables(False),
              "air_orders": unusual_orders}


def kernel_requests(mech, tables, n, case):
    scheme, adaptive, conserve, dt, steps, cap = case
    rng = np.random.default_rng(11)
    mw = np.array(tables.mw[:9])
    req = (_abi.ReactorRequest * n)()
    for i, q in enumerate(req):
        if mech.startswith("h2"):
            y = h2_air_mass_fractions(rng.uniform(0.5, 2.0), mw if mech == "h2" else np.array(load_tables().mw[:9]))
            y = y[:tables.n_spec] / y[:tables.n_spec].sum()
            q.temperature, q.pressure = rng.uniform(900.0, 1600.0), rng.uniform(1.0, 10.0) * P_ATM
        else:
            d = rng.uniform(0.0, 0.3)
            y = np.array([0.767 * (1 - d), 0.233 * (1 - d), 0.0, 0.767 * d, 0.233 * d])
            q.temperature, q.pressure = rng.uniform(3000.0, 8000.0), rng.uniform(0.1, 1.0) * P_ATM
        q.y[:len(y)] = [float(v) for v in y]
        q.t_end, q.dt = (steps - 0.5) * dt if steps else 2e-6, dt
        q.scheme, q.adaptive, q.conserve_mass, q.rtol, q.atol = scheme, adaptive, conserve, 1e-4, 1e-8
        q.max_steps = cap if i % 3 == 0 else 0
    return req


def serve_all(tables, req):
    """Results of every request in order, and the seconds of the stepping."""
    n = len(req)
    srv = ReactorServer(tables, budget_bytes=512 * (n + 64), steps_per_launch=32)
    assert srv.capacity >= n
    for q in req:
        assert srv.lib.corefl_serve_submit(srv.h, C.byref(q)) >= 0
    t0 = time.perf_counter()
    while srv.progress():
        pass
    took = time.perf_counter() - t0
    tickets, res = (C.c_long * n)(), (_abi.ReactorResult * n)()
    assert srv.lib.corefl_serve_drain(srv.h, tickets, res, n) == n
    srv.close()
    return np.ctypeslib.as_array(res)[np.argsort(np.ctypeslib.as_array(tickets))].copy(), took


@pytest.mark.parametrize("mech,case", [(m, c) for m in MECHANISMS for c in KERNEL_CASES
                                       if m != "air_orders" or KERNEL_CASES[c][4]])
def test_result_does_not_depend_on_the_kernel_the_load_picks(mech, case):
    """16,500 requests in flight are stepped with a lane each, 2,000 with a wave each, whatever the mechanism
    (the adaptive ones pass from the first to the second as they finish): every result is the same bit for bit,
    failures at the step cap included."""
    tables = MECHANISMS[mech]()
    n, part = 16500, 2000
    print(f"{mech} {case}: {n} reactors with a lane each", flush=True)
    req = kernel_requests(mech, tables, n, KERNEL_CASES[case])
    lanes, _ = serve_all(tables, req)
    for lo in (0, n - part):
        waves, _ = serve_all(tables, (_abi.ReactorRequest * part)(*req[lo:lo + part]))
        for f in ("temperature", "pressure", "time", "y", "steps", "rejected", "status", "reason"):
            assert np.array_equal(lanes[f][lo:lo + part], waves[f]), f
    failed = (lanes["status"] != 0).sum()
    assert failed > 0 if KERNEL_CASES[case][5] else failed == 0


def test_fewer_reactors_take_no_longer():
    """A step of 12,000 reactors does not take longer than one of 17,000: the switch between the kernels lies
    where their times cross (with a wave each these take 1.4 times as long)."""
    tables = load_air5_tables(False)
    case = KERNEL_CASES["rok4e_fixed"][:4] + (160, 0)
    few, many = (kernel_requests("air_nasa9", tables, n, case) for n in (12000, 17000))
    best = [min(t) for t in zip(*((serve_all(tables, few)[1], serve_all(tables, many)[1]) for _ in range(3)))]
    assert best[0] <= 1.05 * best[1], best
