"""Reaction orders outside the usual 1 and 2: tables handed in through the C ABI may hold any integer (an
inhibiting species has a negative one), and every chemistry kernel forms c^order as the oracle does."""
import ctypes as C

import numpy as np
import pytest

from corefl_amd import ReactorServer, Solver, _abi, air5_box_case, h2_air_mass_fractions, load_air5_tables, load_tables
from oracle import PD, Oracle, air5_tables, h2_tables, load

pytestmark = pytest.mark.gpu

# one operator, FP64 sums of at most 27 terms; an order e multiplies the rounding of a concentration by e
STAGE_TOL = 1e-11
R_U = 8314.462618
P_ATM = 101325.0


def set_order(tables, r, species, order, c_ref):
    """Species enters reaction r with this order on both sides (no net change), its rate unchanged at c_ref."""
    for t in tables:
        t.stoi_f[r][species] = t.stoi_b[r][species] = order
        t.A[r] *= c_ref ** -order


@pytest.mark.parametrize("two_temperature", [False, True])
@pytest.mark.parametrize("order", [-3, -1, 3, 4, 7])
def test_chemistry_operator(order, two_temperature):
    tables, ref = load_air5_tables(two_temperature), air5_tables(two_temperature=two_temperature)
    for r in (0, 7, 16):  # a dissociation and two exchanges
        set_order((tables, ref), r, 0, order, 2e-7)  # N2, present everywhere
    case = air5_box_case(17, 11, 9, seed=21, tables=tables, two_temperature=two_temperature)
    s = Solver(case.run, tables)
    s.add_block(case)
    o = Oracle(case, ref)
    s.initialize()
    o.initialize()
    s.op(_abi.OP_ZERO_DQ)
    o.op("zero_dq")
    s.op(_abi.OP_CHEMISTRY)
    o.op("chemistry")
    got, want = s.download(0, _abi.F_DQ), o.a["dq"]
    s.close()
    got, want = got.reshape(got.shape[0], -1)[5:], want.reshape(want.shape[0], -1)[5:]
    den = np.abs(want).max(axis=1)
    # N2 enters its creation and destruction sums with `order` times the reaction's two rates, which cancel there
    den[0] = max(den[0], abs(order) * den.max())
    err = np.abs(got - want).max(axis=1) / den
    assert np.all(err <= STAGE_TOL), err


@pytest.mark.parametrize("order", [-2, -1, 3, 5])
def test_reactor(order):
    """Served reactors (fixed point-implicit steps) against the oracle's."""
    tables, ref = load_tables(), h2_tables()
    for r in (0, 5):
        set_order((tables, ref), r, 8, order, 2e-5)  # N2
    mw = np.array(tables.mw[:9])
    srv = ReactorServer(tables, budget_bytes=1 << 20, steps_per_launch=4096)
    cases = [(1100.0, 2 * P_ATM, 1.0), (1400.0, 5 * P_ATM, 0.6)]
    tickets = [srv.submit(T0, p0, h2_air_mass_fractions(phi, mw), 2e-5, 1e-8, scheme=0, adaptive=False,
                          conserve_mass=True) for T0, p0, phi in cases]
    res = srv.run_until_done(tickets)
    srv.close()
    for (T0, p0, phi), t in zip(cases, tickets):
        y = h2_air_mass_fractions(phi, mw)
        T, yy = C.c_double(T0), np.ascontiguousarray(np.concatenate([y, np.zeros(11)]))
        load().oc_cv_reactor_ex(C.byref(ref), p0 / (R_U * (y / mw).sum() * T0), C.byref(T), yy.ctypes.data_as(PD),
                                1e-8, 2e-5, 0, 1)
        r = res[t]
        assert r["status"] == 0 and abs(r["temperature"] - T.value) <= 1e-9 * T.value, (r["temperature"], T.value)
        assert np.abs(r["y"] - yy[:9]).max() <= 1e-9 * yy[:9].max()


@pytest.mark.parametrize("scheme", [0, 1])
@pytest.mark.parametrize("what", ["order", "net"])
def test_reactor_with_orders_beyond_a_byte(what, scheme):
    """An irreversible reaction of order 300 (its rate underflows) and a reaction of rate 0 that makes 130 of a
    species leave the reactor as it is without them."""
    mw = np.array(load_tables().mw[:9])
    out = []
    for changed in (False, True):
        tables = load_tables()
        r = 3
        tables.A[r] = 0.0
        tables.b[r] = tables.Ea[r] = 0.0
        if what == "order":
            tables.reac_type[r] = 0
        if changed and what == "order":
            tables.A[r] = 1e300
            tables.stoi_f[r][8] = tables.stoi_b[r][8] = 300
        if changed and what == "net":
            tables.stoi_b[r][8] = 130
        srv = ReactorServer(tables, budget_bytes=1 << 20, steps_per_launch=4096)
        t = srv.submit(1200.0, 5 * P_ATM, h2_air_mass_fractions(1.0, mw), 2e-5, 1e-8, scheme=scheme, adaptive=False)
        out.append(srv.run_until_done([t])[t])
        srv.close()
    assert out[0]["status"] == out[1]["status"] == 0
    assert out[0]["temperature"] == out[1]["temperature"] and np.array_equal(out[0]["y"], out[1]["y"])
