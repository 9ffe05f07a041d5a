"""Parity of the boundary conditions on the GPU with the oracle: a curvilinear
channel with an inflow (supersonic, or subsonic with the characteristic
treatment), an outflow, an isothermal and an adiabatic wall and two symmetry
planes, for the Air perfect gas (WENO5, inviscid) and the 9-species mixture
(WENO7, 8th-order viscous terms, chemistry), and two-temperature 5-species air (WENO5,
2nd-order viscous terms with the E_ve terms, chemistry, V-T relaxation; inflow Tve,
wall Tve from the wall temperature or the interior)."""
import numpy as np
import pytest

from corefl_amd import CoreflError, Solver, _abi, air5_box_case, channel_case, load_air5_tables, load_tables
from oracle import Oracle, air5_tables

pytestmark = pytest.mark.gpu

STAGE_TOL = 1e-11
LONG_TOL = 1e-9
FIELDS = [("cv", _abi.F_CV), ("bv", _abi.F_BV), ("sv", _abi.F_SV)]


def normwise(a, b, vector=None):
    a = a.reshape(a.shape[0], -1)
    b = b.reshape(b.shape[0], -1)
    den = np.abs(b).max(axis=1)
    if vector is not None:
        den[list(vector)] = den[list(vector)].max()
    den = np.maximum(den, 1e-300)
    return np.abs(a - b).max(axis=1) / den


def check(s, o, case, tol, info):
    fields = FIELDS + ([("tve", _abi.F_TVE)] if case.run.get("two_temperature") else [])
    for name, fid in fields:
        if name == "sv" and not case.run["n_scalar"]:
            continue
        ref = o.a[name] if o.a[name].ndim == 4 else o.a[name][None]
        err = normwise(s.download(0, fid), ref, vector=(1, 2, 3) if name in ("cv", "bv") else None)
        assert np.all(err <= tol), f"{name}{info}: {err} > {tol}"


@pytest.fixture(scope="module")
def tables():
    return load_tables()


@pytest.mark.parametrize("physics", ["air", "h2", "air5"])
@pytest.mark.parametrize("subsonic", [False, True])
def test_channel_boundary_parity(tables, h2_oracle_tables, physics, subsonic):
    case = channel_case(24, 16, 12, physics=physics, subsonic=subsonic, seed=3)
    print(f"channel {physics} subsonic={subsonic}", flush=True)
    mix = case.run["mixture"]
    if physics == "air5":
        gpu_tables, oc_tables = load_air5_tables(True), air5_tables(True)
    else:
        gpu_tables, oc_tables = tables, h2_oracle_tables
    s = Solver(case.run, gpu_tables if mix else None)
    s.add_block(case)
    o = Oracle(case, oc_tables if mix else None)
    s.initialize()
    o.initialize()
    check(s, o, case, STAGE_TOL, " after initialize")
    dt = o.cfl_dt() if not mix else 0.5 * o.cfl_dt()
    s.op(_abi.OP_COPY_QN)
    o.op("copy_qn")
    for rk in range(3):
        s.stage(rk, dt)
        o.stage(rk, dt)
        check(s, o, case, STAGE_TOL, f" after stage {rk}")
    for _ in range(10):
        if mix:
            s.step(dt)
            o.step(dt, fixed=True)
        else:
            dg, do = s.step(), o.step(fixed=False)
            assert abs(dg - do) <= 1e-12 * do
    check(s, o, case, LONG_TOL, " after 11 steps")
    s.close()


@pytest.mark.parametrize("two_temperature", [False, True])
@pytest.mark.parametrize("low,high", [(2, 21), (21, 2), (2, 3)])
def test_k_walls_of_a_plane(two_temperature, low, high):
    """Walls on the k faces of a one-plane block: their reference nodes are ghosts, and the labels of the other
    faces beside them are those of the plane."""
    tb, oc = load_air5_tables(two_temperature), air5_tables(two_temperature)
    case = air5_box_case(19, 13, 1, seed=6, tables=tb, two_temperature=two_temperature)
    end = (case.mx - 1, case.my - 1, 0)
    case.boundaries = list(case.boundaries) + [(2, -1, low, (0, 0, 0), end), (2, 1, high, (0, 0, 0), end)]
    case.conditions = [dict(label=2, kind=2, thermal_type=0, wall_temperature=1500.0),
                       dict(label=21, kind=2, thermal_type=1), dict(label=3, kind=3)]
    s = Solver(case.run, tb)
    s.add_block(case)
    o = Oracle(case, oc)
    s.initialize()
    o.initialize()
    check(s, o, case, STAGE_TOL, " after initialize")
    s.op(_abi.OP_BC)
    o.op("bc")
    check(s, o, case, STAGE_TOL, " after the boundary conditions")
    s.close()


def test_unregistered_inflow_label_is_rejected(tables):
    case = channel_case(24, 16, 12, physics="air")
    case.conditions = [c for c in case.conditions if c["kind"] != 5]
    s = Solver(case.run, None)
    with pytest.raises(CoreflError, match="label 5"):
        s.add_block(case)
    s.close()
