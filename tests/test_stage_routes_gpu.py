"""What a step does differently from its operators one by one, against those operators bit for bit: on a 2-D
block the ghost planes are completed only where a stage reads them, the x sweep stores dq instead of adding to a
cleared one (or the viscous derivative stores it, in each of its splits), the recorded step exchanges independent
inner faces in one launch; then outflow faces in numbers above one launch's list, and two-temperature tables
outside the usual ones against the oracle."""
import numpy as np
import pytest

from corefl_amd import (Solver, _abi, air5_box_case, channel_case, load_air5_tables, load_tables, multiblock_case,
                        reacting_box_case, sod_case, square_ogrid_case)
from corefl_amd.cases import Case
from oracle import Oracle, air5_tables

pytestmark = pytest.mark.gpu

# one operator, FP64 sums of at most 27 terms against the same sums in another order
STAGE_TOL = 1e-11
STATE = (_abi.F_CV, _abi.F_BV, _abi.F_SV)
OPS = [_abi.OP_ZERO_DQ, _abi.OP_VISCOUS, _abi.OP_CHEMISTRY, _abi.OP_INVISCID_X, _abi.OP_INVISCID_Y,
       _abi.OP_INVISCID_Z, _abi.OP_UPDATE_RK, _abi.OP_LIMIT_FLOW, _abi.OP_BC, _abi.OP_HALO, _abi.OP_K_GRADIENT,
       _abi.OP_PROPERTIES]


def body_2d(mx, my):
    t = load_air5_tables(True)
    return [square_ogrid_case(mx, my, tables=t)], t, STATE + (_abi.F_TVE, _abi.F_GAMMA, _abi.F_KAPPA_VE)


def plane_8th(mx, my):
    t = load_air5_tables(True)
    c = air5_box_case(mx, my, 1, seed=3, tables=t, two_temperature=True, ngg=4)
    c.run.update(viscous_order=8, inviscid_scheme=72)
    return [c], t, STATE + (_abi.F_TVE,)


def plane_one_temperature(mx, my):
    t = load_air5_tables(False)
    return [air5_box_case(mx, my, 1, seed=4, tables=t)], t, STATE + (_abi.F_GAMMA, _abi.F_ACOUSTIC)


def plane_k_faces(low, high):
    """A plane with boundary faces on its k axis: those read the ghost planes in every stage."""
    def make(mx, my):
        t = load_air5_tables(False)
        c = air5_box_case(mx, my, 1, seed=6, tables=t)
        end = (mx - 1, my - 1, 0)
        c.boundaries = list(c.boundaries) + [(2, -1, low, (0, 0, 0), end), (2, 1, high, (0, 0, 0), end)]
        c.conditions = [dict(label=2, kind=2, thermal_type=0, wall_temperature=1500.0),
                        dict(label=21, kind=2, thermal_type=1), dict(label=3, kind=3)]
        return [c], t, STATE
    return make


def joined_planes(physics):
    """A 2-D channel cut into 2 x 2 one-plane blocks joined at inner faces (their common lines belong to both)."""
    def make(mx, my):
        tt = physics == "air5"
        t = None if physics == "air" else load_air5_tables(True) if tt else load_tables()
        w = channel_case(mx, my, 1, physics=physics, seed=8)
        g, ci, cj = w.ngg, mx // 2, my // 3
        spans = [((0, ci), (0, cj)), ((ci, mx - 1), (0, cj)), ((0, ci), (cj, my - 1)), ((ci, mx - 1), (cj, my - 1))]
        size = [(i1 - i0 + 1, j1 - j0 + 1) for (i0, i1), (j0, j1) in spans]
        out = []
        for n, ((i0, i1), (j0, j1)) in enumerate(spans):
            m, faces, inner = size[n], [], []
            cut = np.s_[..., j0:j1 + 1 + 2 * g, i0:i1 + 1 + 2 * g]
            for axis in (0, 1):
                for side in (-1, 1):
                    at = 0 if side < 0 else m[axis] - 1
                    lo, hi = [0, 0, 0], [m[0] - 1, m[1] - 1, 0]
                    lo[axis] = hi[axis] = at
                    high_block = bool(n & (1 << axis))
                    if high_block == (side > 0):  # an outer side
                        label = [f[2] for f in w.boundaries if f[0] == axis and f[1] == side][0]
                        faces.append((axis, side, label, lo, hi))
                        continue
                    o = n ^ (1 << axis)
                    src, tar = [1, m[0], -1, -m[1], 1, 1], [1, size[o][0], -1, -size[o][1], 1, 1]
                    src[2 * axis:2 * axis + 2] = [at + 1] * 2
                    tar[2 * axis:2 * axis + 2] = [1 if side > 0 else size[o][axis]] * 2
                    inner.append((src, tar, o + 1))
            c = Case(m[0], m[1], 1, g, *(np.ascontiguousarray(a[cut]) for a in (w.metric, w.jac, w.bv, w.sv)), faces,
                     dict(w.run), inner=inner, conditions=w.conditions)
            if tt:
                c.tve = np.ascontiguousarray(w.tve[cut])
            out.append(c)
        return out, t, STATE + (_abi.F_TVE,) if tt else STATE if physics == "h2" else STATE[:2]
    return make


def air_sod(mx, my):
    return [sod_case(mx, my)], None, STATE[:2]


def box_8th(mx, my, mz):
    def make(_mx, _my):
        t = load_tables()
        return [reacting_box_case(mx, my, mz, seed=9, tables=t)], t, STATE
    return make


def blocks(physics, visc):
    def make(_mx, _my):
        t = load_tables() if physics == "h2" else None
        bl = multiblock_case(split=(3, 2, 2) if physics == "air" else (2, 2, 2), seed=5, physics=physics, rotate=True)
        for c in bl:
            c.run.update(viscous_order=visc)
        return bl, t, STATE if physics == "h2" else STATE[:2]
    return make


@pytest.mark.parametrize("make,mx,my", [
    (body_2d, 97, 33), (plane_8th, 33, 21), (plane_one_temperature, 65, 18), (air_sod, 101, 9),
    (plane_k_faces(3, 21), 33, 21), (plane_k_faces(21, 2), 33, 21),
    (joined_planes("air"), 41, 33), (joined_planes("air5"), 41, 33), (joined_planes("h2"), 41, 33),
    (box_8th(101, 67, 53), 0, 0), (box_8th(250, 170, 20), 0, 0),
    (blocks("air", 0), 0, 0), (blocks("h2", 0), 0, 0), (blocks("h2", 8), 0, 0),
], ids=["body", "plane8", "plane1t", "sod", "k_symmetry", "k_walls", "joined_air",
        "joined_body", "joined_h2", "box8_long_chunks", "box8_two_a_block", "blocks_air", "blocks_h2",
        "blocks_h2_visc8"])
def test_step_is_its_operators(make, mx, my):
    bl, tb, fields = make(mx, my)
    run = dict(bl[0].run, fixed_time_step=1)
    s = {}
    for way in ("ops", "step", "recorded"):
        s[way] = Solver(dict(run, step_graph=int(way == "recorded")), tb)
        for c in bl:
            s[way].add_block(c)
        s[way].initialize()
    dt = 0.3 * s["ops"].cfl_dt()
    for _ in range(3):
        s["ops"].op(_abi.OP_COPY_QN)
        for rk in range(3):
            for op in OPS:
                if op != _abi.OP_LIMIT_FLOW or run.get("limit_flow"):
                    s["ops"].op(op, -1, rk, dt)
        s["step"].step(dt)
        s["recorded"].step(dt)
        for b in range(len(bl)):
            for f in fields:
                ref = s["ops"].download(b, f)
                for way in ("step", "recorded"):
                    got = s[way].download(b, f)
                    assert np.array_equal(got, ref), (way, b, f, np.abs(got - ref).max() / np.abs(ref).max())
    for v in s.values():
        v.close()


@pytest.mark.parametrize("pieces", [8, 9, 19])
def test_outflow_face_in_many_ranges(pieces):
    """One outflow face and the same face cut into ranges give the same ghosts."""
    t = load_air5_tables(True)
    out = []
    for n in (1, pieces):
        c = square_ogrid_case(97, 25, tables=t)
        kept, cut = [], []
        for f in c.boundaries:
            (cut if f[2] == 6 else kept).append(f)
        for face, direction, label, a, b in cut:
            edges = np.unique(np.linspace(a[0], b[0] + 1, n + 1).astype(int))
            for lo, hi in zip(edges[:-1], edges[1:]):
                kept.append((face, direction, label, (int(lo), a[1], a[2]), (int(hi) - 1, b[1], b[2])))
        c.boundaries = kept
        s = Solver(c.run, t)
        s.add_block(c)
        s.initialize()
        rng = np.random.default_rng(1)
        bv = s.download(0, _abi.F_BV)
        s.upload(0, bv * rng.uniform(0.9, 1.1, bv.shape), s.download(0, _abi.F_SV))
        s.op(_abi.OP_BC)
        out.append([s.download(0, f) for f in STATE + (_abi.F_TVE,)])
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("change", ["exponents", "order"])
def test_two_temperature_tables_outside_the_usual(change):
    """Reaction-temperature exponents other than the three usual pairs, and electronic levels in falling order
    with one of weight 0 (no early end of the sums)."""
    tables, ref = load_air5_tables(True), air5_tables(two_temperature=True)
    for t in (tables, ref):
        if change == "exponents":
            t.trx_model = 1
            for r in range(0, t.n_reac, 2):
                t.tcf_a[r], t.tcf_b[r] = 0.65, 0.35
                t.tcb_a[r], t.tcb_b[r] = 0.25, 0.75
        else:
            for l in range(t.n_spec):
                n = t.n_elec[l]
                th, g = list(t.elec_theta[l][:n])[::-1], list(t.elec_g[l][:n])[::-1]
                for j in range(n):
                    t.elec_theta[l][j], t.elec_g[l][j] = th[j], g[j]
                if n > 3:
                    t.elec_g[l][1] = 0.0
    case = air5_box_case(17, 11, 9, seed=12, tables=tables, two_temperature=True)
    s = Solver(case.run, tables)
    s.add_block(case)
    o = Oracle(case, ref)
    s.initialize()
    o.initialize()

    def close(a, b):
        a, b = a.reshape(a.shape[0], -1), b.reshape(b.shape[0], -1)
        den = np.abs(b).max(axis=1)
        if len(den) > 4:
            den[1:4] = den[1:4].max()
        err = np.abs(a - b).max(axis=1) / np.maximum(den, 1e-300)
        assert np.all(err <= STAGE_TOL), err

    g = case.ngg
    close(s.download(0, _abi.F_SV)[:, g:-g, g:-g, g:-g], o.a["sv"][:, g:-g, g:-g, g:-g])
    s.op(_abi.OP_ZERO_DQ)
    o.op("zero_dq")
    s.op(_abi.OP_CHEMISTRY)
    o.op("chemistry")
    close(s.download(0, _abi.F_DQ), o.a["dq"])
    s.close()
