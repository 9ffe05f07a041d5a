"""The size rules that split a kernel's work over more or fewer threads, against the oracle at sizes on
both sides of each rule and at ragged ends of its tiles."""
import re
from pathlib import Path

import numpy as np
import pytest

from corefl_amd import ReactorServer, Solver, _abi, channel_case, h2_air_mass_fractions, load_tables
from oracle import Oracle

pytestmark = pytest.mark.gpu

# one operator, FP64 sums of at most 27 terms against the same sums in another order
STAGE_TOL = 1e-11


def normwise(a, b):
    """Per-plane max|a-b| / max|b|, the momentum planes against the largest of the three."""
    a, b = a.reshape(a.shape[0], -1), b.reshape(b.shape[0], -1)
    den = np.abs(b).max(axis=1)
    den[1:4] = den[1:4].max()
    return np.abs(a - b).max(axis=1) / np.maximum(den, 1e-300)


@pytest.fixture(scope="module")
def tables():
    return load_tables()


def column_split(mx, my, mz, fields):
    """column_split of the kernels: (k nodes of a chunk, fields of a block)."""
    src = (Path(__file__).parent.parent / "corefl-cpc_amd" / "csrc" / "kernels.hip").read_text()
    most = int(re.search(r"constexpr long kColumnWaves = (\d+);", src)[1])
    waves = (mx * my * -(-mz // 16) + 63) // 64
    per_block = max(1, waves * fields // most) if waves * 2 < most else fields
    return (4 if per_block == 1 and waves * fields < most // 2 else 16), per_block


@pytest.mark.parametrize("mx,my,mz,chunk,per_block", [
    (16, 9, 5, 4, 1),        # one short chunk of k (4 nodes and 1), boundary closures from both ends
    (21, 13, 18, 4, 1),      # the 4-node chunks with a remainder
    (96, 70, 37, 4, 1),      # the last size before the long chunks
    (101, 67, 53, 16, 1),    # 16-node chunks, a component to a block, remainder of 5
    (250, 170, 20, 16, 2),   # a few components to a block, the last block's fewer
    (520, 510, 9, 16, 13),   # enough columns for all components in one block
])
def test_viscous_column_splits(tables, h2_oracle_tables, mx, my, mz, chunk, per_block):
    """8th-order viscous operator between walls, inflow, outflow and symmetry planes."""
    assert column_split(mx, my, mz, 13) == (chunk, per_block)
    case = channel_case(mx, my, mz, physics="h2", seed=mx)
    s = Solver(case.run, tables)
    s.add_block(case)
    o = Oracle(case, h2_oracle_tables)
    s.initialize()
    o.initialize()
    s.op(_abi.OP_ZERO_DQ)
    o.op("zero_dq")
    s.op(_abi.OP_VISCOUS)
    o.op("viscous")
    gpu, ref = s.download(0, _abi.F_DQ), o.a["dq"]
    s.close()
    err = normwise(gpu, ref)
    # a species whose own gradients are far below Y / dx (fine grids) is dominated by the rounding of Y and of
    # the other species' fluxes in its correction velocity, two derivatives of J |grad xi| each: bound it by
    # 64 roundings of that size beside the relative tolerance
    m, rho_d, y = o.a["metric"], o.a["rhoD"], o.a["sv"]
    k2 = max((o.a["jac"] * (m[3 * d:3 * d + 3] ** 2).sum(axis=0)).max() for d in range(3))
    top = [float((rho_d[l] * y[l]).max()) for l in range(9)]
    for l in range(9):
        bound = 64 * 2.2e-16 * k2 * (top[l] + y[l].max() * sum(top))
        worst = np.abs(gpu[5 + l] - ref[5 + l]).max()
        assert worst <= STAGE_TOL * np.abs(ref[5 + l]).max() + bound, (l, worst, bound)
    assert np.all(err[:5] <= STAGE_TOL), err


def test_reactor_result_across_the_kernel_switch(tables):
    """With many slots in flight (reactor_wave_slots; never more than 16,384) a reactor has a lane, with fewer a
    wave: 16,500 requests start on the first, and once the short ones are done the others finish on the second,
    bit for bit as they do alone."""
    mw = np.array(tables.mw[:9])
    n = 16500

    def request(i):
        r = np.random.default_rng(i)
        return dict(temperature=r.uniform(1000.0, 1600.0), pressure=r.uniform(1.0, 10.0) * 101325.0,
                    y=h2_air_mass_fractions(r.uniform(0.5, 2.0), mw), t_end=2e-5 if i % 16 == 0 else 2e-7, dt=1e-8)

    pick = [0, 16 * 500, 16400]
    alone = {}
    for i in pick:
        srv = ReactorServer(tables, budget_bytes=1 << 20, steps_per_launch=16)
        t = srv.submit(**request(i))
        alone[i] = srv.run_until_done([t])[t]
        srv.close()
    srv = ReactorServer(tables, budget_bytes=32 << 20, steps_per_launch=16)
    assert srv.capacity >= n
    tickets = [srv.submit(**request(i)) for i in range(n)]
    while srv.progress():
        pass
    res = srv.drain(n)
    srv.close()
    assert len(res) == n and all(r["status"] == 0 for r in res.values())
    for i in pick:
        r = res[tickets[i]]
        assert r["steps"] == alone[i]["steps"] and r["rejected"] == alone[i]["rejected"]
        assert r["temperature"] == alone[i]["temperature"] and np.array_equal(r["y"], alone[i]["y"])
