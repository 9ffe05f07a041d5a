"""The size rules that split a kernel's work over more or fewer threads, against the oracle at sizes on
both sides of each rule and at ragged ends of its tiles."""
import numpy as np
import pytest

from corefl_amd import Solver, _abi, channel_case, load_tables
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


@pytest.mark.parametrize("mx,my,mz", [
    (16, 9, 5),        # one short chunk of k (4 nodes and 1), boundary closures from both ends
    (21, 13, 18),      # the 4-node chunks with a remainder
    (96, 70, 37),      # 16-node chunks, components over blocks, remainder of 5
    (520, 510, 9),     # enough columns for all components in one block
])
def test_viscous_column_splits(tables, h2_oracle_tables, mx, my, mz):
    """8th-order viscous operator between walls, inflow, outflow and symmetry planes."""
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
    err = normwise(s.download(0, _abi.F_DQ), o.a["dq"])
    assert np.all(err <= STAGE_TOL), err
    s.close()
