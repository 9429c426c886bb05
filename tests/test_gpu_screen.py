"""The explicit screen at the edges of its launch shape: a workgroup takes 64 cells, its waves draw reaction
rows in no fixed order, and the rows come in chunks (three for GRI-3.0, one for H2/O2).  A quiescent cell's
answer is the same bits in batches of 1, 63, 64, 65 and more cells, and from run to run.  (Against the
oracle: tests/test_gpu_chem.py, tests/test_gpu_mech2.py.)"""
import numpy as np
import pytest

from tests.test_gpu_chem import mixing_line_cells
from tests.test_gpu_mech2 import states

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["gri30", "h2"])
def test_quiescent_cells_independent_of_batch(orc, name):
    from fortrancfd_amd.lib import GRI30, LIDRYER_H2, Mechanism
    from oracle.pyoracle import Oracle
    m = Mechanism(GRI30 if name == "gri30" else LIDRYER_H2)
    n = 193
    if name == "gri30":
        yT, rho, dt = mixing_line_cells(orc, n, 51)
    else:
        Y, T, rho, dt = states(m, Oracle(LIDRYER_H2), n, 52)
        yT = np.column_stack([Y, T])
    yT[:, -1] = np.random.default_rng(53).uniform(280.0, 900.0, n)
    dt[:] = 1e-10
    print(f"{name}: {n} quiescent cells", flush=True)
    whole, st = m.macks(dt, rho, yT)
    assert (st[:, 0] == 1).sum() > n // 2 and (st[:, 3] == 0).all()
    at = 0
    for p in (1, 63, 64, 65):
        part, sp = m.macks(dt[at:at + p], rho[at:at + p], yT[at:at + p])
        np.testing.assert_array_equal(part, whole[at:at + p])
        np.testing.assert_array_equal(sp, st[at:at + p])
        at += p
    for _ in range(3):
        again, _ = m.macks(dt, rho, yT)
        np.testing.assert_array_equal(again, whole)
