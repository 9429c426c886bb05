"""The integrator that gives a cell eight waves (short work lists): a cell's answer does not depend on
the list it is in, and a mechanism that does not suit the kernel's tables takes the one-wave kernel.
The bar is the same bits: the same arithmetic in another list or grid.  (The kernel against the oracle:
tests/test_gpu_chem.py, tests/test_gpu_mech2.py.)"""
import os
import shutil

import numpy as np
import pytest

from tests.test_gpu_chem import mixing_line_cells
from tests.test_gpu_launch_variants import restore_table, set_launch  # noqa: F401 (fixture)
from tests.test_gpu_mech2 import states

pytestmark = pytest.mark.gpu


def h2(text_dir=None):
    from fortrancfd_amd.lib import LIDRYER_H2, Mechanism
    from oracle.pyoracle import Oracle
    return Mechanism(text_dir or LIDRYER_H2, text=text_dir is not None), Oracle(LIDRYER_H2)


def gri30(orc):
    from fortrancfd_amd.lib import Mechanism
    return Mechanism(), orc


@pytest.mark.parametrize("name,n,pieces", [("gri30", 1, (1,)), ("gri30", 600, (1, 37, 562)), ("h2", 1100, (513, 2, 585))])
def test_answer_independent_of_list(orc, name, n, pieces):
    """More cells than workgroups (a workgroup's LDS goes from cell to cell), and the same cells in
    shorter lists down to one cell."""
    if name == "gri30":
        m, o = gri30(orc)
        yT, rho, dt = mixing_line_cells(o, n, 41)
    else:
        m, o = h2()
        Y, T, rho, dt = states(m, o, n, 42)
        yT = np.column_stack([Y, T])
    print(f"{name}: {n} cells at once, then {pieces}", flush=True)
    whole, st = m.macks(dt, rho, yT)
    assert (st[:, 3] == 0).all()
    assert n < 100 or (st[:, 2] > 0).sum() > 10
    at = 0
    for p in pieces:
        part, sp = m.macks(dt[at:at + p], rho[at:at + p], yT[at:at + p])
        np.testing.assert_array_equal(part, whole[at:at + p])
        np.testing.assert_array_equal(sp, st[at:at + p])
        at += p


def test_mechanism_beyond_the_tables(tmp_path):
    """Ten third-body efficiencies, six of them 1 (which change no bit): more than the eight-wave
    kernel holds, so its lists go to the one-wave kernel and give what that gives for the mechanism
    without them."""
    from fortrancfd_amd.lib import LIDRYER_H2
    d = tmp_path / "mech"
    shutil.copytree(LIDRYER_H2, d)
    p = os.path.join(d, "chem.inp")
    lines = open(p).read().splitlines()
    at = next(i for i, l in enumerate(lines) if l.strip().startswith("H2/2.5/ H2O/12/"))
    lines.insert(at + 1, "   O2/1.0/ H/1.0/ O/1.0/ OH/1.0/ HO2/1.0/ H2O2/1.0/")
    open(p, "w").write("\n".join(lines) + "\n")
    more, o = h2(str(d))
    plain, _ = h2()
    Y, T, rho, dt = states(plain, o, 64, 45)
    yT = np.column_stack([Y, T])
    print("64 cells, mechanism with ten third bodies", flush=True)
    a, sa = more.macks(dt, rho, yT)
    set_launch("chem_four_wave_factor", 0, plain.kk)
    b, sb = plain.macks(dt, rho, yT)
    assert (sa[:, 2] > 0).sum() > 10
    np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(sa, sb)
