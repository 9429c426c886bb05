"""A domain of more than 2^29 columns: a row of the state is longer than 4 GB, past what a 32-bit byte offset from
its start reaches.  Only the last blocks hold a gas (the others are zero, and NaN after a step); far enough from
them the last blocks take one step to the same bits as in a domain that ends like this one and has 100 blocks."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TAIL = 100


def step(mech, nblk, cells):
    """One Euler step of nblk blocks of three cells, the last TAIL of them from cells; their state after it."""
    from fortrancfd_amd.lib import Solver, _check, _p, lib
    s = Solver(mech, TAIL, 3, 25e-6, flag_acu=2, flag_weno=2, select_riemann=2, select_time=0)
    s.init_cells(cells)
    if nblk > TAIL:
        Q, q = s.download()
        s = Solver(mech, nblk, 3, 25e-6, flag_acu=2, flag_weno=2, select_riemann=2, select_time=0)
        for b in range(TAIL):
            _check(lib().fcfd_upload(s.handle, C.c_int(nblk - TAIL + b), _p(Q[b]), _p(q[b])))
    dt = s.calc_dt(0.5)
    s.solve_fluid(dt)
    Q, q = np.zeros((TAIL, 9, mech.nequ)), np.zeros((TAIL, 9, mech.nequ))
    for b in range(TAIL):
        _check(lib().fcfd_download(s.handle, C.c_int(nblk - TAIL + b), _p(Q[b]), _p(q[b])))
    return dt, Q, q


def test_last_blocks():
    import torch
    from fortrancfd_amd.lib import LIDRYER_H2, Mechanism
    mech = Mechanism(LIDRYER_H2)
    nblk = (2 ** 29 + 2 ** 16) // 9
    # four states, fluxes, Roe states, cell centres
    need = 8.0 * nblk * (4 * mech.nequ * 9 + (mech.nequ + 3) * 4 + 3) + 4e9
    if torch.cuda.mem_get_info()[0] < need:
        pytest.skip(f"needs {need / 1e9:.0f} GB of GPU memory")
    rng = np.random.default_rng(71)
    n = TAIL * 3
    cells = np.zeros((n, mech.nequ))
    cells[:, 0] = rng.uniform(600.0, 2000.0, n)
    cells[:, 1] = 101325.0 * rng.uniform(0.8, 1.25, n)
    cells[:, 2] = rng.uniform(-20.0, 20.0, n)
    cells[:, 3:] = rng.dirichlet(np.ones(mech.kk), n)
    print(f"100 blocks, then {nblk}", flush=True)
    dt0, Q0, q0 = step(mech, TAIL, cells)
    dt1, Q1, q1 = step(mech, nblk, cells)
    assert dt0 == dt1 and np.isfinite(q0).all()
    # (three cells a side at each end of a step: five blocks are more than enough)
    np.testing.assert_array_equal(Q1[5:], Q0[5:])
    np.testing.assert_array_equal(q1[5:], q0[5:])
