"""The fluid kernels that split a column's species over the waves of a workgroup, against the oracle bit
for bit: cell counts around the tiles' edges (32 interfaces, 64 columns), every reconstruction and
Riemann solver, compositions whose quotients leave the range of the shared-reciprocal division
(subnormal and near-subnormal mass fractions, where the plain division takes over), temperatures on
both sides of the mid temperatures within one wave."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mechs():
    from fortrancfd_amd.lib import LIDRYER_H2, Mechanism
    from oracle.pyoracle import Oracle
    return {"gri30": (Mechanism(), Oracle()), "h2": (Mechanism(LIDRYER_H2), Oracle(LIDRYER_H2))}


def cells_for(kk, n, seed, tiny):
    rng = np.random.default_rng(seed)
    cells = np.zeros((n, 3 + kk))
    cells[:, 0] = rng.uniform(300.0, 2200.0, n)
    cells[:n // 3, 0] = rng.uniform(990.0, 1500.0, n // 3)         # around the mid temperatures
    cells[:, 1] = 101325.0 * rng.uniform(0.7, 1.4, n)
    cells[:, 2] = rng.uniform(-300.0, 300.0, n)
    x = rng.dirichlet(np.full(kk, 0.3), n)
    if tiny:
        x[:, 1] = 10.0 ** rng.uniform(-323.0, -180.0, n)
        x[:, 4] = 0.0
        x[::2, 6] = 3e-310
        x[::5, kk - 1] = 1e-212
    cells[:, 3:] = x
    return cells


SCHEMES = [dict(flag_acu=2, flag_weno=2, select_riemann=2), dict(flag_acu=2, flag_weno=3, select_riemann=1),
           dict(flag_acu=2, flag_weno=1, select_riemann=0), dict(flag_acu=2, flag_weno=4, select_riemann=2),
           dict(flag_acu=1, flag_muscl=4, select_riemann=2), dict(flag_acu=0, select_riemann=1),
           dict(flag_acu=2, flag_weno=3, select_riemann=2, select_time=0)]


@pytest.mark.parametrize("name,nblk,ncell,si,tiny", [
    ("gri30", 1, 8, 0, False), ("gri30", 1, 31, 0, True), ("gri30", 1, 32, 1, False), ("gri30", 3, 33, 1, True),
    ("gri30", 2, 58, 2, True), ("gri30", 2, 64, 3, False), ("gri30", 5, 27, 3, True), ("gri30", 4, 65, 4, True),
    ("gri30", 2, 40, 5, True), ("gri30", 1, 130, 6, True), ("gri30", 7, 64, 0, True), ("h2", 1, 31, 0, True),
    ("h2", 3, 33, 1, False), ("h2", 2, 61, 3, True), ("h2", 4, 65, 4, False)])
def test_split_kernels_bit_exact(mechs, name, nblk, ncell, si, tiny):
    from fortrancfd_amd.lib import Solver
    from oracle.pyoracle import Domain
    mech, orc = mechs[name]
    kw = SCHEMES[si]
    cells = cells_for(mech.kk, nblk * ncell, 100 * ncell + si, tiny)
    print(f"{name} {nblk} x {ncell} {kw} tiny={tiny}", flush=True)
    s = Solver(mech, nblk, ncell, 25e-6, **kw)
    s.init_cells(cells)
    d = Domain(orc, cells, nblk, ncell, 25e-6, **kw)
    np.testing.assert_array_equal(s.download()[0], d.Qc)
    for step in range(3):
        dt_o, dt_g = d.calc_dt(0.3), s.calc_dt(0.3)
        assert dt_o == dt_g, step
        d.solve_fluid(dt_o)
        d.refresh()
        s.solve_fluid(dt_g)
        s.refresh()
    Qc, qf = s.download()
    np.testing.assert_array_equal(Qc, d.Qc)
    np.testing.assert_array_equal(qf, d.qf)


@pytest.mark.parametrize("name,n", [("gri30", 1), ("gri30", 5), ("gri30", 61), ("gri30", 4093), ("gri30", 4094),
                                    ("gri30", 4097), ("h2", 3), ("h2", 4096)])
def test_transport_flux_cell_counts(mechs, name, n):
    """The transport flux on one block of n cells, on both sides of the count from which a wave takes
    two cells and with every remainder, against the oracle: bit for bit (the mixture rules' sums run
    in the same order)."""
    mech, orc = mechs[name]
    lv = 3
    cells = cells_for(mech.kk, n + 2 * lv, 17 + n, False)
    cells[:, 0] = 300.0 + 1900.0 * np.linspace(0.0, 1.0, n + 2 * lv)
    Qc = np.zeros((n + 2 * lv, 3 + mech.kk))
    for i, row in enumerate(cells):
        T, p, u, X = row[0], row[1], row[2], row[3:]
        rho = orc.density(p, T, X)
        e = orc.specific_energy(T, X)
        Qc[i] = np.concatenate([[rho, rho * u, rho * (e + 0.5 * u * u)], rho * orc.xty(X)])
    print(f"transport flux {name} n={n}", flush=True)
    F = mech.calc_flux_tran(Qc, n, lv, 25e-6)
    R = orc.flux_tran(Qc, n, lv, 25e-6)
    np.testing.assert_array_equal(F, R)
