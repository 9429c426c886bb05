"""The eight-wave integrator's own rate and factorisation code where the shipped mechanisms and usual states do not
take it: SRI and Lindemann fall-off, fall-off by one species, matrices whose panels are factored a second time with
the full pivot search.  Against the oracle with the bars of tests/test_gpu_chem.py, and against the one-wave
kernel."""
import os
import shutil
import struct

import numpy as np
import pytest

from tests.test_gpu_chem import REL, cell_errors, mixing_line_cells
from tests.test_gpu_launch_variants import restore_table, set_launch  # noqa: F401 (fixture)
from tests.test_gpu_mech2 import states

pytestmark = pytest.mark.gpu


def edit_link_file(src, dst, falloff=None, reaction=None, third=None):
    """A copy of a mechanism's folder with rows of its link file changed: falloff(f, form, species, par) and
    reaction(i, par) return the new values, third(t, bodies) the row's list of (species, efficiency)."""
    shutil.copytree(src, dst)
    path = os.path.join(dst, "chem.bin")
    data, at, records = bytearray(open(path, "rb").read()), 0, []
    while at < len(data):
        n = struct.unpack_from("<i", data, at)[0]
        records.append(at + 4)
        at += n + 8
    size = struct.unpack_from("<29i", data, records[1])
    ii, mxtb, npar, nfar, nfal, ntb = size[5], size[7], size[10], size[12], size[14], size[15]
    for i in range(ii if reaction else 0):
        p = records[4] + i * (8 + 8 * npar + 48) + 8
        struct.pack_into(f"<{npar}d", data, p, *reaction(i, list(struct.unpack_from(f"<{npar}d", data, p))))
    for f in range(nfal if falloff else 0):
        p = records[5] + f * (12 + 8 * nfar)
        form, sp = struct.unpack_from("<2i", data, p + 4)
        par = list(struct.unpack_from(f"<{nfar}d", data, p + 12))
        form, sp, par = falloff(f, form, sp, par)
        struct.pack_into(f"<2i{nfar}d", data, p + 4, form, sp, *par)
    for t in range(ntb if third else 0):
        p = records[6] + t * (8 + 12 * mxtb) + 4
        bodies = [struct.unpack_from("<id", data, p + 4 + 12 * l) for l in range(struct.unpack_from("<i", data, p)[0])]
        bodies = third(t, bodies)
        struct.pack_into("<i", data, p, len(bodies))
        for l, (k, a) in enumerate(bodies):
            struct.pack_into("<id", data, p + 4 + 12 * l, k, a)
    open(path, "wb").write(data)
    return str(dst)


def second_passes(M):
    """Whether the eight-wave factorisation of M takes a panel again: (a pivot outside 2^-100 .. 2^102 or a multiplier
    below 2^-790 but 0, two open rows of the pivot's upper 32 bits)."""
    M, n = M.copy(), len(M)
    rows, scale, ties = list(range(n)), False, False
    for k in range(n):
        p = max(rows, key=lambda r: abs(M[r, k]))
        high = np.abs(M[rows, k]).view(np.int64) >> 32
        ties |= bool((high == high.max()).sum() > 1)
        rows.remove(p)
        scale |= not 2.0 ** -100 <= abs(M[p, k]) < 2.0 ** 102
        for r in rows:
            f = M[r, k] / M[p, k]
            scale |= 0.0 < abs(f) < 2.0 ** -790
            M[r, k:] -= f * M[p, k:]
    return scale, ties


def newton_matrix(o, dt, rho, yT):
    """Of the first step over dt."""
    return np.eye(o.kk + 1) - 0.4358665 * dt * o.chem_jac(rho * 1e-3, yT)


def forms(h2o):
    """Rows in turn SRI, Lindemann, Troe as they were; every other one by H2O alone."""
    def change(f, form, sp, par):
        if f % 3 == 0:
            form, par[3:8] = 2, [0.54, 201.0, 1024.0, 1.05, 0.02]
        elif f % 3 == 1:
            form = 1
        return form, h2o + 1 if f % 2 == 0 else sp, par
    return change


def mechanism(name, folder):
    from fortrancfd_amd.lib import GRI30, LIDRYER_H2, Mechanism
    from oracle.pyoracle import Oracle
    src = GRI30 if name == "gri30" else LIDRYER_H2
    d = edit_link_file(src, folder / name, falloff=forms(Mechanism(src).names.index("H2O")))
    return Mechanism(d), Oracle(d)


@pytest.fixture(scope="module", params=["gri30", "h2"])
def changed(request, tmp_path_factory, orc):
    m, o = mechanism(request.param, tmp_path_factory.mktemp("mech"))
    n = 48
    if request.param == "gri30":
        yT, rho, dt = mixing_line_cells(orc, n, 91)
    else:
        Y, T, rho, dt = states(m, o, n, 92)
        yT = np.column_stack([Y, T])
    yT[:8, -1], dt[:8] = np.linspace(300.0, 900.0, 8), 1e-10      # cells that the screen accepts
    return request.param, m, o, yT, rho, dt


def test_rates(changed):
    name, m, o, yT, rho, _ = changed
    print(f"{name}: rates of {len(rho)} cells", flush=True)
    _, _, _, qf, qr = m.rates(rho * 1e-3, yT[:, -1], yT[:, :-1])
    for s in range(len(rho)):
        _, of, orv = o.ckwyr(rho[s] * 1e-3, yT[s, -1], yT[s, :-1])
        rel = lambda a, b: np.abs(a - b) / np.maximum(np.abs(b), 1e-300)
        assert rel(qf[s], of).max() <= 1e-14 and rel(qr[s], orv).max() <= 1e-14, s


@pytest.mark.parametrize("factor", [8, 0])
def test_integrator(changed, factor):
    """Eight waves a cell, one wave a cell."""
    name, m, o, yT, rho, dt = changed
    set_launch("chem_four_wave_factor", factor, m.kk)
    print(f"{name}: {len(rho)} cells, factor {factor}", flush=True)
    out, st = m.macks(dt, rho, yT)
    ref, rst = [], []
    for c in range(len(rho)):
        r, s, rc = o.chem_step(dt[c], rho[c], yT[c])
        assert rc == 0
        ref.append(r)
        rst.append((s["steps"], s["rejects"], s["newton"]))
    assert (st[:, 2] > 0).sum() > 10 and (st[:, 2] == 0).sum() >= 4
    assert (st[:, :3] == np.array(rst)).all()
    assert cell_errors(out, np.array(ref)).max() <= REL


@pytest.mark.parametrize("factor", [8, 0])
def test_domain(tmp_path, factor):
    """Steps with heat release; without the eight-wave kernel the lane-per-cell retry runs too."""
    m, o = mechanism("gri30", tmp_path)
    from tests.test_gpu_configs import ch4_air_cells, compare_fields, run_pair
    set_launch("chem_four_wave_factor", factor, m.kk)
    print(f"coupled hot-spot domain, factor {factor}", flush=True)
    cells = ch4_air_cells(m.kk, 64, [(0, 12, 2100.0), (12, 4, 1600.0)])
    s, d, dts_g, dts_o, h = run_pair(m, o, cells, 2, 32, 25e-6, 3, False)
    np.testing.assert_allclose(dts_g, dts_o, rtol=1e-13)
    compare_fields(s, d, dts_o, dts_o, o)


def test_ties(tmp_path, orc):
    """HCNO + H = H + HNCO so fast that 1 - hg J loses its 1: two species of one mass, two equal pivot
    candidates.  The four-wave kernel's sums have the eight-wave kernel's order; it runs for the same mechanism with
    ten third bodies in a row, three of them of efficiency 1."""
    from fortrancfd_amd.lib import GRI30, Mechanism
    from oracle.pyoracle import Oracle
    m = Mechanism(GRI30)
    par, nu, nk, ns, nr = orc.arrhenius()
    a, b, h = (m.names.index(s) + 1 for s in ("HCNO", "HNCO", "H"))
    at = [i for i in range(m.ii) if a in nk[i] and b in nk[i] and h in nk[i]]
    assert len(at) == 1
    fast = lambda i, p: [1e36, 0.0, 0.0] if i == at[0] else p
    ones = [m.names.index(s) + 1 for s in ("O2", "N2", "OH")]
    more = lambda t, rows: rows + [(k, 1.0) for k in ones] if t == 0 else rows
    dirs = [edit_link_file(GRI30, tmp_path / "eight", reaction=fast), edit_link_file(GRI30, tmp_path / "four", reaction=fast, third=more)]
    o = Oracle(dirs[0])
    yT, rho, dt = mixing_line_cells(orc, 32, 94)
    yT[:, h - 1] += 1e-4
    dt = np.maximum(dt, 1e-7)
    assert sum(second_passes(newton_matrix(o, dt[c], rho[c], yT[c])) == (False, True) for c in range(32)) > 16
    out = []
    for d in dirs:
        print(f"32 cells, {os.path.basename(d)} waves", flush=True)
        out.append(Mechanism(d).macks(dt, rho, yT))
    assert (out[0][1][:, 2] > 0).sum() > 16
    np.testing.assert_array_equal(out[0][1], out[1][1])
    np.testing.assert_array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("kind", ["trace", "stiff", "nan"])
def test_second_factorisation(tmp_path, kind):
    """Multipliers near the end of the exponent range (mass fractions of 1e-250), pivots far above 2^102 (a rate
    constant of 1e48), a matrix of NaN.  The sums of H2/O2's 21 reactions have the same order in both kernels, so the
    answers have the same bits."""
    from fortrancfd_amd.lib import LIDRYER_H2, Mechanism
    from oracle.pyoracle import Oracle
    d = LIDRYER_H2
    if kind == "stiff":
        d = edit_link_file(d, tmp_path / "h2", reaction=lambda i, p: [1e48, 0.0, 0.0] if i == 0 else p)
    m, o = Mechanism(d), Oracle(d)
    Y, T, rho, dt = states(m, o, 40, 93)
    if kind == "trace":
        for sp in ("H", "HO2", "H2O2", "O"):
            Y[:, m.names.index(sp)] = 10.0 ** -np.linspace(200.0, 270.0, 40)
    yT = np.column_stack([Y, T])
    if kind != "nan":
        odd = [second_passes(newton_matrix(o, dt[c], rho[c], yT[c]))[0] for c in range(40)]
        assert sum(odd) > 10
    else:
        yT, rho, dt = yT[:2], rho[:2], dt[:2]
        yT[0, m.names.index("OH")] = np.nan
    out = []
    for factor in (8, 0):
        set_launch("chem_four_wave_factor", factor, m.kk)
        print(f"{kind}: factor {factor}", flush=True)
        out.append(m.macks(dt, rho, yT))
    (a, sa), (b, sb) = out
    print("steps, rejects, newton, failed:", sa[:4].tolist())
    np.testing.assert_array_equal(sa, sb)
    np.testing.assert_array_equal(a, b)
    if kind == "nan":
        assert sa[0, 3] == 1 and np.isnan(a[0]).any() and np.isfinite(a[1]).all()
    else:
        assert (sa[odd, 2] > 0).sum() > 10
    if kind == "trace":
        ref = np.array([o.chem_step(dt[c], rho[c], yT[c])[0] for c in range(40)])
        assert cell_errors(a, ref).max() <= REL
