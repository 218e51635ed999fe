"""The energy by log-determinants against the eigenvalue methods
(MBD_EIG_METHOD), at the edges of its kernels' blocks and over every branch:
the first and the second guess of the spectrum's lower end, and matrices that
have eigenvalues not above zero and must take the eigenvalue path."""
import numpy as np
import pytest

from mbd_amd import engine, generators
from mbd_amd.io import BOHR, Geometry, Settings

pytestmark = pytest.mark.gpu


def _both(geo, st, monkeypatch, method="1"):
    with engine.MbdEngine(0) as eng:
        eng.set_geometry(geo, st)
        a, _, _, c, _, _ = eng.scs("fp64")
        monkeypatch.setenv("MBD_EIG_METHOD", method)
        want, om, _, dw = eng.energy(a, c)
        monkeypatch.delenv("MBD_EIG_METHOD")
        eng.profile_enable(True)
        got, _, _, dg = eng.energy(a, c)
        prof = eng.profile_read()
    cells = int(np.prod(dw["supercell"]))
    # both sum 3 N cells square roots of eigenvalues with a backward error of
    # about the order times eps each, divided by the number of cells
    tol = 2.2e-16 * 3 * geo.n_atoms * cells * 1.5 * np.sum(om)
    assert dg["n_negative"] == dw["n_negative"]
    assert dg["supercell"] == dw["supercell"]
    return got, want, tol, dg, prof


def _spread(n, seed, gap=2.2):
    """n atoms on a jittered cubic grid: physical at any n."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    xyz = gap * g + rng.uniform(-0.2, 0.2, (n, 3))
    return Geometry(list(rng.choice(["C", "H", "N", "O"], n)), xyz, rng.uniform(0.6, 0.95, n), None)


# orders 3, 63, 66, 126, 129, 192, 195, 387, 771: one short of and one past the
# bounds' 64-row and the factorisation's 128-row blocks
@pytest.mark.parametrize("n", [1, 21, 22, 42, 43, 64, 65, 129, 257])
def test_matches_eigenvalues(n, monkeypatch):
    got, want, tol, _, prof = _both(_spread(n, n), Settings(), monkeypatch)
    assert prof["logdet_diag"]["launches"] > 0 and prof["bisect"]["launches"] == 0
    assert abs(got - want) <= tol


# orders from 7000 on: the interval from Ritz values (order 7002 and, one short
# of whole 128-row blocks, 7167), and one that shows an eigenvalue below zero
@pytest.mark.parametrize("n", [2334, 2389])
def test_interval_from_ritz_values(n, monkeypatch):
    got, want, tol, _, prof = _both(_spread(n, n), Settings(), monkeypatch, "2")
    assert prof["logdet_diag"]["launches"] == -(-3 * n // 128)  # the first guess holds
    assert abs(got - want) <= tol


def test_ritz_value_below_zero(monkeypatch):
    geo = _spread(2334, 7)
    a = np.full(2334, 60.0)
    with engine.MbdEngine(0) as eng:
        eng.set_geometry(geo, Settings())
        monkeypatch.setenv("MBD_EIG_METHOD", "2")
        want, om, _, dw = eng.energy(a, 0.75 * 0.5 * a * a)
        monkeypatch.delenv("MBD_EIG_METHOD")
        eng.profile_enable(True)
        got, _, _, dg = eng.energy(a, 0.75 * 0.5 * a * a)
        prof = eng.profile_read()
    assert dw["n_negative"] > 0 and dg["n_negative"] == dw["n_negative"]
    assert prof["logdet_diag"]["launches"] == 0 and prof["bisect"]["launches"] > 0
    assert got == want


def test_supercell_with_cells(monkeypatch):
    geo, st = generators.hex_sheet(4, 3, seed=9, rc_scs=40.0)
    got, want, tol, dg, _ = _both(geo, st, monkeypatch)
    assert np.prod(dg["supercell"]) > 1
    assert abs(got - want) <= tol


def _line(n, gap):
    return Geometry(["C"] * n, np.array([[0.0, 0.0, gap * i] for i in range(n)]), np.full(n, 0.95), None)


def _energy(geo, alpha, monkeypatch, method=None):
    """Energy of given polarisabilities at C6 that keep omega at 0.5."""
    a = np.full(geo.n_atoms, alpha)
    with engine.MbdEngine(0) as eng:
        eng.set_geometry(geo, Settings())
        if method:
            monkeypatch.setenv("MBD_EIG_METHOD", method)
        eng.profile_enable(True)
        e, om, rf, d = eng.energy(a, 0.75 * 0.5 * a * a)
        prof = eng.profile_read()
        C = eng.cfdm_matrix(a, om, rf, 1)
        if method:
            monkeypatch.delenv("MBD_EIG_METHOD")
    lam = np.linalg.eigvalsh(np.tril(C) + np.tril(C, -1).T)
    return e, om, d, prof, lam


@pytest.mark.parametrize("lo,hi,path", [(0.3, 1.0, "first"), (0.03, 0.28, "second"), (-9.0, 0.0, "eig")])
def test_every_branch(lo, hi, path, monkeypatch):
    """A line of atoms whose polarisability is raised until the smallest
    eigenvalue over omega^2 falls into (lo, hi)."""
    geo = _line(24, 0.7)
    for alpha in np.arange(2.0, 60.0, 1.0):
        e, om, d, prof, lam = _energy(geo, alpha, monkeypatch)
        if lo < lam[0] / om.min() ** 2 < hi:
            break
    else:
        pytest.fail("no polarisability reaches the range")
    want = 0.5 * np.sqrt(lam[lam >= 0]).sum() - 1.5 * om.sum()
    tol = 2.2e-16 * 72 * 1.5 * om.sum() * (1.0 if path == "first" else 30.0)
    assert d["n_negative"] == int(np.sum(lam < 0))
    assert (prof["bisect"]["launches"] > 0) == (path == "eig")
    # one 72 x 72 diagonal block per attempt
    assert prof["logdet_diag"]["launches"] == (1 if path == "first" else 2)
    assert abs(e - want) <= tol


# cells short enough for 2, 3 and 4 cells along an axis (real wave vectors,
# conjugate pairs, both), with and without a vacuum axis; atoms outside the
# home cell and a skewed lattice, whose image boxes do not cover the cutoff
# sphere, and images on the cutoff sphere to rounding (2 x 30 A at 60 A) keep
# the matrix of the whole supercell
@pytest.mark.parametrize("edges,vac,skew,out,cells,launches", [
    ((13.0, 14.0, 14.5), None, 0.0, 0.0, [2, 2, 2], 2),
    ((13.0, 14.0, 15.0), None, 0.0, 0.0, [2, 2, 2], 3),
    ((9.0, 13.0, 26.0), None, 0.0, 0.0, [3, 2, 1], 2),
    ((8.5, 9.0, 20.0), 2, 0.0, 0.0, [3, 3, 1], 2),
    ((7.0, 26.0, 27.0), None, 0.0, 0.0, [4, 1, 1], 2),
    ((13.0, 14.0, 26.0), None, 0.0, 4.0, [2, 2, 1], 1),
    ((13.0, 14.0, 26.0), None, 20.0, 0.0, [2, 2, 1], 1),
])
def test_supercell_by_wave_vectors(edges, vac, skew, out, cells, launches, monkeypatch):
    rng = np.random.default_rng(int(sum(edges)))
    geo = _spread(18, 5, gap=2.3)
    xyz = geo.coords_ang - geo.coords_ang.min(0)
    if out:
        xyz[0, 0] += out * edges[0]  # an atom some cells away
    lat = np.diag(edges).astype(float)
    lat[1, 0] = skew
    geo = Geometry(geo.names, xyz + rng.uniform(0, 0.1, xyz.shape), geo.hirshfeld, lat)
    st = Settings(mbd_supercell_cutoff=25.0, mbd_cfdm_dip_cutoff=60.0, mbd_scs_dip_cutoff=30.0,
                  mbd_scs_vacuum_axis=tuple(k == vac for k in range(3)))
    got, want, tol, dg, prof = _both(geo, st, monkeypatch)
    assert dg["supercell"] == cells
    # blocks by cell difference and their transform, or the whole matrix
    assert prof["cfdm_build"]["launches"] == launches
    assert abs(got - want) <= tol


# atoms whose C6, and with it omega = 4 C6 / (3 alpha^2), is negative or zero:
# the energy's -3/2 sum omega takes it with its sign, in a molecule and in a
# supercell
@pytest.mark.parametrize("w", [-0.4, 0.0])
@pytest.mark.parametrize("edge", [None, 13.0])
def test_omega_not_positive(w, edge, monkeypatch):
    geo = _spread(5, 3)
    xyz = geo.coords_ang - geo.coords_ang.min(0)
    geo = Geometry(geo.names, xyz, geo.hirshfeld, None if edge is None else np.diag([edge, 26.0, 27.0]))
    st = Settings(mbd_supercell_cutoff=25.0, mbd_cfdm_dip_cutoff=30.0, mbd_scs_dip_cutoff=20.0)
    cells = 1 if edge is None else 2
    a = np.full(5, 3.0)
    omega = np.array([0.5, 0.6, w, 0.55, 0.45])
    with engine.MbdEngine(0) as eng:
        eng.set_geometry(geo, st)
        got, om, rf, d = eng.energy(a, 0.75 * omega * a * a)
        monkeypatch.setenv("MBD_EIG_METHOD", "1")
        by_eig = eng.energy(a, 0.75 * omega * a * a)[0]
        monkeypatch.delenv("MBD_EIG_METHOD")
        C = eng.cfdm_matrix(a, om, rf, cells)
    lam = np.linalg.eigvalsh(np.tril(C) + np.tril(C, -1).T)
    # a row of zeros (omega = 0) has eigenvalue 0 to rounding: either sign, no energy
    want = 0.5 * np.sqrt(lam[lam >= 0]).sum() / cells - 1.5 * omega.sum()
    assert np.allclose(om, omega, rtol=1e-15, atol=0)
    # 15 cells square roots of eigenvalues good to 15 cells eps; sqrt(15 cells eps) at a zero one
    tol = 2.2e-16 * 15 * cells * 1.5 * np.abs(om).sum() if w else 3.0 * np.sqrt(2.2e-16 * 15 * cells)
    assert abs(got - want) <= tol
    assert got == by_eig


def test_supercell_with_negative_eigenvalues(monkeypatch):
    """The wave vectors' matrices have the supercell's eigenvalues: what they
    decline goes to the eigenvalues at once."""
    rng = np.random.default_rng(2)
    g = 3.25 * np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), -1).reshape(-1, 3)
    geo = Geometry(["C"] * 64, g + rng.uniform(0, 0.1, g.shape), np.full(64, 0.8), np.diag([13.0, 13.2, 13.3]))
    st = Settings(mbd_supercell_cutoff=25.0, mbd_cfdm_dip_cutoff=60.0, mbd_scs_dip_cutoff=30.0)
    a = np.full(64, 150.0)
    with engine.MbdEngine(0) as eng:
        eng.set_geometry(geo, st)
        monkeypatch.setenv("MBD_EIG_METHOD", "2")  # the default method of order 1536
        want, _, _, dw = eng.energy(a, 0.75 * 0.5 * a * a)
        monkeypatch.delenv("MBD_EIG_METHOD")
        eng.profile_enable(True)
        got, _, _, dg = eng.energy(a, 0.75 * 0.5 * a * a)
        prof = eng.profile_read()
    assert dw["supercell"] == [2, 2, 2] and dg["n_negative"] == dw["n_negative"] > 0
    # the wave vectors' matrices of order 192, two diagonal blocks in each of
    # two attempts; the whole matrix of order 1536 would add twelve in each
    assert 0 < prof["logdet_diag"]["launches"] <= 4 and prof["bisect"]["launches"] > 0
    assert got == want


def test_second_guess_proved_first(monkeypatch):
    """A matrix of order 3000 with negative eigenvalues: the nodes of the first
    guess are factored, of the second only its proof."""
    geo = _spread(1000, 7)
    a = np.full(1000, 60.0)
    with engine.MbdEngine(0) as eng:
        eng.set_geometry(geo, Settings())
        monkeypatch.setenv("MBD_EIG_METHOD", "2")
        want, _, _, dw = eng.energy(a, 0.75 * 0.5 * a * a)
        monkeypatch.delenv("MBD_EIG_METHOD")
        eng.profile_enable(True)
        got, _, _, dg = eng.energy(a, 0.75 * 0.5 * a * a)
        prof = eng.profile_read()
    assert dg["n_negative"] == dw["n_negative"] > 0
    assert got == want
    # trailing updates are n^3 / 3 operations less the blocks' own per matrix;
    # the nodes of one set are at most 13 (interval ends up to 0.3 : 12) and
    # those of the second at least 12 (0.03 : 1)
    mats = prof["logdet_syrk_gemm"]["flops"] / (3000.0 ** 3 / 3.0)
    assert 8 < mats <= 15


# a set of shifted matrices is left at the first pivot that is not positive: at
# row 231 of 3000 (by numpy's factorisation), and at row 778 of 780, where
# everything before it is factored; the handle's next energy is whole again
@pytest.mark.parametrize("case", ["early", "last"])
def test_set_left_at_first_bad_pivot(case, monkeypatch):
    if case == "early":
        n, alpha, method, geo = 1000, 60.0, "2", _spread(1000, 7)
    else:
        n, alpha, method, geo = 260, 30.0, "1", _spread(260, 4, gap=4.0)
        xyz = geo.coords_ang
        xyz[-1] = xyz[-2] + [0.3, 0.0, 0.0]
        geo = Geometry(["C"] * n, xyz, np.full(n, 0.95), None)
    low, a = np.full(n, 4.0), np.full(n, alpha)
    with engine.MbdEngine(0) as eng:
        eng.set_geometry(geo, Settings())
        eng.profile_enable(True)
        good = eng.energy(low, 0.75 * 0.5 * low * low)[0]
        whole = eng.profile_read()
        monkeypatch.setenv("MBD_EIG_METHOD", method)
        want, om, rf, dw = eng.energy(a, 0.75 * 0.5 * a * a)
        monkeypatch.delenv("MBD_EIG_METHOD")
        eng.profile_enable(True)
        got, _, _, dg = eng.energy(a, 0.75 * 0.5 * a * a)
        prof = eng.profile_read()
        again = eng.energy(low, 0.75 * 0.5 * low * low)[0]
    assert dg["n_negative"] == dw["n_negative"] > 0
    assert got == want and again == good
    assert whole["bisect"]["launches"] == 0 and prof["bisect"]["launches"] > 0
    if case == "early":  # both guesses together take less than half of one whole set
        assert prof["logdet_syrk_gemm"]["ms"] < 0.5 * whole["logdet_syrk_gemm"]["ms"]


# primitive cells, many short axes with different numbers of cells: tens to
# over a thousand wave vectors of order 3, 6 and 60
@pytest.mark.parametrize("n,edge,cells", [(1, 2.5, [11, 10, 11]), (2, 4.6, [6, 6, 6]), (20, 7.6, [4, 4, 4])])
def test_primitive_cells(n, edge, cells, monkeypatch):
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] * edge / m
    lat = np.diag([0.998 * edge, 1.003 * edge, 0.997 * edge])
    geo = Geometry(["H" if n == 1 else "Ar"] * n, g + rng.uniform(0, 0.1, g.shape), np.full(n, 0.8), lat)
    st = Settings(mbd_supercell_cutoff=25.0, mbd_cfdm_dip_cutoff=60.0, mbd_scs_dip_cutoff=20.0)
    a = np.full(n, 2.0)
    with engine.MbdEngine(0) as eng:
        eng.set_geometry(geo, st)
        times = {}
        for method in ("2" if 3 * n * np.prod(cells) >= 1024 else "1", None):
            if method:
                monkeypatch.setenv("MBD_EIG_METHOD", method)
            for _ in range(2):  # the first pass allocates
                e, om, _, d = eng.energy(a, 0.75 * 0.5 * a * a)
            times[method] = (e, d["t_mbd_ms"])
            if method:
                monkeypatch.delenv("MBD_EIG_METHOD")
    (want, t_eig), (got, t_cells) = times.values()
    assert d["supercell"] == cells
    assert abs(got - want) <= 2.2e-16 * 3 * n * np.prod(cells) * 1.5 * np.sum(om)
    assert t_cells < t_eig


def _budget(geo, st, gb, monkeypatch):
    """Energy with room for all shifted matrices and within a memory budget; the
    launches of the diagonal blocks of both; the eigenvalues' energy."""
    with engine.MbdEngine(0) as eng:
        eng.set_geometry(geo, st)
        a, _, _, c, _, _ = eng.scs("fp64")
        out = []
        for env in ({}, {"MBD_SCS_MEM_GB": gb}, {"MBD_EIG_METHOD": "1"}):
            for k, v in env.items():
                monkeypatch.setenv(k, v)
            eng.profile_enable(True)
            e, om, _, d = eng.energy(a, c)
            out.append((e, eng.profile_read()))
            for k in env:
                monkeypatch.delenv(k)
    tol = 2.2e-16 * 3 * geo.n_atoms * np.prod(d["supercell"]) * 1.5 * np.sum(om)
    assert abs(out[0][0] - out[2][0]) <= tol
    return out, d["supercell"]


# a few shifted matrices at a time: of one matrix its nodes in parts (order 771:
# 5.8 MB each, 3 at a time), of several matrices a part of them with all their
# nodes (order 54: 158 KB, order 108 of the paired wave vectors 228 KB; 9 to 13
# shifts each, so 5.5 MB hold two or three of eight, and one or two of four)
@pytest.mark.parametrize("edges,cells,gb", [(None, [1, 1, 1], "0.02"),
                                            ((13.0, 14.0, 14.5), [2, 2, 2], "0.0055"),
                                            ((9.0, 9.1, 26.0), [3, 3, 1], "0.0055")])
def test_shifted_matrices_in_parts(edges, cells, gb, monkeypatch):
    if edges is None:
        geo, st = _spread(257, 257), Settings()
    else:
        geo = _spread(18, 5, gap=2.3)
        geo = Geometry(geo.names, geo.coords_ang - geo.coords_ang.min(0), geo.hirshfeld, np.diag(edges))
        st = Settings(mbd_supercell_cutoff=25.0, mbd_cfdm_dip_cutoff=60.0, mbd_scs_dip_cutoff=30.0)
    out, supercell = _budget(geo, st, gb, monkeypatch)
    assert supercell == cells
    assert out[1][1]["logdet_diag"]["launches"] > out[0][1]["logdet_diag"]["launches"] > 0
    assert out[1][1]["bisect"]["launches"] == 0
    assert out[1][0] == out[0][0]


@pytest.mark.parametrize("edges", [None, (13.0, 14.0, 14.5)])
def test_no_room_for_a_shifted_matrix(edges, monkeypatch):
    geo = _spread(18, 5, gap=2.3)
    lat = None if edges is None else np.diag(edges)
    geo = Geometry(geo.names, geo.coords_ang - geo.coords_ang.min(0), geo.hirshfeld, lat)
    st = Settings(mbd_supercell_cutoff=25.0, mbd_cfdm_dip_cutoff=60.0, mbd_scs_dip_cutoff=30.0)
    out, _ = _budget(geo, st, "0.0001", monkeypatch)
    assert out[1][1]["logdet_diag"]["launches"] == 0 and out[1][1]["bisect"]["launches"] > 0
    assert out[1][0] == out[2][0]


def _energy80(geo, alpha, omega, reff, beta):
    """Energy of a molecule in 80-bit arithmetic by Jacobi's method."""
    L = np.longdouble
    x = (np.asarray(geo.coords_ang) / BOHR).astype(L)
    a, w, R = (np.asarray(v).astype(L) for v in (alpha, omega, reff))
    n = len(x)
    d = x[:, None] - x[None]
    r = np.sqrt((d ** 2).sum(-1)) + np.eye(n, dtype=L)
    damp = 1 + np.exp(-6 * (r / (L(beta) * (R[:, None] + R[None])) - 1))
    c = w[:, None] * w[None] * np.sqrt(a[:, None] * a[None]) / (damp * r ** 5) * (1 - np.eye(n, dtype=L))
    A = np.zeros((n, 3, n, 3), L)
    for i in range(3):
        for j in range(3):
            A[:, i, :, j] = ((r * r if i == j else 0) - 3 * d[..., i] * d[..., j]) * c
    A = A.reshape(3 * n, 3 * n) + np.diag(np.repeat(w * w, 3))
    while np.abs(np.tril(A, -1)).max() > 1e-17:
        for p in range(3 * n - 1):
            for q in range(p + 1, 3 * n):
                if abs(A[p, q]) < 1e-22:
                    continue
                th = (A[q, q] - A[p, p]) / (2 * A[p, q])
                t = (1 if th >= 0 else -1) / (abs(th) + np.sqrt(th * th + 1))
                cs = 1 / np.sqrt(t * t + 1)
                sn = t * cs
                A[p], A[q] = cs * A[p] - sn * A[q], sn * A[p] + cs * A[q]
                A[:, p], A[:, q] = cs * A[:, p] - sn * A[:, q], sn * A[:, p] + cs * A[:, q]
    return np.sqrt(np.diag(A)).sum() / 2 - 1.5 * w.sum()


def test_small_energies_against_80_bits():
    """Eight rings of 12 atoms, energies of 0.007 Ha between sums of 8 Ha: the
    quadrature's 2e-14 of the energy, the matrix elements' (16 eps each, the
    energy is quadratic in them), and eps of every row in the nodes whose
    logarithms come from the diagonal (weights below 0.25 in all)."""
    worst = 0.0
    for seed in range(8):
        rng = np.random.default_rng(seed)
        geo, st = generators.ring()
        geo.coords_ang = geo.coords_ang + rng.normal(0.0, 0.02, geo.coords_ang.shape)
        free = np.array([engine.free_atom_params(s) for s in geo.names])
        a = free[:, 1] * rng.uniform(0.5, 0.8, 12)
        with engine.MbdEngine(0) as eng:
            eng.set_geometry(geo, st)
            got, om, rf, _ = eng.energy(a, free[:, 0] * rng.uniform(0.4, 0.6, 12))
        want = _energy80(geo, a, om, rf, engine.beta(st.flag_xc))
        eps = 2.2e-16
        tol = (2e-14 + 32 * eps) * abs(want) + 0.25 * eps * np.sqrt(36)
        worst = max(worst, float(abs(got - want) / tol))
    assert worst <= 1.0


def test_largest_orders(monkeypatch):
    """Order 16803: log-determinants, which the band reduction overtakes past 22000."""
    n = 5601
    geo = _spread(n, n)
    free = np.array([engine.free_atom_params(s) for s in geo.names])
    a, c = free[:, 1] * geo.hirshfeld, free[:, 0] * geo.hirshfeld ** 2
    with engine.MbdEngine(0) as eng:
        eng.set_geometry(geo, Settings())
        monkeypatch.setenv("MBD_EIG_METHOD", "2")
        want, om, _, dw = eng.energy(a, c)
        monkeypatch.delenv("MBD_EIG_METHOD")
        eng.profile_enable(True)
        got, _, _, dg = eng.energy(a, c)
        prof = eng.profile_read()
    assert prof["logdet_diag"]["launches"] > 0 and prof["bisect"]["launches"] == 0
    assert dg["n_negative"] == dw["n_negative"] == 0
    assert abs(got - want) <= 2.2e-16 * 3 * n * 1.5 * np.sum(om)
