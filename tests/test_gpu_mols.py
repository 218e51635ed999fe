"""Batched molecules above the persistent kernel's size (csrc/mol.hip) against
that kernel (MBD_EIG_METHOD puts every molecule there), at the edges of the
128-column blocks and of the 16-row leading dimensions, with molecules that
have to go back to the persistent kernel, and in several memory chunks."""
import numpy as np
import pytest

from mbd_amd import engine, generators, io

pytestmark = pytest.mark.gpu


def _batch(mols, mode, monkeypatch, method=None):
    if method:
        monkeypatch.setenv("MBD_EIG_METHOD", method)
    with engine.MbdEngine(0) as eng:
        eng.batch_set(mols, io.Settings())
        out = eng.batch_run(mode)
    if method:
        monkeypatch.delenv("MBD_EIG_METHOD")
    return out


def _chain(rng, n):
    return generators.chain_molecule(rng, n - 2)  # n atoms


def _check(got, want):
    # FP64 residuals of both forms are at most 1e-12 and the relay matrices'
    # condition numbers below 1e3
    assert np.allclose(got["alpha_all"], want["alpha_all"], rtol=2e-9, atol=0)
    assert np.allclose(got["c6_eff"], want["c6_eff"], rtol=4e-9, atol=0)
    assert np.allclose(got["c6_mol"], want["c6_mol"], rtol=4e-9, atol=0)
    assert np.allclose(got["energy"], want["energy"], rtol=4e-9, atol=1e-11)
    assert np.array_equal(got["stat"][:, [0, 1, 3]], want["stat"][:, [0, 1, 3]])


# orders 96 (persistent), 99, 126, 129, 255, 258, 384, 387 and 1296, the largest
@pytest.mark.parametrize("mode", ["fp64", "mixed"])
def test_block_edges(mode, monkeypatch):
    rng = np.random.default_rng(3)
    mols = [_chain(rng, n) for n in (33, 128, 32, 42, 86, 432, 43, 85, 129, 5)]
    got = _batch(mols, mode, monkeypatch)
    _check(got, _batch(mols, mode, monkeypatch, "1"))
    assert got["diag"]["max_residual"] <= 1e-12


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
def test_large_molecules_only(mode, monkeypatch):
    mols = [_chain(np.random.default_rng(k), n) for k, n in ((4, 50), (5, 44))]
    _check(_batch(mols, mode, monkeypatch), _batch(mols, mode, monkeypatch, "1"))


# lines of sodium atoms: at 3 A the coupled matrix has negative eigenvalues, at
# 1.5 A relay matrices are indefinite; the persistent kernel's results, with
# its statistics
@pytest.mark.parametrize("mode", ["fp64", "mixed"])
def test_back_to_the_persistent_kernel(mode, monkeypatch):
    rng = np.random.default_rng(5)
    lines = [io.Geometry(["Na"] * 40, np.array([[0.0, 0.0, gap * i] for i in range(40)]), np.ones(40))
             for gap in (3.0, 1.5)]
    mols = [_chain(rng, 60), *lines, _chain(rng, 36),
            _chain(rng, 9)]
    got, want = _batch(mols, mode, monkeypatch), _batch(mols, mode, monkeypatch, "1")
    assert want["stat"][1, 0] == 0 and want["stat"][1, 1] > 0 and want["stat"][2, 0] > 0
    assert np.array_equal(got["stat"][1:3], want["stat"][1:3])
    assert np.array_equal(got["energy"][1:3], want["energy"][1:3], equal_nan=True)
    keep = np.ones(sum(m.n_atoms for m in mols), bool)
    keep[60:140] = False
    assert np.array_equal(got["alpha_all"][:, ~keep], want["alpha_all"][:, ~keep], equal_nan=True)
    assert np.allclose(got["alpha_all"][:, keep], want["alpha_all"][:, keep], rtol=2e-9, atol=0)
    assert np.allclose(got["energy"][[0, 3, 4]], want["energy"][[0, 3, 4]], rtol=4e-9, atol=1e-11)


def test_memory_chunks(monkeypatch):
    mols = [_chain(np.random.default_rng(n), n) for n in (70, 45, 71, 34, 101)]
    want = _batch(mols, "mixed", monkeypatch)
    monkeypatch.setenv("MBD_SCS_MEM_GB", "0.02")  # less than any of them: one at a time
    got = _batch(mols, "mixed", monkeypatch)
    assert np.array_equal(got["energy"], want["energy"])
    assert np.array_equal(got["alpha_all"], want["alpha_all"])


# molecules with close contacts, some of them with an atom of negative alpha
# (a coupled matrix that is not finite) or with omega^2 over four decades and
# more, which the log-determinants do not cover
@pytest.mark.parametrize("mode", ["fp64", "mixed"])
def test_close_contacts(mode, monkeypatch):
    mols = generators.chain_molecules()[0][::11]
    got, want = _batch(mols, mode, monkeypatch), _batch(mols, mode, monkeypatch, "1")
    off = got["offsets"]
    low = np.array([want["alpha_eff"][a:b].min() for a, b in zip(off[:-1], off[1:])])
    assert (low < 0).any() and ((low > 0) & (low < 0.5)).any()
    # as above, alpha relative to its molecule's largest: a small one is a difference
    for a, b in zip(off[:-1], off[1:]):
        w = want["alpha_all"][:, a:b]
        assert np.all(np.abs(got["alpha_all"][:, a:b] - w) <= 2e-9 * np.abs(w).max(1, keepdims=True))
    assert np.array_equal(got["stat"][:, [0, 1, 3]], want["stat"][:, [0, 1, 3]])
    ok = low > 2.0  # omega = 4 C6 / (3 alpha^2) of a difference carries its error
    assert ok.sum() > 20
    assert np.allclose(got["energy"][ok], want["energy"][ok], rtol=4e-9, atol=1e-11)
    assert np.allclose(got["energy"], want["energy"], rtol=1e-6, atol=0, equal_nan=True)
