"""The blocked Cholesky at the edges of its sub-blocks (32), diagonal blocks
(128) and outer blocks, and the pivot it reports in each of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _spd(n, seed):
    M = np.random.default_rng(seed).standard_normal((n, n))
    return M @ M.T / n + np.eye(n)  # condition number about 5


@pytest.mark.parametrize("n", [31, 32, 33, 63, 64, 65, 95, 96, 97, 160, 224, 255, 257])
def test_cholesky_sub_block_edges(n):
    from mbd_amd import engine
    A = np.array([_spd(n, n), _spd(n, n + 1)])
    L, info = engine.device_cholesky(A)
    assert list(info) == [0, 0]
    for b in range(2):
        # forward error of a Cholesky factor: n eps cond(A) |L|, n <= 257
        assert np.allclose(L[b], np.linalg.cholesky(A[b]), rtol=0, atol=257 * 2.3e-16 * 10 * 2)


@pytest.mark.parametrize("at", [1, 32, 33, 64, 97, 128, 129, 200])
def test_cholesky_reports_each_pivot(at):
    from mbd_amd import engine
    A = _spd(200, at)
    A[at - 1, at - 1] = -1.0
    _, info = engine.device_cholesky(A)
    assert info[0] == at


# fewer rows or columns than a 16-byte vector, one short of and one past a
# vector and a tile, odd leading dimensions, K remainders
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 130, 5), (3, 200, 17), (130, 3, 15), (127, 129, 16),
                                   (129, 127, 31), (131, 133, 1), (257, 255, 47), (256, 128, 64)])
def test_gemm_edges(m, n, k, fp32):
    from mbd_amd import engine
    rng = np.random.default_rng(m * 1000 + n)
    t = np.float32 if fp32 else np.float64
    A, B, C = (rng.standard_normal(s).astype(t).astype(np.float64) for s in ((m, k), (n, k), (m, n)))
    got = engine.device_gemm_nt(A, B, C, alpha=-1.0, beta_=1.0, fp32=fp32)
    # k + 1 roundings of sums no larger than |A| |B|^T + |C|
    eps = 6e-8 if fp32 else 1.2e-16
    assert np.all(np.abs(got - (C - A @ B.T)) <= 2 * (k + 2) * eps * (np.abs(A) @ np.abs(B).T + np.abs(C)))


def test_cholesky_pivot_rounding():
    """Column 0 of the factor is a_i / sqrt(d): no further from it than the
    reciprocal square root's 1.5 and the product's 1 unit of 2^-53 (d and a_i
    from 31 of 640 arrow matrices; the two rounded operations and the product
    reach 3 units)."""
    from mbd_amd import engine
    rng = np.random.default_rng(0)
    b, n = 640, 32
    A = np.zeros((b, n, n))
    A[:, np.arange(n), np.arange(n)] = 1e6
    A[:, 0, 0] = np.exp(rng.uniform(-4, 4, b))
    A[:, 1:, 0] = rng.uniform(-1, 1, (b, n - 1))
    A[:, 0, 1:] = A[:, 1:, 0]
    L, info = engine.device_cholesky(A)
    assert not info.any()
    want = A[:, 1:, 0].astype(np.longdouble) / np.sqrt(A[:, 0, 0].astype(np.longdouble))[:, None]
    err = np.abs(L[:, 1:, 0] - want) / np.abs(want)
    assert err.max() <= 2.5 * 2.0 ** -53 * (1 + 1e-6)


# one short of, at and one past outer blocks of 512 columns, and the FP32 form
# (the mixed solve's factor) at the edges of sub-blocks and diagonal blocks too
@pytest.mark.parametrize("n,fp32", [(511, False), (512, False), (513, False), (640, False), (1025, False)] +
                         [(n, True) for n in (1, 31, 33, 64, 97, 128, 129, 257, 511, 512, 513, 1025)])
def test_cholesky_outer_blocks_and_fp32(n, fp32):
    from mbd_amd import engine
    t = np.float32 if fp32 else np.float64
    A = np.array([_spd(n, n), _spd(n, n + 1)]).astype(t)
    L, info = engine.device_cholesky(A, fp32=fp32)
    assert L.dtype == t and list(info) == [0, 0]
    for b in range(2):
        # as above: n eps cond(A) |L|
        want = np.linalg.cholesky(A[b].astype(np.float64))
        assert np.allclose(L[b], want, rtol=0, atol=n * (1.2e-7 if fp32 else 2.3e-16) * 10 * 2)


@pytest.mark.parametrize("at,fp32", [(512, False), (513, False), (700, False), (1, True), (33, True),
                                     (128, True), (129, True), (513, True), (700, True)])
def test_cholesky_reports_pivot_past_outer_block(at, fp32):
    from mbd_amd import engine
    A = _spd(700, at)
    A[at - 1, at - 1] = -1.0
    _, info = engine.device_cholesky(np.array([A, _spd(700, 1)]), fp32=fp32)
    assert list(info) == [at, 0]


def test_cholesky_pivot_rounding_fp32():
    """As test_cholesky_pivot_rounding, in units of 2^-24."""
    from mbd_amd import engine
    rng = np.random.default_rng(0)
    b, n = 640, 32
    A = np.zeros((b, n, n), np.float32)
    A[:, np.arange(n), np.arange(n)] = 1e4
    A[:, 0, 0] = np.exp(rng.uniform(-4, 4, b))
    A[:, 1:, 0] = rng.uniform(-1, 1, (b, n - 1))
    A[:, 0, 1:] = A[:, 1:, 0]
    L, info = engine.device_cholesky(A, fp32=True)
    assert not info.any()
    want = A[:, 1:, 0].astype(np.float64) / np.sqrt(A[:, 0, 0].astype(np.float64))[:, None]
    err = np.abs(L[:, 1:, 0] - want) / np.abs(want)
    assert err.max() <= 2.5 * 2.0 ** -24 * (1 + 1e-6)
