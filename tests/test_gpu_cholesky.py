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
