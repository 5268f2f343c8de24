"""Inputs with a NaN or an infinity: a call returns, never takes an index from a value, and
does not turn such an input into finite results."""
import numpy as np
import pytest

import oracle_py as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.fixture(scope="module")
def sb(torch_dev):
    from hsspack_amd import hsdc
    c = hsdc.SbContext()
    yield c
    c.close()


@pytest.mark.parametrize("n", [2, 5, 64, 65, 98, 100, 128])
def test_band_leaf_keeps_a_nan(sb, n):
    """One leaf, a diagonal matrix: eigenvalues and vectors only change places, in the order of
    the oracle's serial selection sort, for a NaN at any position (beside infinities too)."""
    rng = np.random.default_rng(n)
    at = range(n) if n <= 5 else sorted({0, 1, 62, 63, 64 % n, n // 2, n - 2, n - 1})
    for p in at:
        ab = np.zeros((2, n))
        ab[1] = rng.permutation(n) - n // 2
        if n > 5:
            ab[1, (p + 3) % n], ab[1, (p + 7) % n] = np.inf, -np.inf
        ab[1, p] = np.nan
        w, q, info = sb.sbevd(ab, 1)
        r = O.sbevd(ab, 1, smlsiz=128)
        assert info == 0 and r["info"] >= 0
        np.testing.assert_array_equal(w, r["d"])
        np.testing.assert_array_equal(q, r["q"])
        assert np.isnan(w).sum() == 1 and np.array_equal(np.sort(q.sum(axis=0)), np.ones(n))


@pytest.mark.parametrize("n,kd", [(60, 4), (128, 9)])
def test_band_leaf_nan_beside_rotations(sb, n, kd):
    """No rotation touches a row with a NaN on the diagonal: the other eigenvalues are those of
    the matrix without that row and column, and the NaN stays among them."""
    from hsspack_amd.workloads import band_cfg, band_dense
    ab = band_cfg(n, kd, seed=n)
    a = band_dense(ab)
    for p in (0, n // 3, n - 1):
        bad = ab.copy()
        bad[kd, p] = np.nan
        w, q, info = sb.sbevd(bad, kd)
        keep = np.arange(n) != p
        want = np.linalg.eigvalsh(a[np.ix_(keep, keep)])
        assert info == 0 and np.isnan(w).sum() == 1, p
        assert np.abs(np.sort(w[~np.isnan(w)]) - want).max() <= 4 * n * 2.0 ** -53 * np.abs(want).max()
        assert np.linalg.matrix_rank(q) == n
