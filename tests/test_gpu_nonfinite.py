"""Inputs with a NaN or an infinity: a call returns, never takes an index from a value, and
does not turn such an input into finite results."""
import numpy as np
import pytest

import oracle_py as O
from test_oracle_dhssmm import fmm_matrix

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


@pytest.fixture(scope="module")
def ctx(torch_dev):
    from hsspack_amd import hsdc
    c = hsdc.Context()
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


def same_product(y, ref, rel):
    """The same entries are NaN or infinite, the others agree."""
    fin = np.isfinite(ref)
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))
    np.testing.assert_array_equal(y[np.isinf(ref)], ref[np.isinf(ref)])
    assert fin.any() and np.abs(y[fin] - ref[fin]).max() <= rel * np.abs(ref[fin]).max()


@pytest.mark.parametrize("n,ni", [(300, 40), (330, 99), (420, 130), (500, 160), (151, 100), (900, 60)])
@pytest.mark.parametrize("seed", [None, 7])
def test_dense_to_hss_product(ctx, n, ni, seed):
    """A NaN, an infinity or squares that overflow in an off-diagonal block leave no singular
    values to order, with R and V in LDS, R alone or neither, for contexts wider and narrower
    than the block and after a tree of QRs: the product is taken densely.  On a leaf's diagonal
    block the form is built as ever, and the leaf's rows carry the value."""
    a0 = fmm_matrix(n, 5)
    b = np.random.default_rng(n).uniform(0.5, 1, (n, 30))
    for at, x in (((n - 1, 0), np.nan), ((0, n - 1), np.inf), ((n // 4, 3 * n // 4), -np.inf), ((1, 0), np.nan)):
        a = a0.copy()
        a[at] = x
        y, _, ranks = ctx.dhssmm(a, b, ni, 1e-11, seed=seed)
        assert (ranks is None) == (at != (1, 0)), at
        same_product(y, a @ b, 1e-9)
    y, _, ranks = ctx.dhssmm(a0 * 2.0 ** 520, b, ni, 1e-11, seed=seed)
    assert ranks is None
    same_product(y, (a0 @ b) * 2.0 ** 520, 1e-12)
    y, _, ranks = ctx.dhssmm(a0, b, ni, 1e-11, seed=seed)
    assert ranks is not None
    same_product(y, a0 @ b, 1e-9)


@pytest.mark.parametrize("K,ni", [(513, 64), (1500, 64), (1500, 256)])
def test_structured_product_with_a_nan(ctx, K, ni):
    """A NaN among the row generators stays one row of the Schur complements: the swap check's
    lanes must agree on every column's largest entry all the same.  Every entry of the product
    sums over that row; the call after it is as if the NaN had not been."""
    rng = np.random.default_rng(K)
    d = np.sort(rng.uniform(-1, 1, K))
    z = rng.standard_normal(K)
    z /= np.linalg.norm(z)
    v = O.mdlaed3_vectors(d, z, 1.1)
    x = rng.uniform(0.5, 1, (9, K))

    def product(zz):
        return ctx.hss_evc(v["dlamda"], v["d"], zz, v["alpha"], v["difl"], v["difr"], x, ni, 1e-14)

    want, ranks = product(v["z"])
    for p in (0, 70, K // 2, K - 1):
        zz = v["z"].copy()
        zz[p] = np.nan
        y, _ = product(zz)
        assert np.isnan(y).all(), p
    again, ranks2 = product(v["z"])
    np.testing.assert_array_equal(again, want)
    np.testing.assert_array_equal(ranks2, ranks)
