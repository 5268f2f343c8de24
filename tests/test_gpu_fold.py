"""The ordered folds (Loewner products, column norms) at the edges of their splits: chunks
of 64 poles, 16 or 64 roots per block, and the three ways a level's 256-root chunks are
divided over blocks (up to 16, from 17 and from 1024 chunks).  The fold keeps the pole
order, so every value equals the oracle's bit for bit, and a batch's problems equal the
same problems solved alone."""
import numpy as np
import pytest

import oracle_py as O
from hsspack_amd.workloads import bidiag_toeplitz, tridiag_cfg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.fixture(scope="module")
def ctx(torch_dev):
    from hsspack_amd import hsdc
    c = hsdc.Context()
    yield c
    c.close()


@pytest.mark.parametrize("K", [3, 15, 16, 17, 63, 64, 65, 127, 128, 129, 192, 255, 256, 257, 1025, 4096, 4097])
def test_loewner_and_alpha_edges_bitexact(ctx, K):
    rng = np.random.default_rng(K)
    d = np.sort(rng.uniform(-1, 1, K))
    z = rng.standard_normal(K)
    z /= np.linalg.norm(z)
    g = ctx.loewner(d, z, 0.9)
    r = O.mdlaed3_vectors(d, z, 0.9)
    assert g["info"] == 0
    for key in ("d", "z", "difl", "alpha"):
        assert np.array_equal(g[key], r[key]), key
    assert np.array_equal(g["difr"][:-1], r["difr"][:-1])


@pytest.mark.parametrize("K", [33000])
def test_wide_split_of_one_merge(torch_dev, ctx, K):
    """More than 128 chunks (64 roots per block): the roots' Loewner identity, z unchanged up
    to rounding (a product of K correctly rounded quotients: relative error <= 2 K eps) and
    unit columns."""
    rng = np.random.default_rng(1)
    t = (np.arange(K) + 0.5 + 0.8 * (rng.uniform(0, 1, K) - 0.5)) / K
    d = 2.0 - 2.0 * np.cos(np.pi * t)
    z = rng.uniform(0.5, 1.5, K)
    z /= np.linalg.norm(z)
    g = ctx.loewner(d, z, 1.0)
    assert g["info"] == 0
    assert np.abs(g["z"] / z - 1).max() <= 2 * K * 2.0 ** -53
    j = rng.integers(0, K - 1, 20)
    for q in j:
        below = (d - d[q]) - g["difl"][q]
        above = (d - d[q + 1]) - g["difr"][q]
        v = g["z"] / np.where(np.arange(K) <= q, below, above)
        assert abs(g["alpha"][q] * np.linalg.norm(v) - 1) <= 2 * K * 2.0 ** -53


@pytest.mark.parametrize("count,n", [(5, 61), (150, 61), (1100, 33)])
def test_batch_split_equals_single_solves(torch_dev, ctx, count, n):
    torch = torch_dev
    probs = [tridiag_cfg(1, n, 70, sub=i) for i in range(count)]
    ns = [n] * count
    D = torch.tensor(np.concatenate([d for d, _ in probs]), device="cuda:0")
    E = torch.tensor(np.concatenate([np.append(e, 0.0) for _, e in probs]), device="cuda:0")
    Z = torch.zeros(count * n * n, dtype=torch.float64, device="cuda:0")
    rc = ctx.stedc_batched_dev(ns, np.arange(count) * n, D, E, Z, np.arange(count) * n * n)
    torch.cuda.synchronize()
    assert rc == 0
    for i in (0, count // 2, count - 1):
        d1 = torch.tensor(probs[i][0], device="cuda:0")
        e1 = torch.tensor(np.append(probs[i][1], 0.0), device="cuda:0")
        z1 = torch.zeros((n, n), dtype=torch.float64, device="cuda:0")
        assert ctx.stedc_dev(d1, e1, z1) == 0
        torch.cuda.synchronize()
        assert torch.equal(D[i * n:(i + 1) * n], d1)
        assert torch.equal(Z[i * n * n:(i + 1) * n * n].reshape(n, n), z1)


@pytest.mark.parametrize("n", [65, 130, 257])
def test_svd_fold_edges_bitexact(torch_dev, n):
    from hsspack_amd import hsdc
    c = hsdc.BdContext()
    d, e = bidiag_toeplitz(n, n)
    s, u, vt, info = c.bdsdc(d, e)
    c.close()
    assert info == 0
    r = O.bdsdc(d, e)
    assert np.array_equal(s, r["d"]) and np.array_equal(u, r["u"]) and np.array_equal(vt, r["vt"])


@pytest.mark.parametrize("n,uplo", [(511, "U"), (513, "L"), (1023, "L"), (1025, "U"), (1091, "L")])
def test_svd_vector_products(torch_dev, n, uplo):
    """The products of the singular vectors gather the columns of a merge 512 at a time
    and only those that meet a tile's rows: almost no deflation, so the top merge's K lies
    on both sides of 512 and 1024; the same bits as the oracle's full sums."""
    rng = np.random.default_rng(n)
    d, e = 2.0 + 0.01 * rng.uniform(size=n), 1.0 + 0.01 * rng.uniform(size=n - 1)
    from hsspack_amd import hsdc
    c = hsdc.BdContext()
    try:
        s, u, vt, info = c.bdsdc(d, e, uplo=uplo)
        assert info == 0 and c.trace()["k"].max() > 0.9 * n
    finally:
        c.close()
    r = O.bdsdc(d, e, uplo=uplo.encode())
    np.testing.assert_array_equal(s, r["d"])
    np.testing.assert_array_equal(u, r["u"])
    np.testing.assert_array_equal(vt, r["vt"])
